"""Arrhenius reverse rates (ReReac = 1) at temperatures where ln T does not
exist: a cell without energy (T = 0: pow(0, b) exp(-E/0) is zero for b >= 0,
E > 0) and cells of negative energy (T < 0, where T^b exists for whole b),
beside ordinary cells and one whose energy is not a number, against the
oracle, for both kinds of integrator."""
import copy

import numpy as np
import pytest

from conftest import load_package, gpu_available
import chemcase

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    if not gpu_available():
        pytest.skip("no GPU")
    pkg = load_package()
    import oracle
    from ocfd_amd import chemistry
    b, M, _ = chemcase.jet_batch(1000)
    M2 = copy.deepcopy(M)
    M2.rereac = 1
    M2.af_type[:] = 0
    M2.arrhenius[:] = 0.0
    M2.reverse = np.zeros((M.n_reac, 5))
    for k in range(M.n_reac):
        M2.arrhenius[k, 0] = (1.0e6 * (1 + k), k % 3, 1500.0 + 100.0 * k)
        M2.reverse[k, :3] = (3.0e5 * (2 + k), (k + 1) % 3, 1200.0 + 150.0 * k)
    rho, E = b["rho"][:, :200].copy(), b["E"][:200].copy()
    A1 = ((8.314 / M.mi)[:, None] * (M.coef[:, 0, 0] - 1.0)[:, None] * rho).sum(0)
    E[:20] = 0.0
    E[20:60] = -A1[20:60] * np.linspace(150.0, 300.0, 40)
    E[60] = np.nan
    yield chemistry.ChemBatch(M2), oracle.ChemOracle(pkg, M2), rho, E, b["dt"][:200]
    chemistry.ChemBatch(M)
    oracle.ChemOracle(pkg, M)


@pytest.mark.parametrize("mode", [1, 2, 3, -1])
def test_fixed_integrators(env, mode):
    import torch
    ch, orc, rho, E, dt = env
    s = 1.0 if mode < 0 else 1e-13  # these rates are far beyond the explicit integrators' steps
    T = np.array([orc.T(rho[:, c], E[c]) for c in range(60)])
    assert (T[:20] == 0.0).all() and (T[20:60] < -100.0).all(), T
    r, e, d = (torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda") for a in (rho, E, dt))
    ch.chemical_timeAdv(r, e, d * s, mode=mode, nsub=2)
    ch.synchronize()
    r, e = r.cpu().numpy(), e.cpu().numpy()
    ro, eo = orc.batch(mode, rho.T, E, dt * s, 2)
    ro = ro.T
    # (RK3's stage weights leave a cell at T = 0 an energy of a rounding's size, whose
    # temperature has either sign)
    lo = 20 if mode == 3 else 0
    assert np.isfinite(ro[:, lo:60]).all() and np.isfinite(eo[lo:60]).all()
    assert np.isnan(e[60]) and np.isnan(eo[60]) and np.array_equal(np.isnan(r[:, 60]), np.isnan(ro[:, 60]))
    if lo == 0:  # no rate at T = 0: the cells stay as they are, on both
        assert np.array_equal(r[:, :20], rho[:, :20]) and np.array_equal(ro[:, :20], rho[:, :20])
    # (the implicit system of the T < 0 cells is singular to working precision: the oracle's
    # own result moves by 1e-5 when its input moves by one ulp)
    assert np.isfinite(r[:, lo:60]).all() and np.isfinite(e[lo:60]).all()
    ok = np.array([c for c in range(lo, 200) if c != 60 and not (mode < 0 and 20 <= c < 60)])
    assert np.max(np.abs(r - ro)[:, ok] / rho.sum(0)[ok]) <= 1e-12
    assert np.max(np.abs(e - eo)[ok]) <= 1e-12 * np.abs(E[ok]).max()
