"""Cells of 70 to 80 K, where exp(G/RT) of a dissociation overflows although the
rate that it scales (exp(-E/T) as small) is an ordinary number: finite wherever
the oracle is, and equal to it up to the oracle's own loss there, which divides
by an equilibrium constant Kc in the subnormal range (spacing 2^-1074)."""
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
    b, M, orc = chemcase.jet_batch(1000)
    M2 = copy.deepcopy(M)  # a twentieth reaction without a rate: the kernels for any mechanism
    for a in ("af_type", "third_body", "fc_troe", "arrhenius", "vf", "vr", "eff", "reverse"):
        setattr(M2, a, np.concatenate([getattr(M2, a), getattr(M2, a)[:1]]))
    M2.arrhenius[-1] = 0.0
    M2.n_reac += 1
    yield M, M2, orc, b["rho"][:, :300], b["dt"][:300]
    from ocfd_amd import chemistry
    chemistry.ChemBatch(M)


@pytest.mark.parametrize("any_mechanism", [0, 1])
@pytest.mark.parametrize("T", [70.0, 70.5, 71.0, 71.5, 72.0, 72.5, 73.0, 74.0, 80.0])
@pytest.mark.parametrize("mode", [-1, 1, 3])
def test_cold_cells(env, mode, T, any_mechanism):
    import torch
    from ocfd_amd import chemistry
    M, M2, orc, rho, dt = env
    ch = chemistry.ChemBatch(M2 if any_mechanism else M)
    E = M.energy(rho, np.full(rho.shape[1], T))
    d = dt * (1.0 if mode < 0 else 1e-3)
    r, e, q = (torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda") for a in (rho, E, d))
    ch.chemical_timeAdv(r, e, q, mode=mode, nsub=1)
    ch.synchronize()
    r, e = r.cpu().numpy(), e.cpu().numpy()
    ro, eo = orc.batch(mode, rho.T, E, d, 1)
    ro = ro.T
    ok = np.isfinite(ro).all(0) & np.isfinite(eo)
    assert ok.sum() > 100
    assert np.isfinite(r[:, ok]).all() and np.isfinite(e[ok]).all()
    # per cell: what the oracle's result moves by for one ulp of its input, times the tens of
    # roundings in a rate, and the oracle's loss in a subnormal Kc, of the cell's change
    kc = np.abs(orc.rate_coef(rho[:, 0] / M.mi * 1e-6, T)[2])
    rng = np.random.default_rng(0)
    sr, se = np.zeros_like(E), np.zeros_like(E)
    for _ in range(8):
        u = lambda a: a * (1.0 + 2.0 ** -52 * rng.integers(-1, 2, a.shape))
        r1, e1 = orc.batch(mode, u(rho).T, u(E), d, 1)
        sr, se = np.maximum(sr, np.abs(r1.T - ro).max(0)), np.maximum(se, np.abs(e1 - eo))
    loss = 8.0 * 2.0 ** -1074 / kc[kc > 0].min()
    dr, de = np.abs(ro - rho).max(0), np.abs(eo - E)
    assert (np.abs(r - ro).max(0) <= 64.0 * sr + loss * dr + 1e-15 * rho.sum(0))[ok].all()
    assert (np.abs(e - eo) <= 64.0 * se + loss * de + 1e-15 * E)[ok].all()


@pytest.mark.parametrize("scheduler", [0, 1, 2])
def test_adaptive(env, scheduler):
    """... and the adaptive integrator (the oracle's cells are finite here)."""
    import torch
    from ocfd_amd import chemistry
    M, _, orc, rho, dt = env
    ch = chemistry.ChemBatch(M)
    E = M.energy(rho, np.full(rho.shape[1], 72.0))
    ro, eo, _ = orc.adaptive_batch(rho.T, E, dt, 0.05, 1e-6, 0.01, 2000)
    ok = np.isfinite(ro).all(1) & np.isfinite(eo)
    assert ok.sum() > 100
    r, e, q = (torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda") for a in (rho, E, dt))
    ch.adaptive(r, e, q, scheduler=scheduler, max_sub=2000)
    ch.synchronize()
    assert ch.unfinished() == 0
    r, e = r.cpu().numpy(), e.cpu().numpy()
    assert np.isfinite(r[:, ok]).all() and np.isfinite(e[ok]).all()
    # the cells move away from where they started (radicals recombine)
    assert (np.abs(r - rho)[:, ok].max(0) > 0).any()
