"""The chemistry kernels compiled for the shipped mechanism's structure against
the ones that read any mechanism from the bank: a twentieth reaction whose
rates are zero changes the structure, so the general kernels run, and adds
exact zeros to every sum.  The results are therefore equal bit for bit."""
import copy
import json

import numpy as np
import pytest

from conftest import load_package, gpu_available
import chemcase

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    if not gpu_available():
        pytest.skip("no GPU")
    load_package()
    from ocfd_amd import mechanism
    d = json.load(open(mechanism.JET_JSON))
    g = copy.deepcopy(d)
    r = copy.deepcopy(g["mechanism"]["reactions"][0])
    r["arrhenius"] = [[0.0, 0.0, 0.0]]
    g["mechanism"]["reactions"].append(r)
    g["mechanism"]["n_reac"] += 1
    b = chemcase.jet_batch(1000)[0]
    # some cells above the fits' temperature range (5000 K) and some with
    # species that are absent or slightly negative
    rho, E = b["rho"].copy(), b["E"].copy()
    M = mechanism.Mechanism(data=d)
    T = np.full(50, 5400.0)
    E[:50] = M.energy(rho[:, :50], T)
    rho[5, 50:80] = 0.0
    rho[6, 80:100] = -1e-12
    return M, mechanism.Mechanism(data=g), rho, E, b["dt"]


def both(env, n, call):
    import torch
    from ocfd_amd import chemistry
    out = []
    for M in env[:2]:
        ch = chemistry.ChemBatch(M)
        rho, E, dt = (torch.tensor(np.ascontiguousarray(a[..., :n]), dtype=torch.float64, device="cuda") for a in env[2:])
        ns = call(ch, rho, E, dt)
        torch.cuda.synchronize()
        out.append([rho.cpu().numpy(), E.cpu().numpy()] + ([] if ns is None else [ns.cpu().numpy()]))
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
    return out[0]


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("mode", [-1, 1, 2, 3])
def test_fixed_integrators(env, mode, n):
    both(env, n, lambda ch, r, e, d: ch.chemical_timeAdv(r, e, d * (1.0 if mode < 0 else 1e-3), mode=mode, nsub=2))


def test_implicit_step_that_blows_up(env):
    """Point-implicit steps far beyond the chemistry's time scales leave some
    cells without a number; the same cells, in every species, on both."""
    r, e = both(env, 1000, lambda ch, r, e, d: ch.chemical_timeAdv(r, e, d * 300.0, mode=-1, nsub=8))
    bad = ~np.isfinite(e)
    assert 0 < bad.sum() < 1000
    assert np.all(np.isnan(r[:, np.isnan(e)]))


@pytest.mark.parametrize("n", [1, 2, 3, 63, 65, 1000])
@pytest.mark.parametrize("scheduler", [0, 1, 2])
def test_adaptive(env, scheduler, n):
    """All three schedulers (0: one cell per lane; 1 and 2: also one cell per
    wavefront for the last cells) on both structures."""
    got = both(env, n, lambda ch, r, e, d: ch.adaptive(r, e, d * 20.0, max_sub=2000, scheduler=scheduler))
    ref = both(env, n, lambda ch, r, e, d: ch.adaptive(r, e, d * 20.0, max_sub=2000, scheduler=0))
    for a, b in zip(got, ref):
        assert np.array_equal(a, b, equal_nan=True)
