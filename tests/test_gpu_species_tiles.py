"""The species kernels of large grids (LDS tiles, from 400 blocks of cells) with
periodic directions, remainder tiles and in inviscid runs: a step against the
one-species entries, which take one thread per cell, bit for bit, and one of
them against the oracle."""
import numpy as np
import pytest

from conftest import load_package, gpu_available
import flowcase as fc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    if not gpu_available():
        pytest.skip("no GPU")
    return load_package()


def jet(n, periodic, vis=5, viscous=1):
    """The round jet's state in a box with the given periodic directions; no
    boundary condition where xi is periodic."""
    case = fc.small_jet(*n)
    cfg, mesh, span, st, bc, info = case
    cfg.periodic[:] = periodic
    cfg.scheme_vis = vis
    cfg.if_viscous = viscous
    if periodic[0]:
        cfg.ibc, bc = 0, None
    span = np.zeros(9)
    for d, length in enumerate((0.004, 0.003, 0.003)):
        span[4 * d] = length * n[d] / (n[d] - 1.0) * periodic[d]
    return cfg, mesh, span, st, bc, info


def step_and_entries(pkg, case):
    cfg, dt, ns = case[0], 0.2 * case[5]["dt"], case[0].n_spec
    names = ("F", "FN", "DI", "T", "P") + (("QP",) if cfg.if_viscous else ())
    a = pkg.FlowSolver(cfg)
    fc.setup_jet(a, case)
    a.flow_time_advance(dt)
    fa = {k: a.download(k) for k in names}
    a.close()
    b = pkg.FlowSolver(cfg)
    fc.setup_jet(b, case)
    b.save_stage0()
    for krk in (1, 2, 3):
        b.stage_begin(krk)
        for m in range(1, ns + 1):
            b.du_scaler_invis(m)
            if cfg.if_viscous:
                b.du_scaler_viscous(m)
            b.scalar_time_adv_rk3(krk, m, dt)
        b.du_inviscous()
        if cfg.if_viscous:
            b.du_viscous()
        b.OCFD_time_adv_RK3(krk, dt)
        b.comput_flow_variables()
        b.OCFD_bc()
    for k, v in fa.items():
        w = b.download(k)
        # (ghost cells of T and P hold what the set-up left)
        assert np.isfinite(v).all() and v.tobytes() == w.tobytes(), k
    b.close()


# 75 x 37 x 38: remainder tiles of 32 x 8 in both directions; rows of 9 and of 8 cells
# are shorter than a tile and its periodic image
GRIDS = [(75, 37, 38), (9, 41, 300), (300, 9, 39), (8, 8, 1700)]


@pytest.mark.parametrize("n", GRIDS)
@pytest.mark.parametrize("vis", [5, 6])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1)])
def test_periodic_tiles_equal_one_thread_per_cell(pkg, n, vis, periodic):
    assert n[0] * n[1] * n[2] > 400 * 256
    step_and_entries(pkg, jet(n, periodic, vis))


@pytest.mark.parametrize("n", [(75, 37, 38), (48, 36, 36)])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (0, 0, 1)])
def test_inviscid_step(pkg, n, periodic):
    step_and_entries(pkg, jet(n, periodic, viscous=0))


@pytest.mark.parametrize("periodic", [(1, 1, 1), (0, 1, 1)])
def test_tiles_against_the_oracle(pkg, periodic):
    import oracle
    case = jet((75, 37, 38), periodic)
    g, o = pkg.FlowSolver(case[0]), oracle.Oracle(pkg, case[0])
    for e in (g, o):
        fc.setup_jet(e, case)
        e.flow_time_advance(0.2 * case[5]["dt"])
    fc.compare_state(g, o)  # 1e-12 of each field's largest value: the fits' exp and log differ by ulps
    for m in range(case[0].n_spec):
        d, _ = fc.compare(fc.interior(g.download("DI")[..., m]), fc.interior(o.download("DI")[..., m]))
        assert d <= 1e-12, (m, d)
    g.close()
