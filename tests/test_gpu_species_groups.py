"""Species shared out over blocks (small grids: three shares and two, large
ones: one) against the one-species entries, which never share, bit for bit;
and mixtures of fewer than the largest number of species against the oracle."""
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


def _bits(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint64), np.ascontiguousarray(b).view(np.uint64))


@pytest.mark.parametrize("n", [(17, 9, 8), (48, 36, 36), (64, 48, 40), (97, 64, 56)])
@pytest.mark.parametrize("vis", [5, 6])
def test_shares_equal_single_species(pkg, n, vis):
    case = fc.small_jet(*n)
    case[0].scheme_vis = vis
    dt, ns = case[5]["dt"], case[0].n_spec
    names = ("F", "FN", "DI", "T", "P", "QP")
    a = pkg.FlowSolver(case[0])
    fc.setup_jet(a, case)
    a.flow_time_advance(dt)
    fa = {k: a.download(k) for k in names}
    a.close()
    b = pkg.FlowSolver(case[0])
    fc.setup_jet(b, case)
    b.save_stage0()
    for krk in (1, 2, 3):
        b.stage_begin(krk)
        for m in range(1, ns + 1):
            b.du_scaler_invis(m)
            b.du_scaler_viscous(m)
            b.scalar_time_adv_rk3(krk, m, dt)
        b.du_inviscous()
        b.du_viscous()
        b.OCFD_time_adv_RK3(krk, dt)
        b.comput_flow_variables()
        b.OCFD_bc()
    for k, v in fa.items():
        assert _bits(v, b.download(k)), k
    b.close()


@pytest.mark.parametrize("idx", [(1, 8), (1, 2, 3, 8), (0, 1, 2, 3, 4, 5, 6, 8)])
def test_fewer_species(pkg, idx):
    import oracle
    idx = list(idx)
    ns = len(idx)
    cfg, mesh, span, st, bc, info = fc.small_jet(20, 12, 10)
    mech = info["mech"]
    cfg.n_spec = ns
    st = dict(st)
    di = np.asarray(st["DI"])[..., idx]
    st["DI"] = np.asfortranarray(di * (np.asarray(st["D"]) / di.sum(-1))[..., None])
    inl = np.asarray(bc["inlet2d"])
    part = inl[..., [5 + k for k in idx]]
    part = part * (inl[..., 0] / part.sum(-1))[..., None]
    inl = np.asfortranarray(np.concatenate([inl[..., :5], part], axis=-1))
    sub = lambda a: np.ascontiguousarray(np.asarray(a)[idx])
    engines = []
    for e in (pkg.FlowSolver(cfg), oracle.Oracle(pkg, cfg)):
        e.set_mesh(*mesh, span)
        e.set_species(sub(mech.mi), n_tct=mech.n_tct, tct=mech.tct, tct_max=mech.tct_max, coef=sub(mech.coef))
        e.set_transport(sub(mech.viscosity), sub(mech.conductivity),
                        np.ascontiguousarray(np.asarray(mech.diffusion)[np.ix_(idx, idx)]))
        e.set_bc_jet(inl)
        e.upload_state(st)
        e.comput_flow_variables()
        e.OCFD_bc()
        for _ in range(2):
            e.flow_time_advance(info["dt"])
        engines.append(e)
    g, o = engines
    fc.compare_state(g, o)
    d, _ = fc.compare(fc.interior(g.download("DI")), fc.interior(o.download("DI")))
    assert d <= 1e-12, d
    g.close()
