"""The transport coefficients of several species for every combination of the
transport flags and both gas models against the oracle: viscosity,
conductivity (with Flag_Conductivity = 0 from the mixture's Cp, in either
temperature range and above the fits' range) and diffusion, and a step."""
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


@pytest.mark.parametrize("real", [0, 1])
@pytest.mark.parametrize("flags", [(v, c, d) for v in (0, 1) for c in (0, 1) for d in (0, 1)])
@pytest.mark.parametrize("ns", [9, 3])
def test_flags(pkg, real, flags, ns):
    import oracle
    cfg, mesh, span, st, bc, info = fc.small_jet(20, 12, 10)
    mech = info["mech"]
    idx = list(range(9)) if ns == 9 else [1, 2, 8]
    cfg.n_spec, cfg.if_real_gas = ns, real
    cfg.flag_vis, cfg.flag_cond, cfg.flag_diff = flags
    sub = lambda a: np.ascontiguousarray(np.asarray(a)[idx])
    di = np.asarray(st["DI"])[..., idx]
    st = dict(st, DI=np.asfortranarray(di * (np.asarray(st["D"]) / di.sum(-1))[..., None]))
    inl = np.asarray(bc["inlet2d"])
    part = inl[..., [5 + k for k in idx]]
    inl = np.asfortranarray(np.concatenate([inl[..., :5], part * (inl[..., 0] / part.sum(-1))[..., None]], axis=-1))
    g, o = pkg.FlowSolver(cfg), oracle.Oracle(pkg, cfg)
    for e in (g, o):
        e.set_mesh(*mesh, span)
        e.set_species(sub(mech.mi), n_tct=mech.n_tct, tct=mech.tct, tct_max=mech.tct_max, coef=sub(mech.coef))
        e.set_transport(sub(mech.viscosity), sub(mech.conductivity),
                        np.ascontiguousarray(np.asarray(mech.diffusion)[np.ix_(idx, idx)]))
        e.set_bc_jet(inl)
        e.upload_state(st)
        e.comput_flow_variables()
        e.OCFD_bc()
        # some cells above the fits' range (5000 K)
        T = e.download("T")
        T[8:12, 8, 8] = 5600.0
        e.upload("T", T)
        e.comput_Amu_Amk_AMD()
    # the coefficients take a few exponentials and a logarithm each: 1e-12 of a cell's own value
    for name in ("AMU", "AMK"):
        a, b = g.download(name), o.download(name)
        assert np.max(np.abs(a - b) / np.abs(b)) <= 1e-12, name
    a, b = g.download("AMD"), o.download("AMD")
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))
    for e in (g, o):
        e.flow_time_advance(0.2 * info["dt"])
    fc.compare_state(g, o)
    g.close()
