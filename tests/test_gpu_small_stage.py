"""The one-launch stage of small N_SPEC = 1 grids against the separate
launches that larger grids take (OPT_COLUMN_PLANES >= 0 selects them on any
grid).  Both add the same terms in the same order, so everything is equal bit
for bit: the solution, the saved stage, the inviscid right-hand side that is
left in DU, the masks and the sensor."""
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


def box(n, **kw):
    def make():
        case = fc.small_isotropic(n, **{k: v for k, v in kw.items() if k != "cfg"})
        for k, v in kw.get("cfg", {}).items():
            setattr(case[0], k, v)
        return case
    return make


CASES = {
    "box_8": (box(8), 0, 0),                                  # one tile a direction
    "box_17_graph": (box(17, scheme_invis=3), 0, 1),          # a remainder tile
    "box_33_cd8": (box(33, cfg=dict(scheme_vis=6)), 0, 1),    # a second tile of one cell
    "box_16_mass": (box(16, cfg=dict(if_mass_force=1, mass_force=(0.3, -0.2, 0.1))), 0, 0),
    "plate_37x29x9": (lambda: fc.small_flat_plate(37, 29, 9), 1, 1),
    "plate_65x32x8_tables": (lambda: fc.small_flat_plate(65, 32, 8), 0, 0),
    "box_80": (box(80), 0, 0),                                # 512,000 cells: just below the line
    "box_81": (box(81), 0, 0),                                # 531,441: just above it
}


@pytest.mark.parametrize("name", list(CASES))
def test_one_launch_equals_separate_launches(pkg, name):
    make, sum_mode, graph = CASES[name]
    case = make()
    dt = 0.5 * case[5]["dt"]
    runs = []
    for planes in (-1, 0):
        g = pkg.FlowSolver(case[0])
        fc.setup(g, case)
        g.set_option(pkg.OPT_HYBRID_SUM_MODE, sum_mode)
        g.set_option(pkg.OPT_USE_GRAPH, graph)
        g.set_option(pkg.OPT_METRIC_TABLES, int("tables" in name))
        g.set_option(pkg.OPT_COLUMN_PLANES, planes)
        out = []
        for step in range(3):
            g.flow_time_advance(dt)
            if step == 1:
                out.append(g.download("DU"))
        for f in ("DU", "F", "FN", "DI", "D", "U", "V", "W", "T", "P", "ET", "RHYBRID"):
            out.append(g.download(f))
        # the stage entry points read DU after a step
        g.du_viscous()
        out.append(g.download("DU"))
        g.OCFD_time_adv_RK3(2, dt)
        out.append(g.download("F"))
        out.extend(g.download_mask(d) for d in range(3))
        g.close()
        runs.append(out)
    for a, b in zip(*runs):
        assert np.isfinite(a).all()
        assert a.tobytes() == b.tobytes()


@pytest.mark.parametrize("kind", ["plate", "box"])
@pytest.mark.parametrize("planes", [-1, 0])
def test_step_with_bad_cells(pkg, kind, planes):
    """A step whose stages meet Et <= 0: the boundary kernel's first block
    repairs the cells and then does every face, as the oracle does."""
    import oracle
    if kind == "plate":
        case, cells = fc.small_flat_plate(37, 29, 9), [(1, 5, 3), (20, 10, 0), (35, 14, 8), (18, 27, 4), (18, 12, 4)]
    else:
        case, cells = fc.small_isotropic(16), [(0, 0, 0), (7, 8, 9), (15, 3, 0)]
    g, o = pkg.FlowSolver(case[0]), oracle.Oracle(pkg, case[0])
    g.set_option(pkg.OPT_COLUMN_PLANES, planes)
    for e in (g, o):
        fc.setup(e, case)
        F = e.download("F")
        for c in cells:  # nearly no internal energy, and a step far too long
            d, mu, mv, mw, E = F[c]
            ke = 0.5 * (mu * mu + mv * mv + mw * mw) / d
            F[c][4] = ke + (E - ke) * 1e-3
        e.upload("F", F)
        e.comput_flow_variables()
        e.OCFD_bc()
    counts = []
    for _ in range(2):
        for e in (g, o):
            e.flow_time_advance(8.0 * case[5]["dt"])
        counts.append((g.negative_et_count(), o.negative_et_count()))
    # the library reports the largest count of a step's stages, the oracle its last stage's
    assert counts[1][1] > 0 and all(a >= b for a, b in counts), counts
    rep = fc.compare_state(g, o, tol=0.0)
    assert all(v[1] == 1.0 for v in rep.values()), rep
    g.close()
