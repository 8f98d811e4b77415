"""Cells with Et <= 0 in a step of several species, and what they cost on a
large grid.  The step's boundary kernel repairs them and does the faces; the
entries of a stage repair with a kernel of their own before the boundary
conditions.  Both do the same operations, so they agree bit for bit."""
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


def spoil(g, cells, F=None):
    """The solution's internal energy takes the other sign at the cells.  The
    primitives are kept, so every stage starts from sound fluxes and the first
    two meet Et <= 0 there."""
    F = g.download("F") if F is None else F.copy(order="F")
    for c in cells:
        d, mu, mv, mw, E = F[c]
        ke = 0.5 * (mu * mu + mv * mv + mw * mw) / d
        F[c][4] = 2.0 * ke - E
    g.upload("F", F)


# beside the inflow, on an edge, in a corner, in the middle of a k face, inside
@pytest.mark.parametrize("n", [(20, 12, 10), (75, 37, 38)])
@pytest.mark.parametrize("iflag", [1, 0])
def test_jet_step_with_bad_cells(pkg, n, iflag):
    case = fc.small_jet(*n, iflag=iflag)
    nx, ny, nz = n
    cells = [(1, 5, 3), (nx - 2, ny - 1, 0), (nx - 1, 0, nz - 1), (nx // 2, ny // 2, 0), (nx // 2, ny // 2, nz - 1),
             (10, 5, 5), (11, 5, 5)]
    dt, ns = 0.2 * case[5]["dt"], case[0].n_spec
    a = pkg.FlowSolver(case[0])
    fc.setup_jet(a, case)
    spoil(a, cells)
    a.flow_time_advance(dt)
    assert a.negative_et_count() > 0
    names = ("F", "DI", "D", "U", "V", "W", "T", "P", "ET")
    fa = {k: a.download(k) for k in names}
    a.close()
    b = pkg.FlowSolver(case[0])
    fc.setup_jet(b, case)
    spoil(b, cells)
    b.save_stage0()
    counts = []
    for krk in (1, 2, 3):
        b.stage_begin(krk)
        b.Scalar_time_adv_RK3(krk, dt)
        b.du_inviscous()
        b.du_viscous()
        b.OCFD_time_adv_RK3(krk, dt)
        b.comput_flow_variables()
        counts.append(b.negative_et_count())
        b.OCFD_bc()
    assert counts[0] >= len(cells) - 2, counts  # a face's cells may be set by the conditions
    for k, v in fa.items():
        assert np.isfinite(v).all() and v.tobytes() == b.download(k).tobytes(), k
    b.close()


def test_bad_cell_leaves_the_faces_parallel(pkg):
    """One bad cell costs a stage its repair, a chain of some thirty dependent
    loads (at most 2 us each) and a wait, but not the parallel treatment of
    the faces: less than 0.1 ms more in the boundary kernel, where a single
    block for all of this grid's faces takes many times that."""
    case = fc.small_flat_plate(256, 96, 64)
    g = pkg.FlowSolver(case[0])
    fc.setup(g, case)
    F = g.download("F")
    ms = []
    for cells in ((), ((100, 40, 20),)):
        t = []
        for _ in range(3):
            spoil(g, cells, F)
            g.set_option(pkg.OPT_KERNEL_TIMING, 1)
            g.kernel_stats_reset()
            g.flow_time_advance(0.2 * case[5]["dt"])
            total, launches = g.kernel_stats()["k_bc"]
            assert launches == 3 and g.negative_et_count() == len(cells)
            t.append(total / launches)
        ms.append(min(t))
    print("boundary kernel, ms a launch without and with a bad cell:", ms)
    assert ms[1] < ms[0] + 0.1, ms
    g.close()
