"""Which kernels the host code launches, on the CPU (fake_hip.cpp's log)."""
import pytest

import fakehip


def launches(code, elapsed=""):
    return [ln[1] for ln in fakehip.run(code, elapsed) if ln[0] == "launch"]


@pytest.mark.parametrize("n,marching", [(16, False), (80, False), (81, True)])
def test_stage_entries_march_on_large_grids_only(n, marching):
    """The stage entries of a grid of up to 2^19 cells take one thread per
    cell: the marching kernels fill too few of the chip's wavefronts."""
    names = launches(f"""
g = pkg.FlowSolver(fc.small_isotropic({n})[0])
g.du_viscous()
g.close()
""")
    prep = [k for k in names if "k_visc_prep" in k]
    rk = [k for k in names if "k_rk" in k]
    assert len(prep) == 1 and len(rk) == 1
    assert ("k_visc_prep_col" in prep[0]) == marching and ("k_rk_col" in rk[0]) == marching


@pytest.mark.parametrize("before,one_launch", [("g.autotune(3)", True), ("g.set_tile(1, 2)", False),
                                               ("g.set_tile(1, 2); g.set_tile(1, 0)", True),
                                               ("g.set_tile(1, 2); g.autotune(3)", True)])
@pytest.mark.parametrize("again", [False, True])
def test_tuner_leaves_the_small_stage_on(before, one_launch, again):
    """A tile shape that the tuner finds faster by itself (the second of each
    direction here, by far) does not take a small grid off its one-launch
    stage, in this context or the next; a shape asked for by ocfd_set_tile
    does."""
    names = launches(f"""
g = pkg.FlowSolver(fc.small_isotropic(16)[0])
{before}
if {again}:
    g.close()
    g = pkg.FlowSolver(fc.small_isotropic(20)[0])
print([g.tile_choice(d) for d in range(3)])
g.flow_time_advance(1e-9)
g.close()
""", elapsed="1.0,0.1,1.0,1.0")
    step = names[max(i for i, k in enumerate(names) if "k_fill" in k) + 1:]
    assert sum("k_stage" in k for k in step) == (3 if one_launch else 0)
