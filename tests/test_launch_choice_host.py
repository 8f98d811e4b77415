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
