"""ocfd_init's allocations and fills, on the CPU (fake_hip.cpp): every fill
stays inside its allocation, and the boundary-layer data's covers all of it,
for every kind of inlet and upper data."""
import pytest

import fakehip

CASES = [("fc.small_isotropic(8)[0]", 0, 0)] + [("fc.small_flat_plate(24, 16, 9)[0]", ki, ku)
                                               for ki in (0, 1, 2) for ku in (-1, 0, 1, 2)]


@pytest.mark.parametrize("cfg,ki,ku", CASES)
def test_fills_stay_inside_their_allocations(cfg, ki, ku):
    log = fakehip.run(f"""
cfg = {cfg}
cfg.bc_para[0], cfg.bc_para[1] = {ki}, {ku}
pkg.FlowSolver(cfg).close()
""")
    assert not [ln for ln in log if ln[0] == "fault"], [ln for ln in log if ln[0] == "fault"]
    fills = [tuple(int(x) for x in ln[1:]) for ln in log if ln[0] == "fill"]
    by_size = {}
    for off, n, size in fills:
        by_size.setdefault(size, []).append((off, n))
    nx, ny, nz = (8, 8, 8) if "isotropic" in cfg else (24, 16, 9)
    inlet = {0: 1, 1: ny, 2: ny * nz}[ki] if nx == 24 else 1
    upper = {-1: 1, 0: 1, 1: nx, 2: nx * nz}[ku] if nx == 24 else 1
    n = 6 * inlet + 6 * upper + nx * nz
    assert by_size.get(8 * n) == [(0, n)], (n, by_size)
