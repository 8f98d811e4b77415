"""The device's species bank always has the context's species count: the
species loops of the kernels write that many partial densities, so a count
left by an earlier, larger context would reach past DI.  On the CPU
(fake_hip.cpp logs the first word of every upload of the bank, its count)."""
import fakehip

CODE = """
from ocfd_amd import cases
cfg, mesh, span, st, bc, info = fc.small_jet(12, 10, 9)
g = pkg.FlowSolver(cfg)
cases.jet_gas(g, info["mech"])
g.close()
for ns in {later}:
    cfg.n_spec = ns
    cfg.if_real_gas = cfg.flag_vis = cfg.flag_cond = cfg.flag_diff = 0
    cfg.ibc = 0 if ns == 1 else cfg.ibc
    g = pkg.FlowSolver(cfg)
    if ns > 1:
        g.OCFD_bc()
    g.close()
    cfg.ibc = pkg.BC_JET
"""


def counts(later):
    """The bank's count at each boundary launch of a multi-species context."""
    now, seen = 0, []
    for ln in fakehip.run(CODE.format(later=later)):
        if ln[0] == "symbol" and ln[1] == "fg":
            now = int(ln[3])
        elif ln[0] == "launch" and "k_bc" in ln[1]:
            seen.append(now)
    return seen


def test_bank_follows_the_context():
    assert counts((2, 1, 3, 9)) == [2, 3, 9]
