"""The wave kernels of the FP64 SU(2) dGamma (S and U evaluated once for two
items, one gather per T pair, the lattice bubble on the matrix cores) against
the FP64 oracle, at the sizes where their lane shapes change.

States are random and obey no symmetry of a physical vertex, so an entry that
is read from the wrong row, site or exchange shows at full size; in particular
the density entries with equal outer frequencies, which flows keep small, are
not small.  The integer mesh with cutoffs on mesh points makes frequency
arguments vanish exactly and fall exactly on mesh points.

Tolerance: an entry sums at most 3 (2 N_w + 8) points of 4 products of two
16-support interpolations, fewer than 1e5 terms with an error of 1.1e-16 of
their size each; the terms exceed the largest entry by less than 10, so 1e-10
of the largest entry bounds the difference of two summation orders.
"""
import numpy as np
import pytest

from helpers import GOLDEN_RES, cfg1_problem, exp_problem, manual_task_xml, max_rel, ref1_problem

pytestmark = pytest.mark.gpu

TOL = 1e-10
INTEGER_MESH = "1 2 3 4 6 8 12"


def _integer(lattice, r, model, couplings):
    from spinparser_amd.problem import su2_problem
    from spinparser_amd.task import parse_task
    res = GOLDEN_RES if lattice == "hyperkagome" else None
    return su2_problem(parse_task(manual_task_xml(lattice, r, model, couplings, freqs=INTEGER_MESH), True), res)


def _exp(lattice, r, model, couplings, nw):
    return exp_problem(lattice, r, model, couplings, nw, 0.01, 20.0, 20.0, 0.05, 0.9)


J, J12 = {"j": 1.0}, {"j1": 1.0, "j2": 0.3}
CASES = [
    ("triangular", 1, "triangular-heisenberg", J, 2, 0.3),     # 2 sites, the smallest mesh
    ("square", 2, "square-heisenberg", J, 5, 0.3),
    ("cubic", 3, "cubic-j1j2heisenberg", J12, 9, 0.2),         # 7 sites: half tile
    ("square", 4, "square-heisenberg", J, 17, 0.06),           # 9 sites: full tile
    ("cubic", 5, "cubic-j1j2heisenberg", J12, 6, 0.2),         # 16 sites
    ("kagome", 5, "kagome-heisenberg", J, 7, 0.1),             # 19 sites, bonds not equivalent to their reverse
    ("square", 7, "square-heisenberg", J, 8, 4.0),             # 20 sites: full and half tile
    ("cubic", 6, "cubic-j1j2heisenberg", J12, 5, 0.2),         # 23 sites
    ("kagome", 6, "kagome-heisenberg", J, 5, 0.1),             # two full tiles, not equivalent to the reverse
    ("cubic", 7, "cubic-j1j2heisenberg", J12, 5, 0.3),         # 31 sites
    ("cubic", 8, "cubic-j1j2heisenberg", J12, 4, 0.3),         # 41 sites: general kernel
]


def _check(prob, cut, seed):
    from oracle import Oracle
    from spinparser_amd.capi import FlowContext
    rng = np.random.default_rng(seed)
    v2 = rng.uniform(0.05, 0.3, prob.nw)
    ss, dd = rng.uniform(-1.0, 1.0, prob.vertex_size), rng.uniform(-1.0, 1.0, prob.vertex_size)
    ref = Oracle(prob).compute_step(cut, v2, ss, dd)
    ctx = FlowContext(prob)
    ctx.set_state(cut, v2, ss, dd)
    ctx.compute_step()
    got = ctx.get_flow()
    ctx.compute_step()  # adds to a cleared derivative each time
    again = ctx.get_flow()
    ctx.close()
    for name, g, a, r in zip(("dSigma", "dGamma spin", "dGamma density"), got, again, ref[:3]):
        err = max_rel(g, r)
        print("L=%d nw=%d cutoff %g %s: %.3g" % (prob.L, prob.nw, cut, name, err), flush=True)
        assert err < TOL
        assert np.array_equal(g, a)


@pytest.mark.parametrize("lattice,r,model,couplings,nw,cut", CASES)
def test_random_states(lattice, r, model, couplings, nw, cut):
    _check(_exp(lattice, r, model, couplings, nw), cut, 7)


@pytest.mark.parametrize("lattice,r,model,couplings", [
    ("square", 3, "square-heisenberg", J), ("hyperkagome", 3, "hyperkagome-heisenberg", J),
    ("kagome", 5, "kagome-heisenberg", J), ("kagome", 6, "kagome-heisenberg", J)])
@pytest.mark.parametrize("cut", [1.0, 2.0, 0.5, 12.0])
def test_vanishing_arguments(lattice, r, model, couplings, cut):
    _check(_integer(lattice, r, model, couplings), cut, 11)


def test_group_of_shapes():
    """Flows of several lane shapes and a larger lattice in one group step, each
    equal to the same flow alone."""
    from spinparser_amd.capi import FlowContext, FlowGroup
    probs = [cfg1_problem(nw=9), ref1_problem(), _exp("cubic", 6, "cubic-j1j2heisenberg", J12, 6),
             _exp("cubic", 7, "cubic-j1j2heisenberg", J12, 7), _exp("cubic", 8, "cubic-j1j2heisenberg", J12, 4),
             cfg1_problem(nw=10)]
    flows, alone = [], []
    for p in probs:
        for out in (flows, alone):
            c = FlowContext(p)
            c.set_state(float(p.cutoffs[0]), *p.initial_state(np.float64))
            out.append(c)
    group = FlowGroup(len(probs))
    for k in range(3):
        cuts = [float(p.cutoffs[k + 1]) for p in probs]
        group.step(flows, cuts)
        for c, new in zip(alone, cuts):
            c.compute_step()
            c.finalize_step(new)
    for a, b in zip(flows, alone):
        for x, y in zip(a.get_state()[1:], b.get_state()[1:]):
            assert np.array_equal(x, y)
        a.close()
        b.close()
    group.close()
