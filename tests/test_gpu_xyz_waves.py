"""The wave kernels of the XYZ dGamma against the FP64 oracle, at the sizes
where their lane shapes and tile counts change.

States are random and obey no symmetry of a physical vertex, so an entry read
from the wrong row, site, component or exchange shows at full size.  The integer
mesh with cutoffs on mesh points makes frequency arguments vanish exactly.

Tolerance: an entry sums at most 3 (2 N_w + 8) points of 16 products of two
16-support interpolations, fewer than 1e6 terms with an error of 1.1e-16 of
their size each, of either sign; the terms exceed the largest entry by less
than 10, so 1e-10 of the largest entry bounds the difference of two summation
orders.
"""
import numpy as np
import pytest

from helpers import GOLDEN_RES, manual_task_xml, max_rel

pytestmark = pytest.mark.gpu

TOL = 1e-10
INTEGER_MESH = "1 2 3 4 6 8 12"
JK, J = {"j": 0.1, "k": -1.0}, {"j": 1.0}


def _problem(lattice, r, model, couplings, nw):
    from spinparser_amd.problem import xyz_problem
    from spinparser_amd.task import make_task_xml, parse_task
    if nw is None:
        xml = manual_task_xml(lattice, r, model, couplings, symmetry="XYZ", freqs=INTEGER_MESH)
    else:
        xml = make_task_xml(lattice=lattice, lattice_range=r, model=model, symmetry="XYZ", couplings=couplings,
                            freq_min=0.01, freq_max=20.0, freq_count=nw, cutoff_max=20.0, cutoff_min=0.05,
                            cutoff_step=0.9)
    return xyz_problem(parse_task(xml, True), GOLDEN_RES if lattice == "hyperhoneycomb" else None)


def _check(prob, cut, seed):
    from oracle import XyzOracle
    from spinparser_amd.capi import XyzFlowContext
    rng = np.random.default_rng(seed)
    v2 = rng.uniform(0.05, 0.3, prob.nw)
    v4 = rng.uniform(-1.0, 1.0, prob.vertex_size)
    r2, r4, _ = XyzOracle(prob).compute_step(cut, v2, v4, dtype=np.float64, nthreads=8)
    ctx = XyzFlowContext(prob)
    ctx.set_state(cut, v2, v4)
    _, s2, s4 = ctx.get_state()
    assert np.array_equal(s2, v2) and np.array_equal(s4, v4)
    ctx.compute_step()
    g2, g4 = ctx.get_flow()
    ctx.compute_step()  # adds to a cleared derivative each time
    again = ctx.get_flow()[1]
    ctx.close()
    e2, e4 = max_rel(g2, r2), max_rel(g4, r4)
    print("L=%d O=%d nw=%d cutoff %g: dSigma %.3g dGamma %.3g" % (prob.L, prob.overlap_total, prob.nw, cut, e2, e4),
          flush=True)
    assert e2 < TOL and e4 < TOL
    assert np.array_equal(g4, again)


@pytest.mark.parametrize("lattice,r,model,couplings,nw,cut", [
    ("triangular", 1, "triangular-heisenberg", J, 2, 0.3),   # 2 sites, the smallest mesh
    ("square", 3, "square-heisenberg", J, 9, 0.2),           # no spin permutations
    ("honeycomb", 3, "honeycomb-kitaev", JK, 12, 0.1),       # 5 sites
    ("honeycomb", 5, "honeycomb-kitaev", JK, 7, 0.1),        # 11 sites
    ("kagome", 5, "kagome-heisenberg", J, 6, 4.0),           # 19 sites
    ("honeycomb", 8, "honeycomb-kitaev", JK, 5, 0.1),        # 23 sites: 28 bubble tiles
    ("honeycomb", 9, "honeycomb-kitaev", JK, 4, 0.3),        # more than 28 tiles
    ("honeycomb", 11, "honeycomb-kitaev", JK, 3, 0.3),       # more than 32 sites: general kernels
])
def test_random_states(lattice, r, model, couplings, nw, cut):
    _check(_problem(lattice, r, model, couplings, nw), cut, 7)


@pytest.mark.parametrize("lattice,r,model,couplings", [
    ("square", 3, "square-heisenberg", J), ("hyperhoneycomb", 3, "hyperhoneycomb-kitaev", JK),
    ("honeycomb", 6, "honeycomb-kitaev", JK)])
@pytest.mark.parametrize("cut", [1.0, 2.0, 0.5, 12.0])
def test_vanishing_arguments(lattice, r, model, couplings, cut):
    _check(_problem(lattice, r, model, couplings, None), cut, 11)
