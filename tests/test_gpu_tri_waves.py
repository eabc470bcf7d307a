"""The wave kernels of the TRI dGamma against the FP64 oracle, at the sizes
where their lane shapes, waves per item and product counts change.

States are random and obey no symmetry of a physical vertex, so an entry read
from the wrong row, site, component or exchange shows at full size.  The integer
mesh with cutoffs on mesh points makes frequency arguments vanish exactly.

Tolerance: an entry sums at most 3 (2 N_w + 8) points of 256 products of two
16-support interpolations and the overlap terms, fewer than 1e7 terms with an
error of 1.1e-16 of their size each, of either sign; the terms exceed the
largest entry by less than 10, so 1e-10 of the largest entry bounds the
difference of two summation orders.
"""
import numpy as np
import pytest

from helpers import GOLDEN_RES, manual_task_xml, max_rel

pytestmark = pytest.mark.gpu

TOL = 1e-10
INTEGER_MESH = "1 2 3 4 6 8 12"
DM, JK, JKG, J = {"j": 1.0, "d": 0.2}, {"j": 0.1, "k": -1.0}, {"j": 0.2, "k": 1.0, "g": -0.1}, {"j": 1.0}


def _problem(lattice, r, model, couplings, nw):
    from spinparser_amd.problem import tri_problem
    from spinparser_amd.task import make_task_xml, parse_task
    if nw is None:
        xml = manual_task_xml(lattice, r, model, couplings, symmetry="TRI", freqs=INTEGER_MESH)
    else:
        xml = make_task_xml(lattice=lattice, lattice_range=r, model=model, symmetry="TRI", couplings=couplings,
                            freq_min=0.01, freq_max=20.0, freq_count=nw, cutoff_max=20.0, cutoff_min=0.05,
                            cutoff_step=0.9)
    return tri_problem(parse_task(xml, True), GOLDEN_RES if model == "honeycomb-kitaev-gamma" else None)


def _check(prob, cut, seed):
    from oracle import TriOracle
    from spinparser_amd.capi import TriFlowContext
    rng = np.random.default_rng(seed)
    v2 = rng.uniform(0.05, 0.3, prob.nw)
    v4 = rng.uniform(-1.0, 1.0, prob.vertex_size)
    r2, r4, _ = TriOracle(prob).compute_step(cut, v2, v4, dtype=np.float64, nthreads=8)
    ctx = TriFlowContext(prob)
    ctx.set_state(cut, v2, v4)
    _, s2, s4 = ctx.get_state()
    assert np.array_equal(s2, v2) and np.array_equal(np.ravel(s4), v4)
    ctx.compute_step()
    g2, g4 = ctx.get_flow()
    ctx.compute_step()  # adds to a cleared derivative each time
    again = ctx.get_flow()[1]
    ctx.close()
    e2, e4 = max_rel(g2, r2), max_rel(np.ravel(g4), np.ravel(r4))
    print("L=%d O=%d nw=%d cutoff %g: dSigma %.3g dGamma %.3g" % (prob.L, prob.overlap_total, prob.nw, cut, e2, e4),
          flush=True)
    assert e2 < TOL and e4 < TOL
    assert np.array_equal(g4, again)


@pytest.mark.parametrize("lattice,r,model,couplings,nw,cut", [
    ("honeycomb", 1, "honeycomb-kitaev", JK, 3, 0.4),
    ("honeycomb", 2, "honeycomb-kitaev", JK, 9, 0.7),
    ("honeycomb", 3, "honeycomb-kitaev-gamma", JKG, 11, 0.05),
    ("kagome", 3, "kagome-DM", DM, 8, 0.3),
    ("kagome", 4, "kagome-DM", DM, 7, 2.0),
    ("honeycomb", 5, "honeycomb-kitaev", JK, 7, 0.2),
    ("kagome", 5, "kagome-DM", DM, 6, 0.1),
    ("honeycomb", 7, "honeycomb-kitaev", JK, 5, 0.3),
    ("kagome", 6, "kagome-heisenberg", J, 5, 0.5),
])
def test_shapes(lattice, r, model, couplings, nw, cut):
    _check(_problem(lattice, r, model, couplings, nw), cut, 7)


@pytest.mark.parametrize("cut", [1.0, 2.0, 0.5])
@pytest.mark.parametrize("lattice,r,model,couplings", [("honeycomb", 3, "honeycomb-kitaev", JK),
                                                       ("kagome", 3, "kagome-DM", DM)])
def test_arguments_of_zero(lattice, r, model, couplings, cut):
    _check(_problem(lattice, r, model, couplings, None), cut, 11)
