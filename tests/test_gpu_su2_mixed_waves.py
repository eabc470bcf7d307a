"""The wave kernels of the mixed SU(2) dGamma (FP32 vertex shadow and terms,
FP64 sums) against the FP64 oracle, at the sizes where their lane shapes change.

States are random and obey no symmetry of a physical vertex, so an entry read
from the wrong row, site or exchange shows at full size; the integer mesh with
cutoffs on mesh points makes frequency arguments vanish exactly.

Tolerance: a term goes through at most 16 FP32 roundings of 6e-8 (shadow,
weights, four supports of two bundles, products, weight of the point), 1e-6 of
its size; a sum of n such terms of either sign, which exceed the largest entry by
less than 10, is off by less than 1e-5 of the largest entry.
"""
import numpy as np
import pytest

from helpers import GOLDEN_RES, exp_problem, manual_task_xml, max_rel

pytestmark = pytest.mark.gpu

TOL = 1e-5
J, J12 = {"j": 1.0}, {"j1": 1.0, "j2": 0.3}


def _check(prob, cut, seed, scale=1.0):
    from oracle import Oracle
    from spinparser_amd.capi import SP_PRECISION_MIXED, FlowContext
    rng = np.random.default_rng(seed)
    v2 = rng.uniform(0.05, 0.3, prob.nw)
    ss, dd = (scale * rng.uniform(-1.0, 1.0, prob.vertex_size) for _ in range(2))
    ref = Oracle(prob).compute_step(cut, v2, ss, dd)
    ctx = FlowContext(prob, SP_PRECISION_MIXED)
    ctx.set_state(cut, v2, ss, dd)
    ctx.compute_step()
    got = ctx.get_flow()
    ctx.compute_step()
    again = ctx.get_flow()
    ctx.close()
    for name, g, a, r in zip(("dSigma", "dGamma spin", "dGamma density"), got, again, ref[:3]):
        err = max_rel(g, r)
        print("L=%d nw=%d cutoff %g %s: %.3g" % (prob.L, prob.nw, cut, name, err), flush=True)
        assert err < TOL
        assert np.array_equal(g, a)


@pytest.mark.parametrize("lattice,r,model,couplings,nw,cut", [
    ("triangular", 1, "triangular-heisenberg", J, 2, 0.3),  # 2 sites, the smallest mesh
    ("cubic", 3, "cubic-j1j2heisenberg", J12, 9, 0.2),      # 7 sites: half tile
    ("square", 4, "square-heisenberg", J, 17, 0.06),        # 9 sites: full tile
    ("cubic", 5, "cubic-j1j2heisenberg", J12, 6, 0.2),      # 16 sites
    ("kagome", 5, "kagome-heisenberg", J, 7, 0.1),          # 19 sites, bonds not equivalent to their reverse
    ("square", 7, "square-heisenberg", J, 8, 4.0),          # 20 sites: full and half tile
    ("cubic", 6, "cubic-j1j2heisenberg", J12, 5, 0.2),      # 23 sites
    ("kagome", 6, "kagome-heisenberg", J, 5, 0.1),          # two full tiles, not equivalent to the reverse
    ("cubic", 7, "cubic-j1j2heisenberg", J12, 5, 0.3),      # 31 sites
    ("cubic", 8, "cubic-j1j2heisenberg", J12, 4, 0.3),      # 41 sites: general kernel
])
def test_random_states(lattice, r, model, couplings, nw, cut):
    _check(exp_problem(lattice, r, model, couplings, nw, 0.01, 20.0, 20.0, 0.05, 0.9), cut, 7)


def test_scaled_shadow():
    """A shadow with a scale (2^14), the weights of the points within FP32."""
    _check(exp_problem("cubic", 6, "cubic-j1j2heisenberg", J12, 6, 0.01, 20.0, 20.0, 0.05, 0.9), 0.2, 5, 2.0 ** 30)


@pytest.mark.parametrize("lattice,r,model", [("square", 3, "square-heisenberg"),
                                             ("hyperkagome", 3, "hyperkagome-heisenberg"),
                                             ("kagome", 6, "kagome-heisenberg")])
@pytest.mark.parametrize("cut", [1.0, 2.0, 12.0])
def test_vanishing_arguments(lattice, r, model, cut):
    from spinparser_amd.problem import su2_problem
    from spinparser_amd.task import parse_task
    res = GOLDEN_RES if lattice == "hyperkagome" else None
    _check(su2_problem(parse_task(manual_task_xml(lattice, r, model, J, freqs="1 2 3 4 6 8 12"), True), res), cut, 11)
