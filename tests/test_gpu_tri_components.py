"""Every component of the TRI dGamma to the precision of its own terms.

With e for a spin index, the components (d, d), (d, spin) and (spin, spin) are
given the sizes 1, e and e^2.  In every channel the terms of a component are then
no larger than its own power of e: a spin index of a product comes from at least
one spin index of the factors, and a density index costs nothing.  So a sum that
runs over the component's own terms has an error of a few 1e-16 of its size,
while one that mixes components (as a product of 4 x 4 matrices does) carries
1e-16 of the largest component, e^-2 times as much.

Tolerance: 1e-10 of the component's largest entry bounds the difference of two
orders of its sum (fewer than 1e7 terms, which exceed the largest entry by less
than 10); mixed components would leave 1e-16 / e^2 = 1e-8.
"""
import numpy as np
import pytest

from helpers import max_rel, tri_problem_of

pytestmark = pytest.mark.gpu

TOL = 1e-10
E = 1e-4


@pytest.mark.parametrize("lattice,r,model,couplings,nw,cut", [
    ("kagome", 3, "kagome-DM", {"j": 1.0, "d": 0.2}, 7, 0.3),
    ("honeycomb", 7, "honeycomb-kitaev", {"j": 0.1, "k": -1.0}, 5, 0.2),
    ("kagome", 7, "kagome-DM", {"j": 1.0, "d": 0.2}, 3, 0.3),  # general kernel
])
def test_components_of_different_size(lattice, r, model, couplings, nw, cut):
    from oracle import TriOracle
    from spinparser_amd.capi import TriFlowContext
    p = tri_problem_of(lattice, r, model, couplings, nw, 0.01, 20.0, 20.0, 0.05, 0.9)
    rng = np.random.default_rng(3)
    v2 = rng.uniform(0.05, 0.3, p.nw)
    size = E ** np.array([(c // 4 < 3) + (c % 4 < 3) for c in range(16)], dtype=float)
    v4 = rng.uniform(-1.0, 1.0, (p.n_freq, 16, p.L)) * size[None, :, None]
    ref = TriOracle(p).compute_step(cut, v2, v4.ravel(), dtype=np.float64, nthreads=8)[1].reshape(-1, 16, p.L)
    ctx = TriFlowContext(p)
    ctx.set_state(cut, v2, v4.ravel())
    ctx.compute_step()
    got = np.ravel(ctx.get_flow()[1]).reshape(-1, 16, p.L)
    ctx.close()
    errors = [max_rel(got[:, c], ref[:, c]) for c in range(16)]
    print("L=%d: largest error of a component %.3g" % (p.L, max(errors)), flush=True)
    for c in range(16):
        assert np.abs(ref[:, c]).max() < 1e7 * size[c]  # the premise: fewer than 1e7 terms of the component's size
        assert errors[c] < TOL, (c, errors[c])
