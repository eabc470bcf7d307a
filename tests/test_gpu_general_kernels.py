"""The general dGamma kernels of the TRI and XYZ cores on lattices of at most 32
sites, against the FP64 oracle.  The wave kernels take such a lattice only if its
site tables have the form that a lattice of the factory has and if its distinct
products fit; here the tables are others (sites and spin components mapped by
random tables, which neither the general kernels nor the oracle restrict), or the
products are too many (TRI, honeycomb-Kitaev of range 8 and 9).

The TRI cases have one lattice for each workgroup shape of its 128-thread kernel:
site stride and points per chunk compiled in for 13 to 32 sites, read at run time
below.

States are random.  Tolerance: an entry sums fewer than 1e7 terms with an error
of 1.1e-16 of their size each, of either sign; the terms exceed the largest entry
by less than 10, so 1e-10 of the largest entry bounds the difference of two
summation orders.
"""
import dataclasses

import numpy as np
import pytest

from helpers import max_rel, tri_problem_of

pytestmark = pytest.mark.gpu

TOL = 1e-10
DM, JK, J = {"j": 1.0, "d": 0.2}, {"j": 0.1, "k": -1.0}, {"j": 1.0}


def _xyz_problem(lattice, r, model, couplings, nw):
    from spinparser_amd.problem import xyz_problem
    from spinparser_amd.task import make_task_xml, parse_task
    return xyz_problem(parse_task(make_task_xml(
        lattice=lattice, lattice_range=r, model=model, symmetry="XYZ", couplings=couplings, freq_min=0.01,
        freq_max=20.0, freq_count=nw, cutoff_max=20.0, cutoff_min=0.05, cutoff_step=0.9), True))


def _tri_problem(lattice, r, model, couplings, nw):
    return tri_problem_of(lattice, r, model, couplings, nw, 0.01, 20.0, 20.0, 0.05, 0.9)


def _other_tables(prob, seed):
    """The problem with site tables of no particular form."""
    rng = np.random.default_rng(seed)

    def perms(n):
        return np.array([rng.permutation(3) for _ in range(n)], dtype=np.int32)

    site = rng.permutation(prob.L).astype(np.int32)
    inv = rng.integers(0, prob.L, prob.L).astype(np.int32)
    inv[:2] = 1  # not one-to-one
    return dataclasses.replace(prob, site_rid=site, site_perm=perms(prob.L), inv_rid=inv, inv_perm=perms(prob.L))


def _check(prob, context, oracle, cut):
    rng = np.random.default_rng(9)
    v2 = rng.uniform(0.05, 0.3, prob.nw)
    v4 = rng.uniform(-1.0, 1.0, prob.vertex_size)
    r2, r4, _ = oracle(prob).compute_step(cut, v2, v4, dtype=np.float64, nthreads=8)
    ctx = context(prob)
    ctx.set_state(cut, v2, v4)
    _, s2, s4 = ctx.get_state()
    assert np.array_equal(s2, v2) and np.array_equal(np.ravel(s4), v4)
    ctx.compute_step()
    g2, g4 = ctx.get_flow()
    ctx.close()
    e2, e4 = max_rel(g2, r2), max_rel(np.ravel(g4), np.ravel(r4))
    print("L=%d O=%d: dSigma %.3g dGamma %.3g" % (prob.L, prob.overlap_total, e2, e4), flush=True)
    assert e2 < TOL and e4 < TOL


@pytest.mark.parametrize("lattice,r,model,couplings,nw,L", [
    ("kagome", 3, "kagome-DM", DM, 5, 8), ("kagome", 4, "kagome-DM", DM, 4, 13),
    ("triangular", 7, "triangular-heisenberg", J, 4, 20), ("cubic", 6, "cubic-heisenberg", J, 4, 23),
    ("kagome", 6, "kagome-DM", DM, 4, 26), ("cubic", 7, "cubic-heisenberg", J, 3, 31)])
def test_tri_other_tables(lattice, r, model, couplings, nw, L):
    from oracle import TriOracle
    from spinparser_amd.capi import TriFlowContext
    prob = _tri_problem(lattice, r, model, couplings, nw)
    assert prob.L == L
    _check(_other_tables(prob, 4), TriFlowContext, TriOracle, 0.3)


@pytest.mark.parametrize("r,L", [(8, 23), (9, 28)])
def test_tri_many_products(r, L):
    from oracle import TriOracle
    from spinparser_amd.capi import TriFlowContext
    prob = _tri_problem("honeycomb", r, "honeycomb-kitaev", JK, 4)
    assert prob.L == L
    _check(prob, TriFlowContext, TriOracle, 0.3)


@pytest.mark.parametrize("bubble", ["rank-update", "direct"])
@pytest.mark.parametrize("lattice,r,model,couplings,nw", [
    ("honeycomb", 3, "honeycomb-kitaev", JK, 9), ("kagome", 4, "kagome-heisenberg", J, 6),
    ("honeycomb", 8, "honeycomb-kitaev", JK, 4)])
def test_xyz_other_tables(lattice, r, model, couplings, nw, bubble, monkeypatch):
    from oracle import XyzOracle
    from spinparser_amd.capi import XyzFlowContext
    if bubble == "direct":
        monkeypatch.setenv("SPFRG_XYZ_BUBBLE", "direct")
    _check(_other_tables(_xyz_problem(lattice, r, model, couplings, nw), 4), XyzFlowContext, XyzOracle, 0.3)
