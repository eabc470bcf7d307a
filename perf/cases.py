"""The work a user of this engine has it do, as timed cases.

A pf-FRG run is a cutoff loop: evaluate dSigma/dLambda and dGamma/dLambda at
the present cutoff, measure the static correlations, check for divergence, take
the Euler step.  The cases cover the calls that make up such runs:

* "step": one FP64 SU(2) derivative evaluation on a state that lives on the
  device (``sp_compute_step_noalloc``), from the smallest lattice to the
  64-frequency simple cubic one, at the ends of the cutoff schedule (few and
  many integration points per frequency triple);
* "flow": whole runs of one resident flow through its context, for the three
  cores SU(2), XYZ and TRI and the mixed-precision SU(2) form: state upload,
  the loop over the cutoff schedule, the final state and every record.  The
  larger ones use a coarser cutoff grid (larger Euler steps) than the production
  schedules of the same lattices, over the same range of cutoffs;
* "core": the small multi-sublattice runs through the ``FrgCore`` classes,
  driven the way the cutoff loop of a task file drives them;
* "sweep": a served parameter sweep, many flows of different sizes resident
  together, in the mixed form with the precision schedule.

Seeds change the couplings (flows) or the vertex and self-energy (steps), never
the sizes.  Evaluation points per integral depend on the cutoff and the mesh
alone, so the work of a case is the same for every seed.
"""
import ctypes
import dataclasses
import functools
import math
import random

import numpy as np
import torch

from spinparser_amd.capi import (SP_PRECISION_FP64, SP_PRECISION_MIXED, FlowContext, ProblemBuffers, SpSu2Problem,
                                 TriFlowContext, XyzFlowContext, load_library)
from spinparser_amd.frgcore import FrgCoreFactory
from spinparser_amd.lattice import LatticeUnitCell, SpinModelUnitCell, model_couplings, new_lattice_model
from spinparser_amd.problem import su2_problem_from_lattice, tri_problem_from_lattice, xyz_problem_from_lattice
from spinparser_amd.serve import FlowRequest, PrecisionSchedule, SweepServer
from spinparser_amd.task import MeasurementSpec, exponential_cutoffs, exponential_mesh
from spinparser_amd.workload import channel_calls

# the 14-point mesh and the cutoff schedule of the reference's scripted runs
MANUAL_MESH = (0.31812, 0.36329, 0.41812, 0.46329, 0.51334, 0.56880, 0.63024, 0.69833, 0.77378, 0.85737, 0.95, 1.0,
               3.0, 10.0)
GOLDEN_RESOURCES = "tests/golden/res"  # hyperkagome, hyperhoneycomb and Gamma models, in the resource schema

# coupling of the seed-independent part, and its relative spread over seeds
MODELS = {
    "square-heisenberg": {"j": 1.0}, "triangular-heisenberg": {"j": 1.0}, "honeycomb-heisenberg": {"j": 1.0},
    "kagome-heisenberg": {"j": 1.0}, "cubic-j1j2heisenberg": {"j1": 1.0, "j2": 0.3},
    "honeycomb-kitaev": {"j": 0.1, "k": -1.0}, "kagome-DM": {"j": 1.0, "d": 0.2},
    "hyperkagome-heisenberg": {"j": 1.0}, "hyperhoneycomb-kitaev": {"j": 0.1, "k": -1.0},
    "honeycomb-kitaev-gamma": {"j": 0.2, "k": 1.0, "g": -0.1},
}
SPREAD = 0.05


def listed():
    return [
        # the smallest evaluation: 288 frequency triples, bound by launches and the call itself
        dict(name="su2-step-square-nw8", kind="step", lattice="square", range=4, model="square-heisenberg", nw=8,
             fmin=0.005, fmax=50.0, cutoff=0.9),
        # one evaluation of the 64-frequency cubic J1-J2 flow near its start (few integration points per triple)
        dict(name="su2-step-cubic-high", kind="step", lattice="cubic", range=6, model="cubic-j1j2heisenberg", nw=64,
             fmin=0.002, fmax=100.0, cutoff=60.0),
        # and near its end (all integration windows open)
        dict(name="su2-step-cubic-low", kind="step", lattice="cubic", range=6, model="cubic-j1j2heisenberg", nw=64,
             fmin=0.002, fmax=100.0, cutoff=0.02),
        # the CPU-sized square-lattice run, its whole production schedule (421 evaluations) queued in one call
        dict(name="su2-flow-square", kind="flow", core="SU2", lattice="square", range=4, model="square-heisenberg",
             nw=32, fmin=0.005, fmax=50.0, cmax=50.0, cmin=0.01, cstep=0.98, queued=True),
        # a run on the largest lattice of the J2/J1 sweep (31 sites) with an odd number of frequencies
        dict(name="su2-flow-cubic", kind="flow", core="SU2", lattice="cubic", range=7, model="cubic-j1j2heisenberg",
             nw=45, fmin=0.002, fmax=100.0, cmax=100.0, cmin=0.005, cstep=0.8),
        # the mixed-precision form over the cutoffs the precision schedule gives it (down to three times J)
        dict(name="su2-mixed-cubic", kind="flow", core="SU2", lattice="cubic", range=6, model="cubic-j1j2heisenberg",
             nw=48, fmin=0.002, fmax=100.0, cmax=100.0, cmin=3.0, cstep=0.9, mixed=True),
        # the scripted 14-frequency runs: lattices without an inversion that swaps a bond's ends, a manual mesh
        dict(name="su2-core-hyperkagome", kind="core", core="SU2", lattice="hyperkagome", range=3,
             model="hyperkagome-heisenberg"),
        dict(name="xyz-core-hyperhoneycomb", kind="core", core="XYZ", lattice="hyperhoneycomb", range=3,
             model="hyperhoneycomb-kitaev"),
        # the XYZ core at its largest measured size (honeycomb Heisenberg-Kitaev, 23 sites, 64 frequencies)
        dict(name="xyz-flow-honeycomb", kind="flow", core="XYZ", lattice="honeycomb", range=8, model="honeycomb-kitaev",
             nw=64, fmin=0.005, fmax=50.0, cmax=50.0, cmin=0.01, cstep=0.75),
        # the scripted TRI run (all three off-diagonal exchange types)
        dict(name="tri-core-honeycomb", kind="core", core="TRI", lattice="honeycomb", range=3,
             model="honeycomb-kitaev-gamma"),
        # the TRI core at its largest measured size (kagome with Dzyaloshinskii-Moriya exchange, 48 frequencies)
        dict(name="tri-flow-kagome", kind="flow", core="TRI", lattice="kagome", range=5, model="kagome-DM", nw=48,
             fmin=0.005, fmax=50.0, cmax=50.0, cmin=0.01, cstep=0.7),
        # the served J2/J1 sweep: eight flows of ranges 3 to 6, admitted together
        dict(name="su2-sweep-cubic", kind="sweep", flows=8, maxrange=6, nws="24 32 48", cmax=100.0, cmin=0.05,
             cstep=0.85),
    ]


def draw(rng):
    """One more case: kinds as often as a user meets them, sizes over the ranges
    of the listed cases (logarithmic in the number of frequencies)."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    su2_lattices = [("square", 3, 7, "square-heisenberg"), ("triangular", 2, 6, "triangular-heisenberg"),
                    ("honeycomb", 3, 8, "honeycomb-heisenberg"), ("kagome", 3, 6, "kagome-heisenberg"),
                    ("cubic", 3, 7, "cubic-j1j2heisenberg")]
    kind = rng.choice(["step", "step", "step", "su2", "su2", "mixed", "xyz", "tri", "sweep"])
    if kind == "sweep":
        return dict(kind="sweep", flows=rng.randint(3, 8), maxrange=rng.randint(4, 6),
                    nws="%d %d" % (log_int(12, 24), log_int(24, 48)), cmax=100.0, cmin=0.05,
                    cstep=round(rng.uniform(0.80, 0.86), 3))
    if kind == "step":
        lat, lo, hi, model = rng.choice(su2_lattices)
        return dict(kind="step", lattice=lat, range=rng.randint(lo, hi), model=model, nw=log_int(8, 64), fmin=0.002,
                    fmax=100.0, cutoff=round(math.exp(rng.uniform(math.log(0.01), math.log(80.0))), 4))
    if kind in ("su2", "mixed"):
        lat, lo, hi, model = rng.choice(su2_lattices)
        c = dict(kind="flow", core="SU2", lattice=lat, range=rng.randint(lo, hi), model=model, nw=log_int(10, 48),
                 fmin=0.002, fmax=100.0, cmax=100.0, cmin=0.5, cstep=round(rng.uniform(0.75, 0.9), 3))
        if kind == "mixed":
            c.update(cmin=3.0, mixed=True)
        else:
            c.update(queued=rng.random() < 0.5)
        return c
    if kind == "xyz":
        return dict(kind="flow", core="XYZ", lattice="honeycomb", range=rng.randint(3, 8), model="honeycomb-kitaev",
                    nw=log_int(8, 48), fmin=0.005, fmax=50.0, cmax=50.0, cmin=0.2,
                    cstep=round(rng.uniform(0.7, 0.85), 3))
    lat, hi, model = rng.choice([("kagome", 5, "kagome-DM"), ("honeycomb", 7, "honeycomb-kitaev")])
    return dict(kind="flow", core="TRI", lattice=lat, range=rng.randint(2, hi), model=model, nw=log_int(8, 36),
                fmin=0.005, fmax=50.0, cmax=50.0, cmin=0.2, cstep=round(rng.uniform(0.7, 0.85), 3))


# ---------------------------------------------------------------------------
# problems
# ---------------------------------------------------------------------------
def _couplings(model, seed):
    base = MODELS[model]
    if seed is None:
        return base
    rng = random.Random(seed)
    return {k: v * (1.0 + SPREAD * rng.uniform(-1.0, 1.0)) for k, v in base.items()}


@functools.lru_cache(maxsize=64)
def _lattice(name, extent, model, resources):
    """The lattice and its symmetry tables; they depend on which couplings a
    model has, not on their values, so a sweep of couplings builds them once."""
    return new_lattice_model(LatticeUnitCell.from_resources(name, resources), _model(model, MODELS[model], resources),
                             extent)


def _model(name, couplings, resources):
    return SpinModelUnitCell.from_resources(name, {k: repr(v) for k, v in couplings.items()}, resources)


def _problem_of(core, mesh, cutoffs, lattice, extent, model, couplings, resources=None):
    lat = _lattice(lattice, extent, model, resources)
    bonds = model_couplings(lat.sites[:lat.size], _model(model, couplings, resources))
    build = {"SU2": su2_problem_from_lattice, "XYZ": xyz_problem_from_lattice, "TRI": tri_problem_from_lattice}[core]
    return build(mesh, cutoffs, dataclasses.replace(lat, couplings=bonds), {})


def _problem(case, seed):
    if case["kind"] == "core":
        mesh = np.array(MANUAL_MESH, dtype=np.float32)
        cutoffs = exponential_cutoffs(np.float32(10.0), np.float32(0.3), np.float32(0.9))
        resources = GOLDEN_RESOURCES
    else:
        mesh = exponential_mesh(np.float32(case["fmin"]), np.float32(case["fmax"]), case["nw"])
        cutoffs = np.array([case["cutoff"]], dtype=np.float32) if case["kind"] == "step" else exponential_cutoffs(
            np.float32(case["cmax"]), np.float32(case["cmin"]), np.float32(case["cstep"]))
        resources = None
    return _problem_of(case.get("core", "SU2"), mesh, cutoffs, case["lattice"], case["range"], case["model"],
                       _couplings(case["model"], seed), resources)


def _sweep_requests(case, seed):
    """The sweep's flows: lattice ranges and frequency counts in turn (the same
    for every seed), J2 drawn from the seed."""
    nws = [int(v) for v in case["nws"].split()]
    cutoffs = exponential_cutoffs(np.float32(case["cmax"]), np.float32(case["cmin"]), np.float32(case["cstep"]))
    rng = random.Random(seed)
    out = []
    for i in range(case["flows"]):
        extent, nw, j2 = 3 + i % (case["maxrange"] - 2), nws[i % len(nws)], rng.uniform(0.0, 0.5)
        prob = _problem_of("SU2", exponential_mesh(np.float32(0.002), np.float32(100.0), nw), cutoffs, "cubic", extent,
                           "cubic-j1j2heisenberg", {"j1": 1.0, "j2": j2})
        out.append(FlowRequest(i, prob, 0.0, {"j2": j2, "range": extent, "nw": nw}))
    return out


def _step_state(prob, seed, device="cuda"):
    """Sigma and the interleaved {spin, density} vertex on the device, of the
    size and shape a flow reaches below its first cutoffs: a self-energy that
    grows and saturates, the couplings enhanced at small transfer frequencies,
    a density channel that is odd under the exchange of its outer frequencies,
    and the unsmooth part that renormalisation leaves on both."""
    g = torch.Generator(device=device).manual_seed(int(seed))
    nw, L = prob.nw, prob.L

    def noise(*shape):
        return torch.rand(shape, generator=g, device=device, dtype=torch.float64) * 2.0 - 1.0

    m = torch.from_numpy(prob.mesh.astype(np.float64)).to(device)
    v2 = 0.3 * m / (0.5 + m) * (1.0 + 0.02 * noise(nw))
    su = torch.tril_indices(nw, nw, device=device)
    s, u = m[su[0]][:, None], m[su[1]][:, None]
    t = m[None, :]
    decay = 1.0 / (1.0 + t) + 0.2 / (1.0 + (s - u).abs())
    j = torch.from_numpy(prob.coupling_zz_f64).to(device)
    tail = torch.exp(-0.3 * torch.arange(L, device=device, dtype=torch.float64))
    v4 = torch.empty((su.shape[1], nw, L, 2), device=device, dtype=torch.float64)
    v4[..., 0] = (j + 0.2 * tail) * decay[..., None] * (1.0 + 0.05 * noise(su.shape[1], nw, L))
    v4[..., 1] = 0.1 * tail * ((s - u) / (s + u) * torch.ones_like(t))[..., None] + 0.01 * noise(su.shape[1], nw, L)
    return v2, v4


# ---------------------------------------------------------------------------
# the timed passes
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        prob = _problem(case, seed)
        lib = load_library()
        lib.sp_compute_step_noalloc.argtypes = [ctypes.POINTER(SpSu2Problem), ctypes.c_double] + \
            [ctypes.c_void_p] * 5 + [ctypes.POINTER(ctypes.c_int)]
        v2, v4 = _step_state(prob, seed)
        return dict(kind=kind, lib=lib, prob=prob, buffers=ProblemBuffers(prob), cutoff=float(case["cutoff"]), v2=v2,
                    v4=v4, dv2=torch.zeros_like(v2), dv4=torch.zeros_like(v4))
    if kind == "core":
        core = FrgCoreFactory.newFrgCore(case["core"], _problem(case, seed), [MeasurementSpec("correlation")],
                                         backend="hip")
        return dict(kind=kind, core=core, init=core.problem.initial_state(np.float64),
                    cutoffs=[float(c) for c in core.problem.cutoffs])
    if kind == "sweep":
        return dict(kind=kind, requests=_sweep_requests(case, seed))
    prob = _problem(case, seed)
    if case["core"] == "SU2":
        ctx = FlowContext(prob, SP_PRECISION_MIXED if case.get("mixed") else SP_PRECISION_FP64)
    else:
        ctx = (XyzFlowContext if case["core"] == "XYZ" else TriFlowContext)(prob)
    return dict(kind=kind, ctx=ctx, prob=prob, init=prob.initial_state(np.float64), queued=bool(case.get("queued")))


def _run_step(s):
    p = torch.Tensor.data_ptr
    rc = s["lib"].sp_compute_step_noalloc(ctypes.byref(s["buffers"].struct), s["cutoff"], p(s["v2"]), p(s["v4"]),
                                          p(s["dv2"]), p(s["dv4"]), torch.cuda.current_stream().cuda_stream, None)
    if rc != 0:
        raise RuntimeError("sp_compute_step_noalloc returned %d" % rc)
    return {"dsigma": s["dv2"], "dgamma": s["dv4"]}


def _run_flow(s):
    ctx, cut = s["ctx"], s["prob"].cutoffs
    ctx.set_state(float(cut[0]), *s["init"])
    diverged = False
    if s["queued"]:
        records, diverged = ctx.run_flow(cut)
        records = [np.stack(r) for r in records]
    else:
        records = []
        for k in range(len(cut) - 1):
            ctx.compute_step()
            records.append(np.stack(ctx.measure_correlation()))
            if ctx.is_diverged():
                diverged = True
                break
            ctx.finalize_step(float(cut[k + 1]))
    if not diverged:
        records.append(np.stack(ctx.measure_correlation()))
    return {"records": np.stack(records), "state": ctx.get_state()}


def _run_core(s):
    core = s["core"]
    core.setState(s["cutoffs"][0], *s["init"])
    records = []
    for k in range(len(s["cutoffs"]) - 1):
        core.computeStep()
        records.append(np.stack(core.context.measure_correlation()))
        if core.flow().isDiverged():
            break
        core.finalizeStep(s["cutoffs"][k + 1])
    records.append(np.stack(core.context.measure_correlation()))
    return {"records": np.stack(records), "state": core.flowingFunctional().arrays()}


def _run_sweep(s):
    server = SweepServer(budget_bytes=64 << 30, max_flows=32, precision=SP_PRECISION_MIXED,
                         schedule=PrecisionSchedule())
    try:
        results = server.run(s["requests"])
    finally:
        server.close()
    return {"flow%d" % r.ident: {"zz": np.stack(r.zz), "dd": np.stack(r.dd), "diverged": r.diverged} for r in results}


def run(state):
    return {"step": _run_step, "flow": _run_flow, "core": _run_core, "sweep": _run_sweep}[state["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _evaluation_flops(mesh, L, cut, components, overlap):
    """Operations of one derivative evaluation.  An integration point costs the
    bilinear interpolation of the vertices it multiplies and their products.
    The S and U channels are images of each other under the exchange of s and
    u, so one evaluation of the pair is counted; the two buffers of a T-channel
    pair are images as well.  The lattice bubble is linear in the products of
    site pairs, so it is counted once per point as those products and once per
    frequency triple as the sum over overlap entries."""
    nw = len(mesh)
    calls = float(channel_calls(mesh, float(cut)).sum())
    triples = nw * nw * (nw + 1) / 2.0
    per_su = {2: 64.0 + 28.0, 4: 128.0 + 64.0, 16: 512.0 + 1024.0}[components] * L
    per_t = {2: 32.0 + 16.0, 4: 64.0 + 64.0, 16: 256.0 + 1024.0}[components] * L
    bubble = {2: 4.0 * L * L, 4: 20.0 * L * L, 16: min(128.0 * overlap, 512.0 * L * L)}[components]
    t_points = calls * nw * (nw + 1) / 2.0
    su_points = calls * nw * (nw + 1)
    return su_points * per_su + t_points * (per_t + bubble) + triples * 2.0 * components * overlap


def _work(prob, cutoffs, components):
    n = len(cutoffs)
    vertex = 8.0 * prob.n_freq * prob.L * components
    flops = sum(_evaluation_flops(prob.mesh, prob.L, c, components, prob.overlap_total) for c in cutoffs)
    return 2.0 * vertex * n, flops + 2.0 * prob.n_freq * prob.L * components * n


def work(case):
    if case["kind"] == "sweep":
        b = f = 0.0
        for r in _sweep_requests(case, 1):
            x, y = _work(r.problem, r.problem.cutoffs[:-1], 2)
            b, f = b + x, f + y
        return {"bytes": b, "flops": f}
    prob = _problem(case, None)
    components = {"SU2": 2, "XYZ": 4, "TRI": 16}[case.get("core", "SU2")]
    cutoffs = [case["cutoff"]] if case["kind"] == "step" else prob.cutoffs[:-1]
    b, f = _work(prob, cutoffs, components)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the derivative in plain 64-bit arithmetic
# ---------------------------------------------------------------------------
def exact(case, seed):
    """dSigma and dGamma of a "step" case written out term by term: every
    channel of every frequency triple, the lattice bubble per point.  The runs
    of many evaluations, and the evaluations with many points, would take
    minutes this way (None)."""
    if case["kind"] != "step":
        return None
    prob = _problem(case, seed)
    points = float(channel_calls(prob.mesh, case["cutoff"]).sum())
    if points * prob.nw * (prob.nw + 1) * prob.L * (60.0 + 4.0 * prob.L) > 8e10 or points > 700:
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    v2, v4 = _step_state(prob, seed, device)
    return _Su2Step(prob, float(case["cutoff"]), v2, v4).evaluate()


class _Su2Step:
    def __init__(self, prob, cut, v2, v4):
        self.p, self.cut, self.v2, self.dev = prob, cut, v2, v4.device
        self.nw, self.L = prob.nw, prob.L
        self.m = torch.from_numpy(prob.mesh.astype(np.float64)).to(self.dev)
        self.rows = v4.reshape(-1, prob.L, 2)
        self.site = torch.from_numpy(prob.site_rid.astype(np.int64)).to(self.dev)
        self.inv = torch.from_numpy(prob.inv_rid.astype(np.int64)).to(self.dev)

    # interpolation on the positive mesh, clamped at both ends
    def bracket(self, w):
        w = w.contiguous()
        c = torch.searchsorted(self.m, w, right=True)
        lo = (c - 1).clamp(0, self.nw - 1)
        hi = torch.where(w > self.m[0], c, torch.zeros_like(c)).clamp(0, self.nw - 1)
        lo = torch.where(w > self.m[0], lo, torch.zeros_like(lo))
        width = torch.where(hi > lo, self.m[hi] - self.m[lo], torch.ones_like(w))
        return lo, hi, torch.where(hi > lo, (w - self.m[lo]) / width, torch.zeros_like(w))

    def sigma(self, data, w):
        lo, hi, b = self.bracket(w.abs())
        return torch.where(w < 0, -1.0, 1.0) * ((1 - b) * data[lo] + b * data[hi])

    def stored(self, s, t, u, site):
        """Vertex values at mesh indices for the sites of `site` (.., L): the
        stored half is s >= u, the density channel odd under the exchange."""
        swap = s < u
        big, small = torch.where(swap, u, s), torch.where(swap, s, u)
        v = self.rows[(big * (big + 1) // 2 + small) * self.nw + t]
        v = torch.gather(v, -2, site[..., None].expand(*site.shape, 2))
        sign = torch.stack([torch.ones_like(swap, dtype=v.dtype), torch.where(swap, -1.0, 1.0).to(v.dtype)], -1)
        return v * sign[..., None, :]

    def vertex(self, s, t, u, exact_arg, index, local=False):
        """Both channels at signed frequencies; argument `exact_arg` (0 s, 1 t,
        2 u) sits on mesh index `index`.  Exactly one negative outer frequency
        exchanges the sites."""
        if local:
            site = torch.zeros(s.shape + (1,), dtype=torch.int64, device=self.dev)
        else:
            swap = ((s < 0) != (u < 0))[..., None]
            site = torch.where(swap, self.inv.expand(*s.shape, self.L), self.site.expand(*s.shape, self.L))
        pts = []
        for k, w in enumerate((s, t, u)):
            if k == exact_arg:
                i = torch.full(s.shape, index, dtype=torch.int64, device=self.dev)
                pts.append([(i, 1.0)])
            else:
                lo, hi, b = self.bracket(w.abs())
                pts.append([(lo, (1 - b)[..., None, None]), (hi, b[..., None, None])])
        return sum((ws * wt * wu) * self.stored(i, j, k, site)
                   for k, wu in pts[2] for j, wt in pts[1] for i, ws in pts[0])

    # the list of integration points and weights of one transfer frequency
    def points(self, x, dv2):
        m, n, cut = self.p.mesh.astype(np.float64), self.nw, self.cut
        X = float(m[x])
        at = lambda i: m[i] if i >= 0 else -m[-i - 1]  # noqa: E731
        gpos = lambda w: 0 if w <= m[0] else next((i for i in range(1, n) if m[i] > w), n - 1)  # noqa: E731
        lpos = lambda w: 0 if w <= m[0] else next((i - 1 for i in range(1, n) if m[i] > w), n - 1)  # noqa: E731
        lesser = lambda w: -(gpos(-w) + 1) if w < 0 else lpos(w)  # noqa: E731
        greater = lambda w: -(lpos(-w) + 1) if w < 0 else gpos(w)  # noqa: E731

        def trapezoid(nodes):
            w = [0.0] * len(nodes)
            for i in range(len(nodes) - 1):
                h = 0.5 * (nodes[i + 1] - nodes[i])
                w[i] += h
                w[i + 1] += h
            return list(zip(nodes, w))

        pts = []
        if -(X + cut) > at(-n):
            top = lesser(-(X + cut))
            pts += trapezoid([at(i) for i in range(-n, top + 1)] + [-(X + cut)])
        if X - cut > cut:
            a, b = greater(cut - X), lesser(-cut)
            pts += trapezoid([cut - X] + [at(i) for i in range(a, b + 1)] + [-cut])
        if cut < at(n - 1):
            pts += trapezoid([cut] + [at(i) for i in range(greater(cut), n)])
        w = torch.tensor([q[0] for q in pts], dtype=torch.float64, device=self.dev)
        h = torch.tensor([q[1] for q in pts], dtype=torch.float64, device=self.dev)
        d = w + self.sigma(self.v2, w)
        c = h * self.sigma(dv2, w) / (d * d * (X + w + self.sigma(self.v2, X + w)))
        one = torch.tensor([cut], dtype=torch.float64, device=self.dev)
        prop = lambda a, b: 1.0 / ((a + self.sigma(self.v2, a)) * (b + self.sigma(self.v2, b)))  # noqa: E731
        wl, cl = [one], [prop(one, one + X)]
        if X > 2.0 * cut:
            wl.append(-one)
            cl.append(prop(one, one - X))
        return torch.cat(wl + [w]), torch.cat(cl + [c])

    def dsigma(self):
        p, cut, w = self.p, self.cut, self.m
        R = len(p.range_fwd)
        fwd = torch.from_numpy(p.range_fwd.astype(np.int64)).to(self.dev)
        inv = torch.from_numpy(p.range_inv.astype(np.int64)).to(self.dev)

        def full(s, t, u, f, i):  # all three arguments off the mesh, sites f (or i when exchanged)
            swap = ((s < 0) != (u < 0))[..., None]
            site = torch.where(swap, i.expand(*s.shape, len(i)), f.expand(*s.shape, len(f)))
            br = [self.bracket(x.abs()) for x in (s, t, u)]
            out = 0.0
            for k in range(8):
                idx = [br[a][(k >> a) & 1] for a in range(3)]
                wt = 1.0
                for a in range(3):
                    wt = wt * (br[a][2] if (k >> a) & 1 else 1 - br[a][2])
                out = out + wt[..., None, None] * self.stored(idx[0], idx[1], idx[2], site)
            return out

        zero = torch.zeros_like(w)
        origin = torch.zeros(1, dtype=torch.int64, device=self.dev)
        a = full(w + cut, zero, w - cut, fwd, inv)[..., 1] - full(w - cut, zero, w + cut, fwd, inv)[..., 1]
        b = (full(w + cut, w - cut, zero, origin, origin) - full(w - cut, w + cut, zero, origin, origin))[:, 0]
        v = -4.0 * float(p.spin) * a.sum(-1) + 0.75 * b[:, 0] + b[:, 1]
        one = torch.tensor([cut], dtype=torch.float64, device=self.dev)
        return v / (2.0 * math.pi * (cut + self.sigma(self.v2, one)))

    def evaluate(self):
        p, m, nw, L = self.p, self.m, self.nw, self.L
        S = float(p.spin)
        dv2 = self.dsigma()
        tri = torch.tril_indices(nw, nw, device=self.dev)
        out = torch.zeros((tri.shape[1], nw, L, 2), dtype=torch.float64, device=self.dev)
        entry = torch.from_numpy((p.ovl_rid1.astype(np.int64) * L + p.ovl_rid2)).to(self.dev)
        owner = torch.from_numpy(np.repeat(np.arange(L), np.diff(p.ovl_off)).astype(np.int64)).to(self.dev)
        for x in range(nw):
            wps, cs = self.points(x, dv2)
            X = m[x]
            # s channel: all u <= s = x, every t
            u, t = m[: x + 1][:, None].expand(x + 1, nw), m[None, :].expand(x + 1, nw)
            acc = 0.0
            for wp, c in zip(wps, cs):
                w1p, w1, w2p, w2 = 0.5 * (X + t + u), 0.5 * (X - t + u), 0.5 * (X - t - u), 0.5 * (X + t - u)
                s = X.expand_as(t)
                A = [self.vertex(s, w1 + wp, -w2 - wp, 0, x), self.vertex(s, w1p + wp, -w2p - wp, 0, x),
                     self.vertex(s, w2 + wp, w1 + wp, 0, x), self.vertex(s, w2p + wp, w1p + wp, 0, x)]
                acc = acc + c * self.ladder(A, -0.5)
            out[x * (x + 1) // 2: x * (x + 1) // 2 + x + 1] += acc
            # u channel: all s >= u = x, every t
            s, t = m[x:][:, None].expand(nw - x, nw), m[None, :].expand(nw - x, nw)
            acc = 0.0
            for wp, c in zip(wps, cs):
                w1p, w1, w2p, w2 = 0.5 * (s + t + X), 0.5 * (s - t + X), 0.5 * (s - t - X), 0.5 * (s + t - X)
                u = X.expand_as(t)
                A = [self.vertex(w1 + wp, w2p - wp, u, 2, x), self.vertex(w1p + wp, w2 - wp, u, 2, x),
                     self.vertex(w2p - wp, w1 + wp, u, 2, x), self.vertex(w2 - wp, w1p + wp, u, 2, x)]
                acc = acc - c * self.ladder(A, 0.5)
            i = torch.arange(x, nw, device=self.dev)
            out[i * (i + 1) // 2 + x] += acc
            # t channel: all s >= u at t = x
            s, u = m[tri[0]], m[tri[1]]
            t = X.expand_as(s)
            acc = 0.0
            pairs = torch.zeros((tri.shape[1], L, L, 2), dtype=torch.float64, device=self.dev)
            for wp, c in zip(wps, cs):
                w1p, w1, w2p, w2 = 0.5 * (s + t + u), 0.5 * (s - t + u), 0.5 * (s - t - u), 0.5 * (s + t - u)
                A = [self.vertex(w1 - wp, t, w1p + wp, 1, x), self.vertex(w2p - wp, t, -w2 - wp, 1, x),
                     self.vertex(w1p + wp, t, w1 - wp, 1, x), self.vertex(w2 + wp, t, wp - w2p, 1, x)]
                B = [self.vertex(w2p - wp, w2 + wp, t, 2, x, True), self.vertex(w1 - wp, w1p + wp, t, 2, x, True),
                     self.vertex(w2 + wp, w2p - wp, t, 2, x, True), self.vertex(w1p + wp, w1 - wp, t, 2, x, True)]
                for a, b in zip(A, B):
                    bs, bd = b[..., 0], b[..., 1]
                    acc = acc + c * torch.stack([(0.25 * bs - bd) * a[..., 0], -(0.75 * bs + bd) * a[..., 1]], -1)
                pairs += c * A[2][:, :, None] * A[3][:, None, :]
            flat = pairs.reshape(tri.shape[1], L * L, 2)
            rpa = torch.zeros((tri.shape[1], L, 2), dtype=torch.float64, device=self.dev)
            for i0 in range(0, len(entry), 1024):
                rpa.index_add_(1, owner[i0:i0 + 1024], flat[:, entry[i0:i0 + 1024]])
            rpa = rpa * torch.tensor([2.0 * S, 8.0 * S], dtype=torch.float64, device=self.dev)
            out[:, x] += acc + rpa
        return {"dsigma": dv2, "dgamma": out / (2.0 * math.pi)}

    @staticmethod
    def ladder(A, sign):
        (s0, d0), (s1, d1), (s2, d2), (s3, d3) = [(a[..., 0], a[..., 1]) for a in A]
        h = s0 * s1 + s2 * s3
        return torch.stack([sign * h + d0 * s1 + d2 * s3 + s0 * d1 + s2 * d3, 0.1875 * h + d0 * d1 + d2 * d3], -1)
