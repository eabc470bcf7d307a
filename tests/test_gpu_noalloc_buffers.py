"""sp_compute_step_noalloc with dGamma in memory that the wave kernels' atomics
need not reach: pinned host memory and fine-grained device memory.  Those calls
run the general dGamma kernel, also on lattices that otherwise run the wave
kernels.

Tolerance: as for the wave kernels (fewer than 1e5 terms with an error of 1.1e-16
of their size each, exceeding the largest entry by less than 10): 1e-10 of the
largest entry bounds the difference of two summation orders.
"""
import ctypes

import numpy as np
import pytest

from helpers import exp_problem, max_rel
from test_zz_no_alloc import D2H, H2D, _declare, _hip_runtime

pytestmark = pytest.mark.gpu

TOL = 1e-10
J, J12 = {"j": 1.0}, {"j1": 1.0, "j2": 0.3}
FINE_GRAINED = 1  # hipDeviceMallocFinegrained


@pytest.mark.parametrize("memory", ["pinned", "fine-grained"])
@pytest.mark.parametrize("lattice,r,model,couplings,nw", [
    ("square", 4, "square-heisenberg", J, 9),          # 9 sites
    ("cubic", 5, "cubic-j1j2heisenberg", J12, 6),      # 16 sites
    ("kagome", 5, "kagome-heisenberg", J, 6),          # 19 sites
    ("cubic", 7, "cubic-j1j2heisenberg", J12, 4),      # 31 sites
])
def test_general_kernel_into_other_memory(lattice, r, model, couplings, nw, memory):
    from oracle import Oracle
    from spinparser_amd.capi import ProblemBuffers, load_library
    lib = load_library()
    _declare(lib)
    hip = _hip_runtime()
    prob = exp_problem(lattice, r, model, couplings, nw, 0.01, 20.0, 20.0, 0.05, 0.9)
    rng = np.random.default_rng(5)
    v2 = rng.uniform(0.05, 0.3, prob.nw)
    ss, dd = rng.uniform(-1.0, 1.0, prob.vertex_size), rng.uniform(-1.0, 1.0, prob.vertex_size)
    cut = 0.3
    ref = Oracle(prob).compute_step(cut, v2, ss, dd)
    v4 = np.ascontiguousarray(np.stack([ss, dd], axis=-1))
    out = np.zeros_like(v4)
    dv2 = np.zeros(prob.nw)
    dev = {}
    for name, a in (("v2", v2), ("v4", v4), ("dv2", dv2)):
        dev[name] = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(dev[name]), a.nbytes) == 0
        assert hip.hipMemcpy(dev[name], a.ctypes.data, a.nbytes, H2D) == 0
    buf = ctypes.c_void_p()
    if memory == "pinned":
        assert hip.hipHostMalloc(ctypes.byref(buf), ctypes.c_size_t(out.nbytes), ctypes.c_uint(0)) == 0
    else:
        assert hip.hipExtMallocWithFlags(ctypes.byref(buf), ctypes.c_size_t(out.nbytes),
                                         ctypes.c_uint(FINE_GRAINED)) == 0
    div = ctypes.c_int(-1)
    pb = ProblemBuffers(prob)
    rc = lib.sp_compute_step_noalloc(ctypes.byref(pb.struct), cut, dev["v2"], dev["v4"], dev["dv2"], buf, None,
                                     ctypes.byref(div))
    assert rc == 0 and div.value == 0
    if memory == "pinned":
        ctypes.memmove(out.ctypes.data, buf, out.nbytes)
        assert hip.hipHostFree(buf) == 0
    else:
        assert hip.hipMemcpy(out.ctypes.data, buf, out.nbytes, D2H) == 0
        assert hip.hipFree(buf) == 0
    assert hip.hipMemcpy(dv2.ctypes.data, dev["dv2"], dv2.nbytes, D2H) == 0
    for p in dev.values():
        assert hip.hipFree(p) == 0
    errors = [max_rel(dv2, ref[0]), max_rel(out[:, 0], ref[1]), max_rel(out[:, 1], ref[2])]
    print("%s L=%d: %s" % (memory, prob.L, errors), flush=True)
    assert max(errors) < TOL
