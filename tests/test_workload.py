"""Work models of the benchmark line."""
import re
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("core,lattice,r,model", [("SU2", "square", 4, "square-heisenberg"),
                                                  ("XYZ", "honeycomb", 3, "honeycomb-kitaev"),
                                                  ("TRI", "kagome", 2, "kagome-DM")])
def test_necessary_operations(core, lattice, r, model):
    """The rate of the roofline counts each symmetric image and each product of sites
    once: the count of the timed cases, and less than the reference's kernels do."""
    from perf import cases
    from spinparser_amd.workload import evaluation_flops, necessary_flops
    case = dict(kind="flow", core=core, lattice=lattice, range=r, model=model, nw=9, fmin=0.01, fmax=20.0, cmax=20.0,
                cmin=0.1, cstep=0.7)
    prob = cases._problem(case, None)
    cutoffs = prob.cutoffs[:-1]
    components = {"SU2": 2, "XYZ": 4, "TRI": 16}[core]
    euler = 2.0 * prob.n_freq * prob.L * components * len(cutoffs)
    total = sum(necessary_flops(prob, c) for c in cutoffs)
    assert abs(total + euler - cases.work(case)["flops"]) <= 1e-12 * total
    for c in cutoffs:
        assert necessary_flops(prob, c) < evaluation_flops(prob, c)


def test_benchmark_names_the_kernels_it_times():
    """The kernels named beside the dGamma times exist, and are those the sources
    launch for the workloads, not the general kernels."""
    import bench
    csrc = os.path.join(ROOT, "spinparser_amd", "csrc")
    text = "".join(open(os.path.join(csrc, f)).read() for f in sorted(os.listdir(csrc)))
    labels = [bench.DGAMMA_KERNELS] + [c["kernel"] for c in bench.CORES.values()]
    for name in [n for label in labels for n in label.split(" + ")]:
        assert re.search(r"__global__[^;{]*\b%s\(" % name, text), name
        assert "dgamma" not in name
