"""Registers of the mixed SU(2) wave kernels, as the compiler reports them.

Every instantiation runs whole flows, those for lattices whose bonds differ from
their reverse (honeycomb, kagome) as well.  With two gathers of a tile held at
once those spilled 82 and 157 registers and took up to twice the time of the
kernel they had replaced; a few spilled outside the loop over the points cost
nothing.
"""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAX_SPILLS = 16


def _resources(source):
    from spinparser_amd.build import hipcc
    out = subprocess.run([hipcc(), "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
                          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-fconstexpr-steps=33554432",
                          "-I", os.path.join(ROOT, "include"), "-c", os.path.join(ROOT, "spinparser_amd", "csrc", source),
                          "-o", os.devnull, "--offload-device-only", "-Rpass-analysis=kernel-resource-usage"],
                         capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stderr[-2000:]
    kernels = {}
    for block in out.stderr.split("Function Name: ")[1:]:
        kernels[block.split()[0]] = int(re.search(r"VGPRs Spill: (\d+)", block).group(1))
    return kernels


def test_mixed_wave_kernels_do_not_spill():
    kernels = {k: n for k, n in _resources("su2_flow.hip").items() if "k_t32" in k or "k_su32" in k}
    assert len(kernels) == 8 + 6  # tile shapes x exchange, sites per lane x exchange
    worst = max(kernels, key=kernels.get)
    assert kernels[worst] <= MAX_SPILLS, (worst, kernels[worst])
