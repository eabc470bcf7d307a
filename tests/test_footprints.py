"""Device footprints of the contexts, computed on the host."""
import dataclasses

import numpy as np
import pytest

from helpers import cfg1_problem, tri_problem_of


def _xyz_problem(r=4):
    from spinparser_amd.problem import xyz_problem
    from spinparser_amd.task import make_task_xml, parse_task
    return xyz_problem(parse_task(make_task_xml(
        lattice="honeycomb", lattice_range=r, model="honeycomb-kitaev", symmetry="XYZ",
        couplings={"j": 0.1, "k": -1.0}, freq_min=0.01, freq_max=20.0, freq_count=6, cutoff_max=20.0, cutoff_min=0.05,
        cutoff_step=0.9), True))


def _tri_problem():
    return tri_problem_of("kagome", 3, "kagome-DM", {"j": 1.0, "d": 0.2}, 6, 0.01, 20.0, 20.0, 0.05, 0.9)


def _longer_records(prob):
    """The same problem with twice the sites per record."""
    more = {"Rb": 2 * prob.Rb, "corr_rid": np.concatenate([prob.corr_rid] * 2)}
    if hasattr(prob, "corr_perm"):
        more["corr_perm"] = np.concatenate([prob.corr_perm] * 2)
    return dataclasses.replace(prob, **more)


@pytest.mark.parametrize("core", ["SU2", "XYZ", "TRI"])
def test_records_take_no_device_memory(core):
    """Records go to pinned host memory: a longer one costs its tables alone (site,
    and for XYZ and TRI three spin components per entry)."""
    from spinparser_amd.capi import footprint_bytes, tri_footprint_bytes, xyz_footprint_bytes
    prob, size, ints = {"SU2": (cfg1_problem(nw=8), footprint_bytes, 1), "XYZ": (_xyz_problem(), xyz_footprint_bytes, 4),
                        "TRI": (_tri_problem(), tri_footprint_bytes, 4)}[core]
    assert size(_longer_records(prob)) - size(prob) == 4 * ints * prob.B * prob.Rb


@pytest.mark.parametrize("core", ["XYZ", "TRI"])
def test_tables_of_the_wave_kernels_are_counted(core):
    """A lattice that runs the wave kernels holds their tables besides those of the
    general kernels, which a lattice with other site tables runs: per output a
    lane or more and per lane a count, and at least one entry of four bytes for
    every overlap entry whose products differ."""
    from spinparser_amd.capi import tri_footprint_bytes, xyz_footprint_bytes
    prob, size = {"XYZ": (_xyz_problem(), xyz_footprint_bytes), "TRI": (_tri_problem(), tri_footprint_bytes)}[core]
    components = 4 if core == "XYZ" else 16
    other = dataclasses.replace(prob, site_rid=np.roll(prob.site_rid, 1))
    assert size(prob) - size(other) >= 4 * (components * prob.L + 64 + len(prob.ovl_rid1) // 4)
