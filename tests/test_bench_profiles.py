"""The profile tool's names of kernels: what bench.py's trace calls them, from what rocprofv3 does."""
import os
import re
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


@pytest.mark.parametrize("kernel,name", [
    # key type, threads, items, whether rectangles go along, bits of a digit
    ("void dsx::onesweep32_kernel<unsigned int, 1024, 4, true, 9>(dsx::Sort32)", "onesweep32_kernel<sort>"),
    ("void dsx::onesweep32_kernel<unsigned int, 1024, 4, true, 8>(dsx::Sort32)", "onesweep32_kernel<sort>"),
    ("void dsx::onesweep32_kernel<unsigned int, 1024, 12, false, 9>(dsx::Sort32)", "onesweep32_kernel<sort>"),
    ("void dsx::onesweep32_kernel<unsigned int, 1024, 12, false, 8>(dsx::Sort32)", "onesweep32_kernel<tile partition>"),
    ("void dsx::onesweep32_kernel<unsigned short, 1024, 8, false, 8>(dsx::Sort32)", "onesweep32_kernel<tile partition>"),
    ("void dsx::onesweep32_first_kernel<12, true>(dsx::Sort32)", "onesweep32_kernel<sort>"),
    ("void dsx::blend_fwd_tile_kernel<true>(int const*)", "blend_fwd_kernel"),
    ("dsx::blend_fwd_wide_kernel(int const*)", "blend_fwd_kernel"),
    ("void dsx::blend_bwd_kernel<false>(int const*)", "blend_bwd_kernel"),
    ("dsx::project_fwd_kernel(float)", "project_fwd_kernel"),
])
def test_trace_names(kernel, name):
    import bench_profiles
    assert bench_profiles.trace_name(bench_profiles.short_name(kernel)) == name


def test_the_sorts_template_is_what_the_names_assume():
    source = open(os.path.join(ROOT, "ds_splat_amd", "csrc", "tile_lists.hip")).read()
    head = re.search(r"template <([^>]*)>\s*__global__[^;{]*onesweep32_kernel\(", source)
    assert [p.split("=")[0].split()[-1] for p in head.group(1).split(",")] == ["KeyT", "kSort32Threads", "kSort32Items",
                                                                              "kCarry", "kBits"]


@pytest.mark.parametrize("emitting", [300000, 120000, 0])
def test_bytes_of_the_depth_sorts_passes(emitting):
    """The first pass and the later two have bytes of their own; the trace's name for all three has their average."""
    import bench
    work = [bench.algorithmic_work("onesweep32_kernel<sort%s>" % which, 300000, 0, 0, 0, 0, None, 0, emitting=emitting)[1]
            for which in (", first", ", later", "")]
    assert work[0] == 12 * 300000 + 4 * (300000 - emitting) + 12 * emitting and work[1] == 24 * emitting
    assert work[2] == pytest.approx((work[0] + 2 * work[1]) / 3)
