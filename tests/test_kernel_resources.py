"""Host-only checks of the built kernels' registers, from the compiler's remarks
(``build/resource-usage.txt``).

The split-KV merge is bound by memory latency, so its speed follows the waves
that fit a SIMD: 8 waves and 64 VGPRs, 5 and 96, 4 and 128, 2 and 256.
"""
import re

import pytest

from tests.conftest import load_package

# Least waves per SIMD of combine_kernel<lane groups per row, ...>.
MERGE_WAVES = {1: 5, 2: 5, 4: 5, 8: 2}


@pytest.fixture(scope="module")
def resources():
    pkg = load_package().fav4_bshd
    if not pkg.RESOURCE_LOG.exists():
        pkg.build_library()
    return pkg.parse_resource_usage(pkg.RESOURCE_LOG.read_text())


@pytest.mark.parametrize("per", MERGE_WAVES)
def test_merge_keeps_its_waves(resources, per):
    kernels = {n: r for n, r in resources.items() if re.search(rf"combine_kernelILi{per}E", n)}
    assert len(kernels) == 4                                    # BSHD and packed, decode and prefill
    for name, r in kernels.items():
        assert r["Occupancy [waves/SIMD]"] >= MERGE_WAVES[per], (name, r)
        assert r["ScratchSize [bytes/lane]"] == 0, name


def test_contiguous_prefill_chunks_have_one_shape(resources):
    """Split-KV plans of contiguous K/V have 256-row q tiles only: the 128-row
    chunk kernel is built for packed and paged K/V alone."""
    rows128 = [n for n in resources if re.search(r"fwd_kernel_chunkILb[01]ELb[01]ELi4E", n)]
    assert rows128 and not [n for n in rows128 if "Li4ELi0E" in n]
