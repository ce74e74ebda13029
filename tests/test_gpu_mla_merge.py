"""GPU parity of MLA decode over the number of partitions a sequence merges: one (finished by the
attention kernel), the merge's batches of eight partial loads and 64 partitions' (max, sum) per
lane at their edges, and few heads through the four copy waves with contexts of one to four
pipeline steps. Tolerances as for the other MLA tests; sequences of other counts stand beside."""

import pytest

from test_gpu_decode import _mla_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [16, 32, 64, 128])
def test_mla_merge_partition_counts(cuda, heads):
    """32-token partitions: 1, 2, 7, 8, 9, 16, 63, 64, 65 and 130 of them, exact and one token over."""
    counts = (1, 2, 7, 8, 9, 16, 63, 64, 65, 130)
    lens = [32 * n - 31 for n in counts] + [32 * n for n in counts[:6]] + [0]
    _mla_case(cuda, lens, heads=heads, bs=16, partition_size=32, tag=f"merge{heads}")


@pytest.mark.parametrize("heads", [16, 32])
def test_mla_copy_waves_short_contexts(cuda, heads):
    """One to five pipeline steps in one partition, blocks of 16 to 256."""
    for bs in (16, 64, 256):
        _mla_case(cuda, [1, 31, 32, 33, 64, 65, 96, 97, 128, 160], heads=heads, bs=bs, partition_size=160,
                  tag=f"copyw{heads}{bs}")
