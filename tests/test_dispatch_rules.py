"""Which kernels a call gets, where the choice is made from sizes alone: asked of the library on the CPU
(which then counts 256 compute units)."""
import pytest

from bladedisc_amd import _lib


@pytest.mark.parametrize("channels,inner,folds", [
    # a tensor: up to 4096 pairs of 4096 elements
    (1, 4, True), (1, 3, False), (1, 3072 * 768, True), (1, 1 << 24, True), (1, (1 << 24) + 4, False),
    # rows: up to six pairs each, below 1024 rows and 8 M elements
    (2, 6 * 4096, True), (2, 6 * 4096 + 4, False), (2, 1 << 20, False), (16, 131072, False), (64, 40960, False),
    (740, 240, True), (1023, 4, True), (1024, 4, False), (2048, 1024, False), (341, 24576, True),
    (342, 24576, False), (5, 30, False)])
def test_the_observed_range_is_folded_with_the_fake_quantization_where_that_is_short(channels, inner, folds):
    """One workgroup folds every row's pairs on a thread a row ahead of the answer that the host waits for:
    2 rows of 2^20 elements, 256 pairs each, took 39 us a step in that form and 18 with a kernel that
    folds once."""
    L = _lib.hooks()
    assert bool(L.dq8_observe_folds_range(1, channels, inner)) == folds
    assert not L.dq8_observe_folds_range(2, channels, inner)
