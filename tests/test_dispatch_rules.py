"""Which kernels a call gets, where the choice is made from sizes alone: asked of the library on the CPU
(which then counts 256 compute units)."""
import ctypes as C
import random

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


def _weight_only_plan(m, n, k, dtype, ragged=False):
    plan = (C.c_int * 4)()
    _lib.hooks().dq8_weight_only_plan(m, n, k, dtype, int(ragged), plan)
    return dict(form=plan[0], splits=plan[1], bm=plan[2], bn=plan[3])


@pytest.mark.parametrize("n,k,tiles", [
    (16, 2048, False), (4096, 256, False), (4096, 2048, False), (16, 2064, True), (4096, 2064, True),
    # 32 channels and more to a workgroup of the staged kernel
    (4097, 384, True), (4097, 400, False), (4097, 2048, False), (4097, 2064, True), (6143, 2064, True),
    (6144, 2816, False), (6144, 2832, True), (8192, 384, True), (8192, 1024, False), (8192, 2816, False),
    (8192, 2832, True), (8193, 400, True), (8193, 2048, True), (11008, 1024, True)])
def test_weight_only_f32_rows_run_on_tiles_where_they_are_faster_or_more_exact(n, k, tiles):
    """17 to 32 rows of f32: tiles on all weights wider than 4096 channels took 7.1 us in place of 6.1 at 24 x
    1024 -> 4104, 10.8 in place of 9.7 at 2304 -> 8192."""
    for m in (17, 24, 32):
        assert (_weight_only_plan(m, n, k, 0)["form"] >= 0) == tiles
    assert _weight_only_plan(16, n, k, 0)["form"] < 0 and _weight_only_plan(33, n, k, 0)["form"] >= 0
    assert _weight_only_plan(32, n, k, 1)["form"] < 0 and _weight_only_plan(33, n, k, 1)["form"] >= 0


@pytest.mark.parametrize("dtype", [0, 1])
def test_weight_only_scratch_is_what_the_plan_uses(dtype):
    """The bytes asked for are the partial sums of the plan that the call then takes, none where it is
    unsplit (1757 x 9360 -> 6560 in f32 asked for 131 MB that nothing used)."""
    L = _lib.lib()
    rng = random.Random(dtype)
    sizes = [(1757, 6560, 9360), (64, 768, 3072), (33, 256, 1024)]
    for _ in range(400):
        m, n, k = (int(2 ** rng.uniform(low, 11.5)) for low in (0, 0, 5))
        sizes.append((m, n, max(16, 2 * k) // 16 * 16 if rng.random() < 0.7 else 2 * k))
    split = 0
    for m, n, k in sizes:
        want = {}
        for ragged in (False, True):
            plan = _weight_only_plan(m, n, k, dtype, ragged)
            want[ragged] = 4 * m * n * plan["splits"] if plan["splits"] > 1 else 0
            if k < 16:
                want[ragged] = 0
        esz = 2 if dtype else 4
        assert L.dq8_weight_only_qgemm_workspace_bytes_ex(m, n, k, 1, dtype) == want[k % 16 != 0], (m, n, k)
        # aligned operands; activations and weights off 16 bytes; rows off 16 bytes
        for x, ldx, w, ldw, ragged in ((256, k, 512, k, k % 16 != 0), (256 + esz, k, 512, k, True),
                                       (256, k, 513, k, True), (256, k + 1, 512, k, True), (256, k, 512, k + 1, True)):
            got = L.dq8_weight_only_qgemm_workspace_bytes_for(x, dtype, ldx, w, ldw, 1, m, n, k)
            assert got == want[ragged], (m, n, k, ldx, ldw)
        # weights as [K, N]: their copy in front, which is aligned wherever K is
        got = L.dq8_weight_only_qgemm_workspace_bytes_for(256, dtype, k, 513, n, 0, m, n, k)
        assert got == ((n * k + 255) // 256 * 256 + want[k % 16 != 0] if want[k % 16 != 0] else n * k)
        split += want[k % 16 != 0] > 0
    assert split >= 40 and split < 300
    # operands that the tiles cannot address run without a split
    assert L.dq8_weight_only_qgemm_workspace_bytes_for(256, dtype, 1 << 23, 512, 3072, 1, 64, 768, 3072) == 0


@pytest.mark.parametrize("m,n,k,out,kernel", [
    # up to 256 tiles of 32 x 32, then of 32 x 64, then (from 1280 of k on) of 64 x 64, of 96 x 64
    (512, 512, 1008, 1, "wave_32x32_w4"), (512, 512, 1024, 1, "wave_32x32_w8"), (512, 513, 1024, 4, "wave_32x64_w4"),
    (513, 512, 1024, 1, "wave_32x64_w4"), (513, 960, 2048, 1, "wave_32x64_w4"), (512, 1024, 256, 4, "wave_32x64_w4"),
    (1024, 1024, 1280, 1, "wave_64x64_w4"), (1024, 1024, 1264, 1, "pipe_64x64x128"), (1025, 1024, 1280, 1, "pipe_64x64x128"),
    (1300, 1024, 2048, 1, "wave_96x64_w4"), (1300, 1024, 2032, 1, "pipe_64x64x128"), (1300, 1024, 2560, 4, "wave_96x64_w4"),
    (1300, 1024, 2544, 4, "pipe_64x64x128"), (1537, 1024, 2048, 1, "pipe_64x64x128"),
    # int8 rows off 16 bytes, 8192 of k
    (512, 504, 1024, 1, "wave_32x32_w8"), (512, 504, 1008, 1, "pipe_64x64x128"), (512, 504, 1024, 4, "wave_32x32_w8"),
    (1024, 1000, 2288, 1, "pipe_64x64x128_k2"), (1024, 1000, 2304, 1, "wave_64x64_w4"), (1300, 1000, 2544, 1, "pipe_64x64x128"),
    (1300, 1000, 2560, 1, "wave_96x64_w4"), (512, 512, 8176, 1, "wave_32x32_w8"), (512, 512, 8192, 1, "pipe_64x64x128_k4"),
    # few rows: the small-M kernel where it is estimated as fast
    (64, 768, 768, 1, "skinny_16"), (16, 4096, 1088, 1, "skinny_16"), (128, 384, 2048, 1, "skinny_16"),
    (320, 64, 512, 1, "skinny_16"), (321, 64, 512, 1, "wave_32x32_w4"), (256, 72, 1024, 1, "skinny_16"),
    (257, 72, 1024, 1, "wave_32x32_w8"),
    (118, 1536, 5248, 1, "wave_32x32_w8"), (34, 3232, 5392, 1, "wave_32x32_w8"), (30, 8640, 1088, 1, "wave_32x64_w4"),
    (16, 16448, 4096, 1, "pipe_64x64x128_k2"),
    # two 64 x 64 tiles to a compute unit, then 128 x 128 ones on eight waves, four for a deep k
    (2048, 1024, 768, 1, "pipe_64x64x128"), (2049, 1024, 768, 1, "pipe_128x128x128_w8"), (512, 4096, 2032, 1, "pipe_64x64x128"),
    (512, 4096, 2048, 1, "pipe_128x128x128_w8"), (1024, 2048, 3072, 4, "pipe_64x64x128"),
    (4096, 1152, 768, 1, "pipe_128x128x128_w8"), (4096, 1152, 4096, 1, "pipe_128x128x128")])
def test_few_tiles_run_on_waves_of_their_own(m, n, k, out, kernel):
    """The smallest tile of which a launch has one per compute unit: 343 x 512 x 4608 took 11.9 us on 64 x 64
    tiles, 7.1 on these; one more than that and a compute unit does two."""
    assert _lib.hooks().dq8_qgemm_kernel_name(m, n, k, out).decode() == kernel


WORDS, SMALL_M, REGISTERS, COPIED = 1, 2, 3, 0


def rows_kernel(m, n, k, lda=0, ldw=0, a_at=0, w_at=0, zw=0, out_bytes=1):
    form = C.c_int()
    name = _lib.hooks().dq8_qgemm_rows_kernel(m, n, k, lda or k, ldw or k, a_at, w_at, zw, out_bytes, C.byref(form))
    return form.value, name.decode()


@pytest.mark.parametrize("m,n,k,form,kernel", [
    # tiles on waves of their own estimated at or below the small-M kernel, in the forms next to them too
    (400, 256, 500, WORDS, "wave_32x32_w8"), (335, 1152, 324, WORDS, "wave_32x64_w4"), (1023, 897, 4108, WORDS, "wave_64x64_w4"),
    (1300, 1024, 2500, WORDS, "pipe_64x64x128"), (320, 513, 8204, WORDS, "pipe_64x64x128_k2"),
    (4097, 1281, 264, WORDS, "pipe_128x128x128_w8"), (4090, 3500, 396, WORDS, "pipe_256x256x128_w8"),
    # the small-M kernel estimated below them: within the limits it has by itself, else those tiles from 128 of k on
    (256, 64, 2000, SMALL_M, "skinny_16"), (16, 768, 500, SMALL_M, "skinny_16"), (257, 64, 2000, WORDS, "wave_32x32_w8"),
    (283, 618, 2628, WORDS, "wave_32x32_w8"), (130, 1306, 1416, WORDS, "wave_32x32_w8"), (320, 64, 500, WORDS, "wave_32x32_w8"),
    (32, 8640, 2052, WORDS, "wave_32x64_w4"), (320, 64, 132, WORDS, "wave_32x32_w8"), (320, 64, 124, REGISTERS, "pipe_64x64x128"),
    # rows at other bytes
    (283, 618, 2029, REGISTERS, "pipe_64x64x128"), (283, 618, 2629, COPIED, ""), (4097, 1281, 265, COPIED, "")])
def test_rows_off_16_bytes_keep_the_choice_that_was_made_for_them(m, n, k, form, kernel):
    """Of 33 to 330 rows on four bytes an eighth had the small-M kernel chosen against the tiles and then ran on
    neither, but on 64 x 64 tiles through registers: 297 x 530 x 4892 13.2 us in place of 7.1."""
    assert rows_kernel(m, n, k) == (form, kernel)


def test_rows_of_drawn_products_run_on_what_was_compared():
    """Whole words, 128 of k and more: nothing through registers or copied first where a form for words exists."""
    rng = random.Random(5)
    for _ in range(2000):
        m, n = (int(2 ** rng.uniform(1, 12)) for _ in range(2))
        k = 4 * int(2 ** rng.uniform(5, 11))
        assert rows_kernel(m, n, k, k + 4, k + 12, 4, 8, out_bytes=rng.choice((1, 4)))[0] in (WORDS, SMALL_M), (m, n, k)
        assert rows_kernel(m, n, k, k + 4, k + 12, 4, 8, zw=3)[0] in (COPIED, SMALL_M)
        assert rows_kernel(m, n, k, k + 4, k + 12, 4, 9)[0] in (COPIED, SMALL_M, REGISTERS)
