"""Which kernel, tiles and shares a matmul gets at both sides of the lines of its rules (no device is touched)."""
import ctypes as C

import pytest

from coeus_amd import _lib


def plan(dtype, k, n, rows, prompt=0):
    p = _lib.CMatmulPlan()
    assert _lib.load().coeus_plan_matmul(dtype, k, n, rows, prompt, C.byref(p)) == 0
    return p


def test_what_no_weight_can_be_is_refused():
    p, call = _lib.CMatmulPlan(), _lib.load().coeus_plan_matmul
    for dtype, k, n, rows, prompt in [(9, 64, 64, 1, 0), (0, 0, 64, 1, 0), (0, 64, 0, 1, 0), (3, 48, 64, 1, 0), (0, 64, 64, 0, 0), (0, 64, 64, 17, 0), (0, 64, 64, 0, 1)]:
        assert call(dtype, k, n, rows, prompt, C.byref(p)) != 0
    assert call(0, 64, 64, 1, 0, None) != 0


# Few chunks of 128: a tile of 16 outputs or two a workgroup, a wave per chunk (six tiles of one wave were 12.9 us at 64 x 16400 and 16 rows, one is 6.3)
@pytest.mark.parametrize("dtype,k,n,outputs,waves", [
    (_lib.W_Q4_0, 64, 4096, 16, 1), (_lib.W_Q4_0, 64, 16400, 16, 1), (_lib.W_Q8_0, 128, 100000, 16, 1), (_lib.W_Q4_0, 256, 16400, 16, 2), (_lib.W_Q4_0, 256, 32768, 16, 2),
    (_lib.W_Q4_0, 256, 32784, 32, 2), (_lib.W_Q8_0, 384, 24576, 16, 3), (_lib.W_Q8_0, 512, 24592, 32, 4), (_lib.W_Q4_0, 512, 8192, 16, 4), (_lib.W_Q4_0, 768, 16400, 48, 6),
    (_lib.W_Q4_0, 1024, 16400, 48, 8), (_lib.W_Q4_0, 1152, 16400, 96, 9), (_lib.W_Q4_0, 4096, 22016, 96, 12), (_lib.W_Q8_0, 4096, 22016, 48, 8), (_lib.W_Q8_0, 768, 50257, 32, 3),
    (_lib.W_Q8_0, 768, 768, 16, 6), (_lib.W_Q4_0, 11008, 4096, 16, 12)])
@pytest.mark.parametrize("rows", [5, 16])
def test_decode_rows_on_quantised_weights(dtype, k, n, outputs, waves, rows):
    p = plan(dtype, k, n, rows)
    assert (p.kernel, p.tile_cols, p.waves) == (b"gemv_rows_kernel", outputs, waves)


def test_decode_batches_of_up_to_four_on_quantised_weights():
    assert all(plan(d, 768, 2304, b).kernel == b"gemv_quad_kernel" for d in (_lib.W_Q8_0, _lib.W_Q4_0) for b in (1, 2, 3, 4))


# 3 and 4 rows: gemv_rows_kernel from k = 1024 on; Q8_0 not where the quads of up to 256 tiles are one pass of few or many waves (4 rows, quads and rows: 1056 x 1024
# 5.6 and 5.4 us, 1152 x 4096 6.2 and 6.1, 1280 x 2048 5.9 and 5.9)
@pytest.mark.parametrize("dtype,k,n,rows", [
    (_lib.W_Q4_0, 992, 4096, False), (_lib.W_Q4_0, 1024, 64, True), (_lib.W_Q4_0, 8192, 2048, True), (_lib.W_Q4_0, 4096, 32000, True), (_lib.W_Q8_0, 992, 4096, False),
    (_lib.W_Q8_0, 1024, 4096, True), (_lib.W_Q8_0, 1056, 4096, True), (_lib.W_Q8_0, 1152, 256, True), (_lib.W_Q8_0, 1184, 4096, False), (_lib.W_Q8_0, 2048, 4096, False), (_lib.W_Q8_0, 2048, 4098, True), (_lib.W_Q8_0, 2080, 1024, True),
    (_lib.W_Q8_0, 3072, 768, True), (_lib.W_Q8_0, 3104, 768, False), (_lib.W_Q8_0, 8192, 2048, False), (_lib.W_Q8_0, 8224, 2048, True)])
def test_three_and_four_rows_on_quantised_weights(dtype, k, n, rows):
    want = b"gemv_rows_kernel" if rows else b"gemv_quad_kernel"
    assert [plan(dtype, k, n, b).kernel for b in (1, 2, 3, 4, 5)] == [b"gemv_quad_kernel"] * 2 + [want] * 2 + [b"gemv_rows_kernel"]


# One row: where two weight rows a wave were slower than what there was before (bf16 64 x 128000 2.98 times, 512 x 50257 1.16), or are than a wave a row (f32 3072 x 2304 1.15 times,
# x 3600 1.03, but x 4096 0.98)
@pytest.mark.parametrize("dtype,k,n,kernel", [
    (_lib.W_BF16, 64, 16384, b"gemv_mfma_kernel"), (_lib.W_BF16, 512, 50257, b"gemv_mfma_kernel"), (_lib.W_BF16, 512, 16383, b"gemv_many_kernel"),
    (_lib.W_BF16, 576, 50257, b"gemv_many_kernel"), (_lib.W_BF16, 520, 50257, b"gemv_many_kernel"), (_lib.W_BF16, 200, 50257, b"gemv_many_kernel"),
    (_lib.W_BF16, 11008, 3072, b"gemv_mfma_kernel"), (_lib.W_BF16, 11008, 2048, b"gemv_many_kernel"), (_lib.W_BF16, 11008, 4096, b"gemv_many_kernel"),
    (_lib.W_BF16, 8192, 3072, b"gemv_many_kernel"), (_lib.W_BF16, 16384, 4608, b"gemv_dense_kernel"), (_lib.W_BF16, 16384, 6144, b"gemv_many_kernel"),
    (_lib.W_BF16, 16384, 4096, b"gemv_many_kernel"), (_lib.W_BF16, 770, 770, b"gemv_dense_kernel"), (_lib.W_BF16, 768, 50257, b"gemv_many_kernel"),
    (_lib.W_BF16, 512, 768, b"gemv_dense_kernel"), (_lib.W_BF16, 448, 8192, b"gemv_dense_kernel"), (_lib.W_BF16, 512, 8193, b"gemv_many_kernel"), (_lib.W_BF16, 520, 768, b"gemv_many_kernel"),
    (_lib.W_F32, 3072, 2304, b"gemv_dense_kernel"), (_lib.W_F32, 3072, 2048, b"gemv_many_kernel"), (_lib.W_F32, 1536, 3201, b"gemv_dense_kernel"),
    (_lib.W_F32, 3072, 1900, b"gemv_many_kernel"), (_lib.W_F32, 3072, 1890, b"gemv_dense_kernel"), (_lib.W_F32, 3072, 3600, b"gemv_dense_kernel"), (_lib.W_F32, 3072, 4090, b"gemv_many_kernel"),
    (_lib.W_F32, 2048, 9216, b"gemv_dense_kernel"), (_lib.W_F32, 2048, 17408, b"gemv_many_kernel"), (_lib.W_F32, 4096, 22016, b"gemv_dense_kernel"), (_lib.W_F32, 768, 32000, b"gemv_dense_kernel"),
    (_lib.W_F32, 1032, 8192, b"gemv_dense_kernel"), (_lib.W_F32, 1024, 50257, b"gemv_dense_kernel"),
    (_lib.W_F32, 768, 50257, b"gemv_many_kernel"), (_lib.W_F32, 768, 11008, b"gemv_dense_kernel"), (_lib.W_F32, 512, 50257, b"gemv_dense_kernel"),
    (_lib.W_F32, 768, 3072, b"gemv_dense_kernel"), (_lib.W_F32, 3072, 768, b"gemv_dense_kernel")])
def test_decode_of_one_row(dtype, k, n, kernel):
    assert plan(dtype, k, n, 1).kernel == kernel


# Up to 1024 rows of more than two steps: a wave each (bf16 11008 x 1024 8.3 us with two rows a wave, 6.9 so)
@pytest.mark.parametrize("k,n,kernel", [(1024, 1024, b"gemv_many_kernel"), (1032, 1024, b"gemv_dense_kernel"), (1032, 1025, b"gemv_many_kernel"),
                                        (11008, 1024, b"gemv_dense_kernel"), (11008, 1025, b"gemv_many_kernel")])
def test_few_long_rows_of_bf16(k, n, kernel):
    assert plan(_lib.W_BF16, k, n, 1).kernel == kernel


# Several rows on few outputs: tiles of 4 or 8 weight rows, sixteen lines of parts of k (f32 3072 x 768, 4 rows 8.3 us with tiles of 16, 5.1 so)
@pytest.mark.parametrize("dtype,k,n,rows,cols,waves", [
    (_lib.W_F32, 768, 768, 4, 4, 4), (_lib.W_F32, 3072, 768, 4, 4, 6), (_lib.W_F32, 3072, 768, 5, 8, 8), (_lib.W_F32, 3072, 768, 9, 16, 16), (_lib.W_F32, 8192, 1024, 4, 4, 16),
    (_lib.W_F32, 8192, 2048, 8, 8, 16), (_lib.W_F32, 2048, 2048, 2, 8, 8), (_lib.W_F32, 2048, 2049, 4, 16, 8), (_lib.W_F32, 1024, 4608, 4, 16, 4), (_lib.W_F32, 4096, 1024, 3, 4, 8), (_lib.W_F32, 768, 768, 2, 4, 4), (_lib.W_F32, 1536, 1024, 3, 4, 6), (_lib.W_F32, 128, 768, 2, 16, 4),
    (_lib.W_F32, 96, 700, 4, 16, 3), (_lib.W_BF16, 768, 768, 4, 16, 4), (_lib.W_BF16, 1024, 1024, 4, 4, 2), (_lib.W_BF16, 1024, 1024, 5, 16, 8), (_lib.W_BF16, 3072, 768, 4, 4, 6),
    (_lib.W_BF16, 3072, 768, 8, 8, 12), (_lib.W_BF16, 5632, 2048, 4, 4, 11), (_lib.W_BF16, 5632, 2048, 5, 8, 8), (_lib.W_BF16, 4096, 2048, 4, 8, 16), (_lib.W_BF16, 2048, 10272, 4, 16, 8),
    (_lib.W_BF16, 4096, 12352, 4, 4, 8), (_lib.W_BF16, 4096, 12352, 5, 8, 16), (_lib.W_BF16, 8192, 8192, 4, 4, 16), (_lib.W_BF16, 8192, 8192, 8, 16, 8), (_lib.W_BF16, 11008, 4096, 4, 16, 8),
    (_lib.W_BF16, 3072, 768, 16, 16, 16)])
def test_several_rows_on_dense_weights(dtype, k, n, rows, cols, waves):
    p = plan(dtype, k, n, rows)
    assert (p.kernel, p.tile_cols, p.waves) == (b"gemv_mfma_kernel", cols, waves)


# f32 beyond 4096 outputs, where parts of k or four waves were slower than tiles of 16 with sixteen: us, sixteen / parts or four / now: 4 rows of 8704 x 8192
# 44.9 / 67.3 / 44.1, 8224 x 8192 48.1 / 60.1 / 46.2, 5632 x 8192 30.5 / 36.8 / 29.3, 16 of 4096 x 8192 26.5 / 30.4 / 24.6; and 256 pairs: 4 rows of 8192 x 4096 with sixteen,
# eight and twelve waves 27.4 / 30.0 / 24.0
@pytest.mark.parametrize("k,n,rows,cols,waves", [
    (8704, 8192, 4, 16, 8), (8704, 8192, 2, 16, 8), (8224, 8192, 4, 16, 8), (5632, 8192, 8, 16, 8), (4096, 8192, 16, 16, 8), (4096, 5121, 4, 16, 8), (4096, 5120, 4, 4, 8),
    (5632, 5000, 4, 4, 11), (8704, 4112, 4, 8, 16), (9216, 4112, 4, 8, 16), (8192, 8192, 8, 8, 16), (8192, 8192, 4, 4, 16), (16384, 4112, 16, 16, 4), (4064, 8192, 16, 16, 4),
    (2048, 8192, 4, 16, 4), (8192, 4096, 4, 16, 12), (8192, 4096, 8, 16, 12), (8192, 4096, 16, 16, 16), (16384, 4096, 4, 16, 12), (12288, 4096, 4, 16, 8), (8224, 4096, 4, 16, 8)])
def test_wide_rows_of_f32(k, n, rows, cols, waves):
    p = plan(_lib.W_F32, k, n, rows)
    assert (p.kernel, p.tile_cols, p.waves) == (b"gemv_mfma_kernel", cols, waves)


# bf16, 5 - 8 rows beyond 4096 outputs: two parts of k where the waves' shares are two pairs then (2560 x 12352 20.4 us in one part, 14.2 in two; 4224 x 8192 17.0 and 24.1)
@pytest.mark.parametrize("k,n,rows,cols,waves", [
    (2048, 8192, 8, 16, 8), (2176, 4098, 8, 8, 9), (2560, 12352, 5, 8, 10), (3584, 22016, 8, 8, 14), (3968, 4097, 8, 8, 16), (4096, 12352, 8, 8, 16), (2112, 12352, 8, 16, 8),
    (4160, 8192, 8, 16, 8), (4224, 8192, 8, 16, 8), (2560, 4096, 8, 16, 8), (2560, 12352, 9, 16, 16)])
def test_two_parts_of_eight_rows(k, n, rows, cols, waves):
    p = plan(_lib.W_BF16, k, n, rows)
    assert (p.kernel, p.tile_cols, p.waves) == (b"gemv_mfma_kernel", cols, waves)


# f32, short rows of very many outputs: four waves a workgroup took 1.14 times as long as those that have two pairs each (128 x 50257, 2 - 16 rows)
@pytest.mark.parametrize("k,n,rows,waves", [
    (96, 28747, 4, 2), (128, 50257, 2, 2), (128, 50257, 16, 2), (320, 28747, 8, 5), (512, 50257, 4, 8), (128, 20001, 4, 2), (128, 20000, 4, 4), (544, 50257, 4, 4),
    (320, 8192, 4, 4), (64, 28747, 8, 2)])
def test_short_rows_of_f32(k, n, rows, waves):
    p = plan(_lib.W_F32, k, n, rows)
    assert (p.kernel, p.tile_cols, p.waves) == (b"gemv_mfma_kernel", 16, waves)


# bf16, waves by pairs a wave: eight waves of three pairs were slower than twelve of two (4 rows of 1536 x 12352 10.7 us and 8.5, 8 of 1536 x 5000 7.1 and 6.4), eight of 32
# where sixteen keep two in registers (4 of 2048 x 12352 12.4 and 11.6), eight that begin 4 KiB apart (4 of 16384 x 3600 26.2, with twelve 22.4); sixteen of 33 and more
# (8 of 2112 x 12352 21.2, with eight 15.7)
@pytest.mark.parametrize("k,n,rows,waves", [
    (1536, 12352, 4, 12), (1536, 5000, 8, 12), (1536, 8192, 4, 8), (2048, 12288, 4, 8), (2048, 12304, 4, 16), (2048, 12352, 2, 16), (2048, 4096, 8, 8), (2048, 8192, 5, 8),
    (2048, 8208, 8, 16), (2112, 12352, 8, 8), (2112, 12352, 16, 16), (4224, 4096, 4, 8), (16384, 3600, 4, 12), (16384, 6176, 8, 12), (16384, 3072, 1, 12), (11008, 3072, 1, 8),
    (11264, 3072, 1, 8), (32768, 3072, 8, 12), (24576, 3072, 8, 8), (11008, 4096, 16, 16)])
def test_waves_of_bf16_rows(k, n, rows, waves):
    p = plan(_lib.W_BF16, k, n, rows)
    assert (p.kernel, p.tile_cols, p.waves) == (b"gemv_mfma_kernel", 16, waves)


# Prompts: the shapes that test_gpu_narrow_gemm.py, test_gpu_sum_error.py and test_gpu_large_tiles.py multiply reach all five small tiles, shares of k on
# small and on large ones, and one workgroup a large tile
@pytest.mark.parametrize("m,k,n,kernel,rows,cols,shared", [
    (65, 64, 128, b"gemm_narrow_kernel", 128, 64, False), (512, 3072, 768, b"gemm_narrow_kernel", 128, 64, True), (201, 4096, 4098, b"gemm_narrow_kernel", 128, 128, True),
    (257, 1024, 7000, b"gemm_narrow_kernel", 128, 96, False), (201, 1024, 22016, b"gemm_narrow_kernel", 256, 96, False), (2036, 4096, 2560, b"gemm_narrow_kernel", 256, 96, False),
    (700, 2048, 8192, b"gemm_narrow_kernel", 256, 128, False), (300, 11008, 4096, b"gemm_h256k64_kernel", 256, 256, True), (5000, 64, 5100, b"gemm_h256k64_kernel", 256, 256, False),
    (17, 96, 512, b"gemm_h256_kernel", 256, 256, False), (300, 90, 512, b"gemm_h_kernel", 128, 128, False)])
def test_prompts(m, k, n, kernel, rows, cols, shared):
    p = plan(_lib.W_BF16, k, n, m, 1)
    assert (p.kernel, p.tile_rows, p.tile_cols, p.shares > 1) == (kernel, rows, cols, shared)
    if k % 32 == 0:
        assert plan(_lib.W_Q8_0, k, n, max(m, 65), 1).kernel == plan(_lib.W_BF16, k, n, max(m, 65), 1).kernel


def test_other_prompts():
    assert plan(_lib.W_Q4_0, 4096, 4096, 64, 1).kernel == b"gemm_qskinny_kernel" and plan(_lib.W_Q4_0, 4096, 4096, 65, 1).kernel == b"gemm_narrow_kernel"
    assert plan(_lib.W_Q4_0, 4096, 22016, 4071, 1).tail_shares == 2 and plan(_lib.W_BF16, 512, 4090, 4100, 1).tail_shares == 2
    assert plan(_lib.W_F32, 768, 768, 5, 1).kernel == b"gemv_mfma_kernel" and plan(_lib.W_F32, 768, 768, 128, 1).kernel == b"gemm_f32_small_kernel"
    assert plan(_lib.W_F32, 3072, 768, 128, 1).shares == 8 and plan(_lib.W_F32, 768, 50257, 128, 1).kernel == b"gemm_f32_kernel"


# f32 prompts of very many outputs: the tiles' grid has one dimension, of at most 2^32 threads (17 rows of 4 x 2^29, 36 GB of results: 2^23 tiles of eight waves are one thread too many)
@pytest.mark.parametrize("k,n,m", [(4, 1 << 28, 17), (4, 1 << 28, 32), (4, (1 << 28) - 256, 32), (4, (1 << 28) + 4, 33), (4, 1 << 29, 17), (4, 1 << 29, 200), (8192, 1 << 22, 1024), (64, 1 << 24, 5000),
                                   (4, 1 << 20, 100000), (4, 1 << 16, 1 << 22), (4, 1 << 31, 17), (1 << 20, 256, 1 << 20)])
def test_the_grid_of_f32_tiles(k, n, m):
    p = plan(_lib.W_F32, k, n, m, 1)
    tiles = -(-m // p.tile_rows) * -(-n // p.tile_cols)
    if p.kernel in (b"gemm_f32_small_kernel", b"gemm_f32_kernel"):
        assert -(-tiles * p.shares // 8) * 8 * p.waves * 64 < 1 << 32
    else:
        assert p.kernel == b"gemm_f32_any_kernel" and tiles >= 1 << 22
