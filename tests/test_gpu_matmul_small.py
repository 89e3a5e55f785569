"""The GEMM kernels for few tiles, whose four waves split K (csrc/gemm_small.hip, gemm32_small.hip): stand-in for the reference's
examples/matmul.jl:21-58 and batchmatmul.jl:28-65 at small sizes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _operands(orc, M, N, K, T, pad, batch=1):
    """Integer-valued operands as views with NaN right behind every row and behind the arrays."""
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(-1, 2, (batch, K, M)).astype(np.float32); B = rng.integers(-1, 2, (batch, N, K)).astype(np.float32)
    lda, ldb = M + pad[0], K + pad[1]
    views = []
    for X, rows, cols, ld in ((A, K, M, lda), (B, N, K, ldb)):
        flat = torch.full((batch * rows * ld + 16,), float("nan"), dtype=T, device="cuda")
        v = flat[:batch * rows * ld].view(batch, rows, ld)[:, :, :cols]
        v.copy_(torch.from_numpy(X).to(T))
        views.append(v)
    return views[0], views[1], np.matmul(B, A)


@pytest.mark.parametrize("M,N,K,T,out32,pad,tile", [
    # 32 x 32: one tile and edges of one row / column, every number of stages per wave that ends differently (K = 256: one
    # each; 264, 320, 328, 511: a part-filled last stage), K - Kd = 0, 1, 7 and 8
    (8, 1, 256, torch.float16, True, (0, 0), "32x32"), (31, 33, 264, torch.bfloat16, True, (1, 0), "32x32"),
    (33, 31, 263, torch.float16, False, (0, 0), "32x32"), (256, 256, 320, torch.bfloat16, False, (0, 0), "32x32"),
    (257, 320, 328, torch.float16, True, (0, 0), "32x32"), (320, 255, 511, torch.bfloat16, True, (3, 5), "32x32"),
    (96, 2000, 513, torch.float16, False, (0, 7), "32x32"), (256, 320, 4096, torch.float16, True, (0, 0), "32x32"),
    # 64 x 32
    (1152, 320, 1813, torch.float16, True, (0, 0), "64x32"), (640, 513, 2112, torch.bfloat16, True, (0, 0), "64x32"),
    (1025, 450, 447, torch.float16, False, (2, 1), "64x32"),
    # 64 x 64
    (704, 897, 1408, torch.float16, True, (0, 0), "64x64"), (577, 1001, 961, torch.float16, False, (0, 0), "64x64"),
    (768, 725, 1280, torch.bfloat16, True, (8, 8), "64x64"),
    # 128 x 64
    (3648, 375, 3264, torch.float16, True, (0, 0), "128x64"), (1793, 927, 2499, torch.bfloat16, True, (0, 0), "128x64"),
    (1088, 1728, 2999, torch.float16, True, (1, 3), "128x64"),
])
def test_few_tiles_exact(ct, orc, M, N, K, T, out32, pad, tile):
    """Exact integer sums; C a view of a buffer with a sentinel."""
    A, B, ref = _operands(orc, M, N, K, T, pad)
    buf = torch.full((N + 2, M + 9), -77.0, dtype=torch.float32 if out32 else T, device="cuda")
    ct.matmul_kernel(A[0], B[0], buf[:N, :M], 64, 64, 64)
    assert ct.last_variant() == f"gemm16_small_{tile}x64"
    assert out32 or np.abs(ref).max() <= (2048 if T == torch.float16 else 256)
    assert np.array_equal(buf[:N, :M].float().cpu().numpy(), ref[0])
    assert bool((buf[N:] == -77.0).all()) and bool((buf[:, M:] == -77.0).all())


@pytest.mark.parametrize("M,N,K,nb", [(65, 100, 300, 3), (130, 129, 1000, 7), (72, 64, 257, 33)])
def test_few_tiles_batched_exact(ct, orc, M, N, K, nb):
    A, B, ref = _operands(orc, M, N, K, torch.float16, (0, 1), nb)
    C = torch.empty((nb, N, M), dtype=torch.float32, device="cuda")
    ct.batch_matmul_kernel(A, B, C, 64, 64, 64)
    assert ct.last_variant().startswith("gemm16_small_"), ct.last_variant()
    assert np.array_equal(C.cpu().numpy(), ref)


@pytest.mark.parametrize("M,N,K,small", [(512, 512, 255, False), (512, 512, 256, True), (256, 256, 4096, True), (256, 256, 4104, False),
                                         (2048, 1024, 320, False), (2049, 1024, 2048, False), (1536, 735, 576, True), (1664, 1792, 832, False),
                                         # estimated close to the other kernels: 128 x 64 tiles, and against a split
                                         (512, 3584, 1216, False), (832, 2240, 1280, False), (2816, 384, 2191, False), (512, 1443, 3043, True),
                                         (1249, 704, 4032, True)])
def test_both_sides_of_the_rule(ct, orc, M, N, K, small):
    A, B, ref = _operands(orc, M, N, K, torch.float16, (0, 0))
    C = torch.empty((N, M), dtype=torch.float32, device="cuda")
    ct.matmul_kernel(A[0], B[0], C, 64, 64, 64)
    assert ct.last_variant().startswith("gemm16_small_") == small, ct.last_variant()
    assert np.array_equal(C.cpu().numpy(), ref[0])


def test_few_tiles_infinities_and_nan_stay_in_their_rows_and_columns(ct, orc):
    A, B, ref = _operands(orc, 200, 96, 520, torch.bfloat16, (0, 0))
    A[0, 519, 7] = float("inf"); A[0, 3, 130] = float("nan")
    B[0, :, 519] = 1.0
    C = torch.empty((96, 200), dtype=torch.float32, device="cuda")
    ct.matmul_kernel(A[0], B[0], C, 64, 64, 64)
    want = B[0].cpu().double() @ A[0].cpu().double()
    assert torch.equal(C.cpu().double().nan_to_num(nan=-1e30), want.nan_to_num(nan=-1e30))


@pytest.mark.parametrize("M,N,K,nb,pad,kernel", [
    # one tile and edges of one row / column, stages per wave that end differently, K - Kd = 0 to 4
    (4, 1, 64, 1, (0, 0), "small_32x32x32"), (31, 33, 65, 2, (1, 0), "small_32x32x32"), (33, 31, 127, 5, (0, 0), "small_32x32x32"),
    (165, 543, 131, 4, (0, 0), "small_"), (192, 128, 320, 2, (0, 0), "small_32x32x32"), (130, 525, 449, 2, (3, 1), "small_32x32x32"),
    (128, 100, 1024, 2, (0, 0), "small_32x32x32"), (101, 63, 1023, 3, (0, 0), "small_32x32x32"),
    (720, 128, 500, 3, (0, 0), "small_64x32x32"), (249, 181, 384, 8, (0, 0), "small_64x32x32"), (629, 141, 143, 9, (2, 3), "small_64x32x32"),
    # the tiles of gemm32_big.hip where they are estimated to be the quicker ones
    (832, 384, 489, 12, (0, 0), "big_"), (320, 2007, 160, 10, (0, 0), "big_64x64x16_ring4"), (2056, 2311, 388, 1, (0, 0), "big_64x64x16_ring4"),
    (765, 256, 384, 8, (0, 0), "big_64x64x16_ring4"), (192, 1283, 383, 6, (0, 0), "big_64x64x16_ring4"),
    (576, 201, 384, 12, (0, 0), "big_64x64x16_ring4"),   # (two of them share a CU)
])
def test_few_fp32_tiles_exact(ct, orc, M, N, K, nb, pad, kernel):
    A, B, ref = _operands(orc, M, N, K, torch.float32, pad, nb)
    buf = torch.full((nb, N + 2, M + 5), -77.0, device="cuda")
    C = buf[:, :N, :M]
    if nb == 1:
        ct.matmul_kernel(A[0], B[0], C[0], 64, 64, 64)
    else:
        ct.batch_matmul_kernel(A, B, C, 64, 64, 64)
    assert ct.last_variant().startswith("gemm32_" + kernel), ct.last_variant()
    assert np.array_equal(C.cpu().numpy(), ref)
    assert bool((buf[:, N:] == -77.0).all()) and bool((buf[:, :, M:] == -77.0).all())


@pytest.mark.parametrize("K", [63, 64, 1024, 1025])
def test_fp32_infinities_and_nan_stay_in_their_rows_and_columns(ct, orc, K):
    A, B, ref = _operands(orc, 70, 40, K, torch.float32, (0, 0))
    A[0, K - 1, 7] = float("inf"); A[0, 3, 50] = float("nan")
    B[0, :, K - 1] = 1.0
    C = torch.empty((40, 70), device="cuda")
    ct.matmul_kernel(A[0], B[0], C, 64, 64, 64)
    assert ("small" in ct.last_variant()) == (64 <= K <= 1024), ct.last_variant()
    want = B[0].cpu().double() @ A[0].cpu().double()
    assert torch.equal(C.cpu().double().nan_to_num(nan=-1e30), want.nan_to_num(nan=-1e30))
