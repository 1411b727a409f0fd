"""GPU parity: evk::ai::matmul through the C ABI vs the CPU oracle.

Bar: fp16 outputs within max-abs/relative 1e-2 of the fp32-accumulated
oracle; known-answer tests bit-exact (reference tests.h:163-219).
"""
import numpy as np
import pytest

from conftest import assert_close_f16, f32, from_dev, to_dev

pytestmark = pytest.mark.gpu


def f16(x):
    return np.asarray(x, np.float32).astype(np.float16).view(np.uint16)


def run_mm(evk, dev, a, b, c_shape, ta=False, tb=False, acc=False, c0=None, tiles=(80, 80)):
    import torch
    A, B = to_dev(a, dev), to_dev(b, dev)
    C = to_dev(c0, dev) if c0 is not None else torch.zeros(c_shape, dtype=torch.float16, device=dev)
    evk.matmul(A, B, C, ta, tb, acc, *tiles)
    torch.cuda.synchronize()
    return from_dev(C)


def test_identity_kat_400(dev, orc):
    # tests.h:163-194 with the default 80x80 tile hints
    import evk_amd as evk
    n = 400
    eye2 = np.zeros((n, n), np.uint16)
    eye2[np.arange(n), np.arange(n)] = f16(2.0)
    c = run_mm(evk, dev, eye2, eye2, (n, n))
    want = np.zeros((n, n), np.uint16)
    want[np.arange(n), np.arange(n)] = f16(4.0)
    assert np.array_equal(c, want)


def test_broadcast_kat(dev, orc):
    # tests.h:196-219: a (1,32,32) ones, b (32,32) identity, c (3,32,32)
    import evk_amd as evk
    ones = np.full((1, 32, 32), f16(1.0), np.uint16)
    eye = np.zeros((32, 32), np.uint16)
    eye[np.arange(32), np.arange(32)] = f16(1.0)
    c = run_mm(evk, dev, ones, eye, (3, 32, 32), tiles=(16, 16))
    assert np.all(c == f16(1.0))


def test_config1_gemm_1024(dev, orc):
    import evk_amd as evk
    a = orc.uniform_f16((1024, 1024), 101)
    b = orc.uniform_f16((1024, 1024), 102)
    got = run_mm(evk, dev, a, b, (1024, 1024))
    assert_close_f16(got, orc.matmul(a, b), what="C1 1024^3")


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("M,N,K", [(200, 136, 72), (64, 64, 64), (520, 264, 328), (32, 8, 8)])
def test_transposes_ragged(dev, orc, ta, tb, M, N, K):
    import evk_amd as evk
    a = orc.uniform_f16((K, M) if ta else (M, K), 11 + M)
    b = orc.uniform_f16((N, K) if tb else (K, N), 12 + N)
    got = run_mm(evk, dev, a, b, (M, N), ta, tb)
    assert_close_f16(got, orc.matmul(a, b, transpose_a=ta, transpose_b=tb), what=f"{ta}{tb} {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(600, 1100, 968), (1536, 1536, 256)])
def test_large_tile_paths(dev, orc, M, N, K):
    import evk_amd as evk
    a = orc.uniform_f16((M, K), 41)
    b = orc.uniform_f16((K, N), 42)
    got = run_mm(evk, dev, a, b, (M, N))
    assert_close_f16(got, orc.matmul(a, b), what=f"{M}x{N}x{K}")


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_k_groups_ragged(dev, orc, ta, tb):
    """Grids that fit the CUs once with a long K run two K groups per workgroup
    whose sums meet in LDS: ragged M, N and a K that is not a multiple of the
    64-deep tile (the last group's range is shorter), every operand order."""
    import evk_amd as evk
    M, N, K = 200, 136, 1096
    a = orc.uniform_f16((K, M) if ta else (M, K), 61 + ta)
    b = orc.uniform_f16((N, K) if tb else (K, N), 62 + tb)
    got = run_mm(evk, dev, a, b, (M, N), ta, tb)
    assert_close_f16(got, orc.matmul(a, b, transpose_a=ta, transpose_b=tb), what=f"K groups {ta}{tb}")


def test_k_groups_batched_acc(dev, orc):
    """K groups with accumulation into C (one rounding of the fp32 sum per
    element) over a batch."""
    import evk_amd as evk
    a = orc.uniform_f16((3, 96, 2056), 63)
    b = orc.uniform_f16((2056, 72), 64)
    c0 = orc.uniform_f16((3, 96, 72), 65)
    got = run_mm(evk, dev, a, b, None, acc=True, c0=c0)
    assert_close_f16(got, orc.matmul(a, b, c=c0, acc_c=True), what="K groups batched acc")


def test_batched_broadcast_acc(dev, orc):
    import evk_amd as evk
    a = orc.uniform_f16((3, 96, 80), 51)
    b = orc.uniform_f16((80, 48), 52)
    c0 = orc.uniform_f16((3, 96, 48), 53)
    got = run_mm(evk, dev, a, b, None, acc=True, c0=c0)
    assert_close_f16(got, orc.matmul(a, b, c=c0, acc_c=True), what="batched acc")
    # broadcast A over a batched B, transposed B
    a1 = orc.uniform_f16((40, 64), 54)
    b3 = orc.uniform_f16((2, 24, 64), 55)
    got = run_mm(evk, dev, a1, b3, (2, 40, 24), tb=True)
    want = orc.matmul(a1, b3, transpose_b=True, out_shape=(2, 40, 24))
    assert_close_f16(got, want, what="broadcast A")


def test_unaligned_fallback(dev, orc):
    import evk_amd as evk
    a = orc.uniform_f16((13, 7), 61)
    b = orc.uniform_f16((7, 5), 62)
    got = run_mm(evk, dev, a, b, (13, 5))
    assert_close_f16(got, orc.matmul(a, b), what="scalar path")


@pytest.mark.parametrize("M", [1, 4, 16])
def test_skinny_gemv_config5(dev, orc, M):
    import evk_amd as evk
    K, N = 4096, 11008
    a = orc.uniform_f16((M, K), 501 + M)
    b = orc.uniform_f16((K, N), 510)
    got = run_mm(evk, dev, a, b, (M, N))
    assert_close_f16(got, orc.matmul(a, b), what=f"gemv M={M}")
    # second call reuses the split-K workspace: must give identical bits
    got2 = run_mm(evk, dev, a, b, (M, N))
    assert np.array_equal(got, got2)


def test_skinny_acc_and_small(dev, orc):
    import evk_amd as evk
    # M <= 4 runs on the VALU kernel, 4 < M <= 16 on the MFMA one; K ranges of
    # 512 rows: single-range (direct C write) and ragged split-K cases
    for (M, K, N) in [(1, 768, 2304), (3, 3072, 768), (2, 8, 16), (1, 4096, 32000),
                      (5, 512, 64), (8, 1000, 136), (16, 520, 2000), (12, 4096, 1032), (9, 24, 40)]:
        a = orc.uniform_f16((M, K), 71 + K)
        b = orc.uniform_f16((K, N), 72 + N)
        c0 = orc.uniform_f16((M, N), 73)
        got = run_mm(evk, dev, a, b, None, acc=True, c0=c0)
        assert_close_f16(got, orc.matmul(a, b, c=c0, acc_c=True), what=f"gemv acc {M}x{K}x{N}")


def test_skinny_batched(dev, orc):
    """Batched skinny products: per-batch A over a shared B (MFMA kernel,
    split-K), and a shared A over per-batch B (VALU kernel)."""
    import evk_amd as evk
    a = orc.uniform_f16((3, 12, 1040), 81)
    b = orc.uniform_f16((1040, 200), 82)
    got = run_mm(evk, dev, a, b, (3, 12, 200))
    assert_close_f16(got, orc.matmul(a, b, out_shape=(3, 12, 200)), what="batched A")
    a1 = orc.uniform_f16((1, 520), 83)
    b3 = orc.uniform_f16((2, 520, 72), 84)
    got = run_mm(evk, dev, a1, b3, (2, 1, 72))
    assert_close_f16(got, orc.matmul(a1, b3, out_shape=(2, 1, 72)), what="batched B")


def _rows_check(orc, a, b, got, rows):
    want = orc.matmul(a[rows], b)
    assert_close_f16(got[rows], want, what="row sample")


def half_ulp(x):
    """Half an fp16 ulp of each |x| (the rounding bound of the fp16 store)."""
    ax = np.maximum(np.abs(x.astype(np.float64)), 2.0 ** -14)
    return 0.5 * 2.0 ** (np.floor(np.log2(ax)) - 10)


def test_config5_square_4096(dev, orc):
    import evk_amd as evk
    n = 4096
    a = orc.uniform_f16((n, n), 501)
    b = orc.uniform_f16((n, n), 502)
    got = run_mm(evk, dev, a, b, (n, n))
    rows = np.random.RandomState(0).choice(n, 48, replace=False)
    _rows_check(orc, a, b, got, np.sort(rows))
    # checksum over every row: C.1 == A.(B.1) up to the fp16 rounding of each
    # stored element (bounded by half an ulp) plus fp32 accumulation slack
    A, B = f32(a).astype(np.float64), f32(b).astype(np.float64)
    G = f32(got)
    err = np.abs(G.astype(np.float64).sum(1) - A @ B.sum(1))
    bound = half_ulp(G).sum(1) + 1e-2 * np.sqrt(n)
    assert np.all(err <= bound), float((err - bound).max())


def test_config5_qkv_shape(dev, orc):
    import evk_amd as evk
    M, N, K = 8192, 12288, 4096
    a = orc.uniform_f16((M, K), 503)
    b = orc.uniform_f16((K, N), 504)
    got = run_mm(evk, dev, a, b, (M, N))
    rows = np.sort(np.random.RandomState(1).choice(M, 16, replace=False))
    _rows_check(orc, a, b, got, rows)
    A, B = f32(a).astype(np.float64), f32(b).astype(np.float64)
    G = f32(got)
    err = np.abs(G.astype(np.float64).sum(0) - A.sum(0) @ B)
    bound = half_ulp(G).sum(0) + 1e-2 * np.sqrt(M)
    assert np.all(err <= bound), float((err - bound).max())


@pytest.mark.parametrize("ta", [False, True])
def test_operand_over_2gib(dev, orc, ta):
    """A 2.15 GB A operand (past the 32-bit buffer descriptors of the LDS-direct
    loads) runs on 64-bit addresses through registers; sampled rows of C and
    whole-matrix column sums are checked against fp32 on the host.  Inputs
    are drawn on the device from a seeded torch generator (2 GB is too much
    to push from the host in a test)."""
    import torch
    import evk_amd as evk
    M, K, N = 131072 + 64, 8192, 256
    assert M * K * 2 > 2**31
    g = torch.Generator(device=dev).manual_seed(7)
    shape_a = (K, M) if ta else (M, K)
    A = (torch.rand(shape_a, generator=g, device=dev, dtype=torch.float16) * 2 - 1)
    B = (torch.rand((K, N), generator=g, device=dev, dtype=torch.float16) * 2 - 1)
    C = torch.empty((M, N), dtype=torch.float16, device=dev)
    evk.matmul(A, B, C, ta, False, False)
    torch.cuda.synchronize()
    rows = torch.tensor([0, 1, 255, 256, 70000, M // 2 + 3, M - 65, M - 1], device=dev)
    a_rows = (A[:, rows].t() if ta else A[rows]).float().cpu().numpy()
    want = a_rows @ B.float().cpu().numpy()
    got = C[rows].float().cpu().numpy()
    assert np.abs(got - want).max() <= 1e-2 * (1 + np.abs(want).max())
    # every row: column sums of C against (column sums of A) . B
    a_sum = (A.float().sum(dim=1) if ta else A.float().sum(dim=0)).cpu().numpy()
    want_cs = a_sum @ B.float().cpu().numpy()
    got_cs = C.float().sum(dim=0).cpu().numpy()
    assert np.abs(got_cs - want_cs).max() <= 2e-3 * np.abs(want_cs).max() + 1.0
    del A, B, C
    torch.cuda.empty_cache()


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (65, 63, 64), (64, 66, 129), (130, 71, 1031), (1000, 1001, 77), (9, 3000, 515)])
def test_any_row_length(dev, orc, ta, tb, M, N, K):
    """Row lengths that are no multiple of a 16-byte chunk, in every operand
    order: tile edges, a K tail of one element, grids of one and of many
    tiles, the two-group K split (K >= 1024)."""
    import evk_amd as evk
    a = orc.uniform_f16((K, M) if ta else (M, K), 91 + M)
    b = orc.uniform_f16((N, K) if tb else (K, N), 92 + N)
    got = run_mm(evk, dev, a, b, (M, N), ta, tb)
    assert_close_f16(got, orc.matmul(a, b, transpose_a=ta, transpose_b=tb), what=f"{ta}{tb} {M}x{N}x{K}")


@pytest.mark.parametrize("shift", [(1, 0, 0), (0, 3, 0), (0, 0, 5), (7, 1, 2)])
def test_two_byte_aligned_operands(dev, orc, shift):
    """Operands that start off a 16-byte boundary (batched, accumulating, so
    each batch starts elsewhere), guarded by sentinels around C."""
    import torch
    import evk_amd as evk
    B, M, N, K = 3, 70, 88, 72
    a, b, c0 = orc.uniform_f16((B, M, K), 95), orc.uniform_f16((K, N), 96), orc.uniform_f16((B, M, N), 97)

    def at(x, off):
        buf = torch.full((x.size + 16,), 7.0, dtype=torch.float16, device=dev)
        buf[off:off + x.size] = to_dev(x, dev).reshape(-1)
        return buf, buf[off:off + x.size].view(x.shape)

    (_, A), (_, W), (buf, C) = at(a, shift[0]), at(b, shift[1]), at(c0, shift[2])
    evk.matmul(A, W, C, acc_c=True)
    torch.cuda.synchronize()
    assert_close_f16(from_dev(C), orc.matmul(a, b, c=c0, acc_c=True), what=f"shift {shift}")
    assert bool((buf[:shift[2]] == 7).all()) and bool((buf[shift[2] + c0.size:] == 7).all())


@pytest.mark.parametrize("K", [1, 63, 2741])
def test_weight_gradient_of_ragged_token_count(dev, orc, K):
    """X^T dY over K tokens: K is the row count of both operands and needs no
    multiple; the rows past K must not enter the sums (LDS-direct loads)."""
    import evk_amd as evk
    a, b, c0 = orc.uniform_f16((K, 136), 98), orc.uniform_f16((K, 264), 99), orc.uniform_f16((136, 264), 100)
    got = run_mm(evk, dev, a, b, None, True, False, True, c0)
    assert_close_f16(got, orc.matmul(a, b, c=c0, transpose_a=True, acc_c=True), what=f"K={K}")


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("M,N,K", [(2888, 2880, 552), (2320, 1736, 24), (1120, 1952, 1376), (336, 2752, 328), (40, 24, 24),
                                   (1136, 1824, 336), (1680, 264, 208), (24, 24, 72), (24, 88, 1248), (200, 24, 4104)])
def test_each_instance(dev, orc, ta, tb, M, N, K):
    """One product per instance of the MFMA kernel (256 x 256 down to 32 x 64
    tiles, one or two K groups, two to four LDS stages): ragged last tiles, K
    ranges of unequal length and groups without any; a sample of rows in every
    row tile against the oracle, accumulating into C."""
    import evk_amd as evk
    a = orc.uniform_f16((K, M) if ta else (M, K), 111 + M)
    b = orc.uniform_f16((N, K) if tb else (K, N), 112 + N)
    c0 = orc.uniform_f16((M, N), 113)
    got = run_mm(evk, dev, a, b, None, ta, tb, True, c0)
    rows = np.unique(np.r_[np.arange(0, M, 29), M - 1])
    A = f32(a[:, rows].T if ta else a[rows])
    want = (A @ f32(b.T if tb else b) + f32(c0[rows])).astype(np.float16).view(np.uint16)
    assert_close_f16(got[rows], want, what=f"{ta}{tb} {M}x{N}x{K}")


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 1, 1), (4100, 5, 5, 5), (3, 37, 33, 13), (2, 300, 301, 17), (1, 3000, 3, 23), (1, 257, 255, 80),
                                     (300, 3, 7, 81), (1, 1001, 1003, 2)])
def test_short_k(dev, orc, ta, tb, B, M, N, K):
    """Odd rows with a short K, accumulating, on both sides of the line between
    a thread per element and MFMA tiles; sentinels around C."""
    import torch
    import evk_amd as evk
    a = orc.uniform_f16((B, K, M) if ta else (B, M, K), 121 + M)
    b = orc.uniform_f16((B, N, K) if tb else (B, K, N), 122 + N)
    c0 = orc.uniform_f16((B, M, N), 123)
    buf = torch.full((c0.size + 16,), 7.0, dtype=torch.float16, device=dev)
    C = buf[5:5 + c0.size].view(c0.shape)
    C.copy_(to_dev(c0, dev))
    evk.matmul(to_dev(a, dev), to_dev(b, dev), C, ta, tb, True)
    torch.cuda.synchronize()
    want = orc.matmul(a, b, c=c0, transpose_a=ta, transpose_b=tb, acc_c=True)
    assert_close_f16(from_dev(C), want, what=f"{ta}{tb} {B}x{M}x{N}x{K}")
    assert bool((buf[:5] == 7).all()) and bool((buf[5 + c0.size:] == 7).all())


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_large_odd_rows(dev, orc, ta, tb):
    """Odd rows on 128 x 128 tiles through registers (the grids of the other
    such tests are small enough for 64 x 64), accumulating."""
    import evk_amd as evk
    M, N, K = 3001, 2003, 70
    a = orc.uniform_f16((K, M) if ta else (M, K), 131)
    b = orc.uniform_f16((N, K) if tb else (K, N), 132)
    c0 = orc.uniform_f16((M, N), 133)
    got = run_mm(evk, dev, a, b, None, ta, tb, True, c0)
    want = (f32(a.T if ta else a) @ f32(b.T if tb else b) + f32(c0)).astype(np.float16).view(np.uint16)
    assert_close_f16(got, want, what=f"{ta}{tb}")


def test_output_past_2_31_elements(dev):
    """More than 2^31 elements of C from small operands: rows at both ends and
    around the 2^31st element, and the sum of every row."""
    import torch
    import evk_amd as evk
    M, N, K = 70000, 32000, 64
    assert M * N > 2**31
    g = torch.Generator(device=dev).manual_seed(8)
    A = torch.rand((M, K), generator=g, device=dev, dtype=torch.float16) - 0.5
    B = torch.rand((K, N), generator=g, device=dev, dtype=torch.float16) - 0.5
    C = torch.full((M, N), 7.0, dtype=torch.float16, device=dev)
    evk.matmul(A, B, C)
    torch.cuda.synchronize()
    rows = torch.tensor([0, 1, 2**31 // N - 1, 2**31 // N, 2**31 // N + 1, M - 2, M - 1], device=dev)
    want = A[rows].double() @ B.double()
    assert (C[rows].double() - want).abs().max() <= 2e-3
    # fp16 rounding of up to 2^-11 |c| an element, sqrt(N) of them: far below 0.2
    for r0 in range(0, M, 10000):
        got = C[r0:r0 + 10000].float().sum(1).double()
        assert (got - A[r0:r0 + 10000].double() @ B.double().sum(1)).abs().max() <= 0.2
    del A, B, C
    torch.cuda.empty_cache()
