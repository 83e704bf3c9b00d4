"""mjt_matmul on the library's own kernels (kernels/gemm_mfma.h, kernels/gemm_plain.h), called through the C-ABI.
What the reference relays to a library GEMM is by definition broadcast * broadcast -> sum
(python/jittor/src/opt/tuner/matmul_tuner.cc:16-104), so the oracle is that meta-op expression for small
operands and the float64 matrix product of the same (rounded) operands beyond; every element is held to
1e-4 * sum_k |a_ik * b_kj| (float32 accumulation in another order), plus one rounding of a 16-bit result."""
import ctypes

import numpy as np
import pytest

from jittor_amd import _lib as L
from jittor_amd.dtypes import f32_to_bf16_bits
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _to_dev(arr):
    p = L.alloc(max(arr.nbytes, 256))
    L.h2d(p, arr)
    return p


def _operand(rng, shape, dt):
    """(what goes to the device, its exact float64 value)"""
    v = rng.standard_normal(shape).astype(np.float32)
    if dt == "bfloat16":
        bits = f32_to_bf16_bits(v)
        return bits, (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    if dt == "float16":
        h = v.astype(np.float16)
        return h, h.astype(np.float64)
    if dt == "float64":
        d = v.astype(np.float64) + 1e-9 * rng.standard_normal(shape)
        return d, d
    return v, v.astype(np.float64)


def _from_dev(ptr, shape, dt):
    if dt == "bfloat16":
        return (L.d2h(ptr, shape, np.uint16).astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    return L.d2h(ptr, shape, {"float16": np.float16, "float32": np.float32, "float64": np.float64}[dt]).astype(np.float64)


def _run(lib, dt, odt, M, K, N, ta, tb, batch=(), seed=0):
    rng = np.random.default_rng(seed)
    ash, bsh = tuple(batch) + ((K, M) if ta else (M, K)), tuple(batch) + ((N, K) if tb else (K, N))
    a_dev, a64 = _operand(rng, ash, dt)
    b_dev, b64 = _operand(rng, bsh, dt)
    pa, pb = _to_dev(a_dev), _to_dev(b_dev)
    csh = tuple(batch) + (M, N)
    pc = L.alloc(max(int(np.prod(csh)) * 8, 256))
    try:
        ta_, tb_, tc_ = L.tensor(pa, dt, ash), L.tensor(pb, dt, bsh), L.tensor(pc, odt, csh)
        L.check(lib.mjt_matmul(ctypes.byref(ta_), ctypes.byref(tb_), ctypes.byref(tc_), ta, tb))
        kern = L.last_kernel()
        got = _from_dev(pc, csh, odt)
    finally:
        for p in (pa, pb, pc):
            L.free(p)
    A = np.swapaxes(a64, -1, -2) if ta else a64
    B = np.swapaxes(b64, -1, -2) if tb else b64
    want = A @ B
    bound = 1e-4 * (np.abs(A) @ np.abs(B))
    if odt == "bfloat16":
        bound = bound + np.abs(want) * 2.0 ** -7
    elif odt == "float16":
        bound = bound + np.abs(want) * 2.0 ** -10
    elif dt == "float64":
        bound = 1e-12 * (np.abs(A) @ np.abs(B))
    bad = np.abs(got - want) > bound
    assert not bad.any(), (kern, dt, odt, M, K, N, ta, tb, int(bad.sum()), float(np.abs(got - want).max()))
    return kern


SHAPES = [(256, 256, 256), (304, 200, 136), (64, 64, 64), (1000, 72, 520), (40, 24, 48), (520, 264, 328), (8, 520, 8)]


@pytest.mark.parametrize("dt", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_mfma_layouts_and_edges(gpu, dt, ta, tb):
    """Row lengths that are multiples of 16 bytes take the MFMA kernel: all four layouts, tiles that hang over
    every edge, a k that ends inside a stage and inside a 16-byte chunk."""
    lib = L.load()
    for i, (M, K, N) in enumerate(SHAPES):
        kern = _run(lib, dt, dt, M, K, N, ta, tb, seed=i)
        assert kern.startswith("mjt_gemm_mfma_"), kern
    if dt != "float32":                                   # the float32 sum of 16-bit operands, before it is narrowed
        assert _run(lib, dt, "float32", 304, 200, 136, ta, tb).startswith("mjt_gemm_mfma_")


@pytest.mark.parametrize("tile", ["256", "128"])
@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
def test_gemm_direct_copy_kernel(gpu, dt, ta, tb, tile, monkeypatch):
    """16-bit operands with K a multiple of 64 have a kernel of their own (operands go from memory to LDS without
    passing through registers; an operand whose memory has m or n innermost is read from LDS with transposing
    reads) once there are enough 256 x 256 tiles (two stage buffers) or 128 x 128 tiles (a ring of four); here it is
    asked for by name and tile so that small shapes reach it too: all four layouts, tiles that hang over both edges, fewer
    stages than buffers (K = 64, 128, 192), many stages, a float32 result, a batch."""
    lib = L.load()
    monkeypatch.setenv("MJT_GEMM_DMA", tile)
    for i, (M, K, N) in enumerate([(256, 64, 256), (512, 256, 256), (304, 128, 136), (1000, 192, 520), (8, 512, 8), (520, 2048, 264)]):
        kern = _run(lib, dt, dt, M, K, N, ta, tb, seed=20 + i)
        assert kern.endswith("%sx%s_%s%s_direct" % (tile, tile, "nt"[ta], "nt"[tb])), kern
    assert _run(lib, dt, "float32", 304, 128, 520, ta, tb, seed=30).endswith("_direct")
    assert _run(lib, dt, dt, 264, 64, 248, ta, tb, seed=31, batch=(3,)).endswith("_direct")
    # K = 96 is no multiple of 64: the general kernel
    assert not _run(lib, dt, dt, 256, 96, 256, ta, tb, seed=32).endswith("_direct")


@pytest.mark.parametrize("tile", ["256", "128"])
def test_gemm_direct_copy_kernel_random_shapes(gpu, tile, monkeypatch):
    """Seeded sweep over shapes, layouts, result types and batches for the direct-copy kernel: M and N anywhere
    between 1 and 700 (tiles cut on every side, operands whose last rows or columns end at the tensor's end),
    K a multiple of 64 up to 1024."""
    lib = L.load()
    monkeypatch.setenv("MJT_GEMM_DMA", tile)
    rng = np.random.default_rng(2024)
    for i in range(24):
        M, N = int(rng.integers(1, 88)) * 8, int(rng.integers(1, 88)) * 8       # rows of 16-byte multiples in every layout
        K = 64 * int(rng.integers(1, 17))
        ta, tb = int(rng.integers(0, 2)), int(rng.integers(0, 2))
        dt = ("bfloat16", "float16")[i % 2]
        odt = (dt, "float32")[int(rng.integers(0, 2))]
        batch = () if i % 3 else (int(rng.integers(2, 4)),)
        kern = _run(lib, dt, odt, M, K, N, ta, tb, seed=100 + i, batch=batch)
        assert kern.endswith("_direct"), (kern, M, K, N, ta, tb)


def test_gemm_k_tail_inside_a_chunk(gpu):
    """k-innermost operands whose K is no multiple of the chunk: the row length (leading dimension) is what has to
    be aligned, and a product's operands are dense, so this route is only reachable with a K that is aligned;
    K = 72 ends inside a 64-wide stage for 16-bit operands, K = 36 inside one for float32."""
    lib = L.load()
    assert _run(lib, "bfloat16", "bfloat16", 128, 72, 128, 0, 1).startswith("mjt_gemm_mfma_")
    assert _run(lib, "float32", "float32", 128, 36, 128, 0, 1).startswith("mjt_gemm_mfma_")
    assert _run(lib, "float16", "float32", 96, 8, 64, 0, 1).startswith("mjt_gemm_mfma_")


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_single_stage_uses_one_staging_buffer(gpu, ta, tb, monkeypatch):
    """A sum that fits one stage of the k loop (64 elements of 16 bits, 32 of float32) runs on a variant of the kernel
    with one staging buffer; one element more and it is the two-buffer kernel again.  Tiles over every edge, a batch."""
    lib = L.load()
    for dt, K in (("bfloat16", 64), ("float16", 40), ("float32", 32), ("float32", 8)):
        assert _run(lib, dt, dt, 304, K, 264, ta, tb, seed=K).endswith("_k1")
        assert _run(lib, dt, "float32", 72, K, 520, ta, tb, seed=K + 1, batch=(3,)).endswith("_k1")
    assert not _run(lib, "bfloat16", "bfloat16", 304, 72, 264, ta, tb, seed=3).endswith("_k1")
    assert not _run(lib, "float32", "float32", 304, 36, 264, ta, tb, seed=4).endswith("_k1")
    monkeypatch.setenv("MJT_GEMM_TWO_BUFFERS", "1")
    assert not _run(lib, "bfloat16", "bfloat16", 304, 64, 264, ta, tb, seed=64).endswith("_k1")


@pytest.mark.parametrize("dt", ["bfloat16", "float32", "float64"])
def test_gemm_plain_unaligned_and_float64(gpu, dt):
    lib = L.load()
    for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
        kern = _run(lib, dt, dt, 70, 129, 45, ta, tb)
        assert kern.startswith("mjt_gemm_plain_"), kern
    assert _run(lib, dt, dt, 1, 1, 1, 0, 0).startswith("mjt_gemm_plain_")
    assert _run(lib, dt, dt, 130, 3, 67, 0, 1).startswith("mjt_gemm_plain_")


def test_gemm_batched(gpu):
    lib = L.load()
    assert _run(lib, "bfloat16", "bfloat16", 136, 64, 200, 0, 0, batch=(3, 2)).startswith("mjt_gemm_mfma_")
    assert _run(lib, "float32", "float32", 100, 36, 52, 1, 0, batch=(5,)).startswith("mjt_gemm_mfma_")
    assert _run(lib, "float32", "float32", 33, 17, 9, 0, 0, batch=(4,)).startswith("mjt_gemm_plain_")


def test_gemm_is_the_meta_op_expression(gpu):
    """The product equals the expression the reference's tuner matches: broadcast(a,[n,m,k]) * broadcast(b,[n,m,k])
    summed over m, evaluated by the oracle's meta-ops in float32 (python/jittor/nn.py:118-158)."""
    lib = L.load()
    rng = np.random.default_rng(3)
    a = rng.standard_normal((24, 40)).astype(np.float32)
    b = rng.standard_normal((40, 16)).astype(np.float32)
    prod = O.binary(O.broadcast_to(a, [24, 40, 16], [2]), O.broadcast_to(b, [24, 40, 16], [0]), "multiply")
    want = O.reduce(prod, "add", 1)
    pa, pb, pc = _to_dev(a), _to_dev(b), L.alloc(24 * 16 * 4)
    try:
        ta_, tb_, tc_ = L.tensor(pa, "float32", a.shape), L.tensor(pb, "float32", b.shape), L.tensor(pc, "float32", (24, 16))
        L.check(lib.mjt_matmul(ctypes.byref(ta_), ctypes.byref(tb_), ctypes.byref(tc_), 0, 0))
        got = L.d2h(pc, (24, 16), np.float32)
    finally:
        for p in (pa, pb, pc):
            L.free(p)
    assert np.allclose(got, want, rtol=1e-5, atol=1e-5 * np.abs(want).max())


def test_gemm_2048_runs_on_128_tiles_of_the_direct_copy_kernel(gpu):
    """2048^3 has 64 tiles of 256 x 256 for 256 compute units: the direct-copy kernel takes it on 128 x 128 tiles (a ring
    of four stages), in every layout; 1536^3 (144 such tiles) too; the whole result against float64."""
    lib = L.load()
    for ta, tb in ((0, 1), (0, 0), (1, 0), (1, 1)):
        kern = _run(lib, "bfloat16", "bfloat16", 2048, 2048, 2048, ta, tb, seed=40 + 2 * ta + tb)
        assert kern.endswith("128x128_%s%s_direct" % ("nt"[ta], "nt"[tb])), kern
    assert _run(lib, "float16", "float32", 1536, 1536, 1536, 0, 1, seed=44).endswith("128x128_nt_direct")


def test_gemm_more_128_tiles_than_compute_units_run_two_workgroups_per_unit(gpu):
    """With more 128 x 128 tiles than compute units (and too few 256 x 256 ones, or a sum too short for those) the
    direct-copy kernel runs on two stage buffers, two workgroups per compute unit: every layout, one to five stages of
    the sum, tiles hanging over both edges, a batch; the whole result against float64."""
    lib = L.load()
    for i, (ta, tb) in enumerate(((0, 1), (0, 0), (1, 0), (1, 1))):
        kern = _run(lib, "bfloat16", "bfloat16", 2176, 128, 2120, ta, tb, seed=50 + i)
        assert kern.endswith("128x128_%s%s_direct2" % ("nt"[ta], "nt"[tb])), kern
    assert _run(lib, "float16", "float16", 2304, 320, 2200, 0, 1, seed=54).endswith("128x128_nt_direct2")
    assert _run(lib, "bfloat16", "float32", 2304, 64, 2304, 1, 0, seed=55).endswith("128x128_tn_direct2")
    assert _run(lib, "bfloat16", "bfloat16", 640, 192, 904, 0, 0, seed=56, batch=(9,)).endswith("128x128_nn_direct2")


def test_gemm_full_size_4096_bf16_properties(gpu):
    """4096^3 in bfloat16 (the shape the throughput figure is quoted on): rows of the result against float64 on a
    sample, and linearity in b, which holds exactly for power-of-two factors."""
    lib = L.load()
    n = 4096
    rng = np.random.default_rng(9)
    a_bits = f32_to_bf16_bits(rng.standard_normal((n, n)).astype(np.float32))
    b_bits = f32_to_bf16_bits(rng.standard_normal((n, n)).astype(np.float32))
    pa, pb, pc = _to_dev(a_bits), _to_dev(b_bits), L.alloc(n * n * 4)
    try:
        ta_, tb_, tc_ = L.tensor(pa, "bfloat16", (n, n)), L.tensor(pb, "bfloat16", (n, n)), L.tensor(pc, "float32", (n, n))
        for trans_b in (1, 0):
            L.check(lib.mjt_matmul(ctypes.byref(ta_), ctypes.byref(tb_), ctypes.byref(tc_), 0, trans_b))
            assert L.last_kernel().startswith("mjt_gemm_mfma_bfloat16_float32_256x256"), L.last_kernel()
            got = L.d2h(pc, (n, n), np.float32)
            A = (a_bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
            B = (b_bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
            Bm = B.T if trans_b else B
            for r in (0, 1, 255, 256, 2049, 4095):
                want = A[r] @ Bm
                bound = 1e-4 * (np.abs(A[r]) @ np.abs(Bm))
                assert (np.abs(got[r] - want) <= bound).all(), (trans_b, r)
        L.h2d(pb, (b_bits.astype(np.uint32) + (2 << 7)).astype(np.uint16))     # exponent + 2: b * 4, exactly
        L.check(lib.mjt_matmul(ctypes.byref(ta_), ctypes.byref(tb_), ctypes.byref(tc_), 0, 0))
        assert np.array_equal(L.d2h(pc, (n, n), np.float32), got * 4)
    finally:
        for p in (pa, pb, pc):
            L.free(p)


@pytest.mark.parametrize("dt", ["bfloat16", "float32"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_stage_pipeline_lengths(gpu, dt, ta, tb):
    """Sums of one stage up to several (64 elements of 16 bits, 32 of float32), whole and with a remainder: fewer stages than are
    in flight, the last whole ones, a last one that ends inside a chunk; tiles of 64 and more, over both edges."""
    lib = L.load()
    ks = 32 if dt == "float32" else 64
    for stages in range(1, 9):
        for rest in (0, 8):
            _run(lib, dt, "float32", 72, ks * stages + rest, 136, ta, tb, seed=stages)
    _run(lib, dt, dt, 1032, 7 * ks + 8, 1160, ta, tb, seed=9)
    _run(lib, dt, dt, 72, 3 * ks + 8, 72, ta, tb, seed=10, batch=(5,))


@pytest.mark.parametrize("dt", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_slices_of_a_long_sum(gpu, dt, ta, tb):
    """Few tiles and a long sum: slices of the sum, added up by a reduce; the last slice shorter and ending inside a stage."""
    lib = L.load()
    for M, K, N in ((64, 4104, 72), (8, 2000, 520), (264, 8200, 200)):
        assert _run(lib, dt, dt, M, K, N, ta, tb, seed=K).endswith("_slices")
        assert _run(lib, dt, "float32", M, K, N, ta, tb, seed=K + 1).endswith("_slices")


@pytest.mark.parametrize("dt", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_unaligned_rows_are_copied(gpu, dt, ta, tb):
    """Rows that are no 16-byte multiples, from a few million multiply-adds on: one operand copied, both, batches."""
    lib = L.load()
    for i, (M, K, N) in enumerate([(301, 203, 129), (304, 201, 136), (129, 336, 201), (1001, 1001, 67), (257, 4099, 65)]):
        assert _run(lib, dt, dt, M, K, N, ta, tb, seed=i).startswith("mjt_gemm_mfma_"), (M, K, N)
    assert _run(lib, dt, dt, 61, 203, 129, ta, tb, seed=7, batch=(5,)).startswith("mjt_gemm_mfma_")


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,K,N", [(1001, 128, 1024), (1001, 1024, 1024), (1151, 192, 1016)])
def test_gemm_odd_rows_of_a_transposed_operand(gpu, dt, tb, M, K, N):
    """a^T b with an odd number of result rows on the kernel that copies its operands into LDS: the last element of a, half of the
    last dword in range, belongs to the last row's sum."""
    assert "_direct" in _run(L.load(), dt, "float32", M, K, N, 1, tb, seed=M + K)


@pytest.mark.parametrize("dt", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("batch,M,N,K", [(1, 40, 40, 64), (3, 64, 128, 96), (8, 65, 64, 64), (17, 200, 70, 128), (21, 130, 257, 192), (9, 640, 640, 64), (300, 24, 40, 72)])
@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0)])
def test_gemm_batches_of_few_tiles(gpu, dt, batch, M, N, K, ta, tb):
    """The tiles of a batch's matrices begin one XCD further on with each: every tile of every matrix is made, with less than eight
    tiles a matrix, with eight and with more, on the general kernel and on the one that copies its operands into LDS."""
    M, N = (M, N) if dt == "float32" else ((M + 7) // 8 * 8, (N + 7) // 8 * 8)
    _run(L.load(), dt, dt, M, K, N, ta, tb, batch=(batch,), seed=M + K)
    if dt != "float32" and K % 64 == 0:
        with pytest.MonkeyPatch.context() as m:
            m.setenv("MJT_GEMM_DMA", "128")
            assert "_direct" in _run(L.load(), dt, dt, M, K, N, ta, tb, batch=(batch,), seed=M + K)


# ---- float32 products of bfloat16 parts: a value is h + m + l, six of nine products are summed, an MFMA rounds once per 16 of them ----
def _parts_bound(A, B, K):
    """Two sums of K / 16 MFMAs of up to three products each and one addition, every rounding at most 2^-23 (the MFMA may truncate) of
    the sum of magnitudes; what is left out of a product is below 2^-25 of it."""
    with np.errstate(all="ignore"):
        return (K / 16 * 4 + 8) * 2.0 ** -23 * (np.abs(A) @ np.abs(B))


def _parts_product(lib, A, B, ta, tb, batch=()):
    pa, pb = _to_dev(A), _to_dev(B)
    M, K = A.shape[-1 if ta else -2], A.shape[-2 if ta else -1]
    N = B.shape[-2 if tb else -1]
    pc = L.alloc(int(np.prod(batch, dtype=np.int64)) * M * N * 4)
    try:
        t = [L.tensor(pa, "float32", A.shape), L.tensor(pb, "float32", B.shape), L.tensor(pc, "float32", tuple(batch) + (M, N))]
        L.check(lib.mjt_matmul(*[ctypes.byref(q) for q in t], ta, tb))
        return L.d2h(pc, tuple(batch) + (M, N), np.float32).astype(np.float64), L.last_kernel()
    finally:
        for p in (pa, pb, pc):
            L.free(p)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,K,N,batch,tile", [(2044, 1020, 1000, (), "128x64"), (1916, 260, 2100, (), "128x128"), (1020, 2052, 1012, (), "slices"),
                                              (384, 380, 364, (12,), "parts"), (100, 2500, 4100, (), "parts")])
def test_gemm_float32_parts(gpu, M, K, N, batch, tile, ta, tb):
    """Tiles that hang over both edges, a sum that ends inside a stage and inside a chunk, slices, a batch; operands over nine decades with
    zeros among them."""
    rng = np.random.default_rng(M + K)
    scale = lambda shape: 10.0 ** rng.integers(-4, 5, shape) * (rng.random(shape) > 0.1)
    A = (rng.standard_normal(batch + ((K, M) if ta else (M, K)))).astype(np.float32)
    B = (rng.standard_normal(batch + ((N, K) if tb else (K, N)))).astype(np.float32)
    A = (A * scale(A.shape)).astype(np.float32)
    got, kern = _parts_product(L.load(), A, B, ta, tb, batch)
    assert "_parts" in kern and (tile in kern), kern
    a64 = np.swapaxes(A, -1, -2).astype(np.float64) if ta else A.astype(np.float64)
    b64 = np.swapaxes(B, -1, -2).astype(np.float64) if tb else B.astype(np.float64)
    assert (np.abs(got - a64 @ b64) <= _parts_bound(a64, b64, K)).all(), kern


@pytest.mark.parametrize("what", ["inf", "nan", "rounds to inf", "denormal", "tiny", "small products", "overflow", "zeros"])
def test_gemm_float32_parts_hand_over(gpu, what):
    """Operands at the ends of float32's range and sums that are not finite, 2^48 times as large as they come: the tiles of the latter run
    on the float32 MFMAs, results are what float32 gives; the other tiles stay."""
    rng = np.random.default_rng(5)
    M, K, N = 2048, 1024, 1024
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    if what == "inf":
        A[5, 7], A[700, 1000], B[1000, 3] = np.inf, -np.inf, np.inf
    elif what == "nan":
        A[1500, 1023], B[64, 0] = np.nan, np.nan
    elif what == "rounds to inf":                                      # finite, but the first part is not
        A[9, 11], A[1400, 900] = 3.4e38, -3.4028e38
        B *= 1e-3
    elif what == "denormal":
        A[130], A[1999, ::2] = 1e-40, 1.1e-39
        B[:, :] *= np.float32(1e25)
    elif what == "tiny":                                               # the second and third parts of the value itself are below the normal range
        A *= np.float32(1e-35)
        B *= np.float32(1e33)
    elif what == "small products":
        A *= np.float32(1e-17)
        B *= np.float32(1e-19)
    elif what == "overflow":
        A[77] *= np.float32(1e30)
        B[900] *= np.float32(1e12)
    else:
        A[:200], B[:, 100:300] = 0.0, 0.0
    got, kern = _parts_product(L.load(), A, B, 0, 1)
    assert "_parts" in kern, kern
    a, b = A.astype(np.float64), B.astype(np.float64).T
    with np.errstate(all="ignore"):
        want, bound = a @ b, _parts_bound(a, b, K)
        f32 = want.astype(np.float32)
    if what == "overflow":                                             # partial sums may pass the largest float before the total does
        sure = (np.abs(a) @ np.abs(b) < 3e38) | (np.abs(want) > 1e39)
        assert np.array_equal(np.isfinite(got)[sure], np.isfinite(f32)[sure]) and (~np.isfinite(f32)).any()
    else:
        assert np.array_equal(np.isnan(got), np.isnan(f32))
        assert np.array_equal(got[np.isinf(f32)], f32[np.isinf(f32)].astype(np.float64))
    ok = np.isfinite(f32) & np.isfinite(got)
    # (a sum below the normal range may be taken for zero)
    assert (np.abs(got[ok] - want[ok]) <= bound[ok] + K * 2.0 ** -126).all(), np.abs(got[ok] - want[ok]).max()


@pytest.mark.parametrize("what", ["inf", "nan", "rounds to inf"])
def test_gemm_float32_parts_of_a_single_stage(gpu, what):
    """43 stages in slices of 6: the last slice is one stage, whose workgroups have no barrier between their first operands and their sums.
    Sums that are not finite there, in every other tile, run on the float32 MFMAs."""
    rng = np.random.default_rng(6)
    M, K, N = 512, 1376, 512
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    A[3::256, 1350 + (what == "nan")] = {"inf": np.inf, "nan": np.nan, "rounds to inf": 3.4e38}[what]
    if what == "rounds to inf":
        B *= np.float32(1e-3)
    for _ in range(3):
        got, kern = _parts_product(L.load(), A, B, 0, 1)
        assert "_parts_slices" in kern and "128x64" in kern, kern
        a, b = A.astype(np.float64), B.astype(np.float64).T
        with np.errstate(all="ignore"):
            want, bound = a @ b, _parts_bound(a, b, K)
        ok = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), ok) and np.array_equal(np.isnan(got), np.isnan(want))
        assert (np.abs(got[ok] - want[ok]) <= bound[ok]).all()


def _scaled_runs(call, inputs, out_shape):
    """Results of call(*tensors, out) with the first input times 2^-105, 1 and 2^40, taken back, with the kernel's name."""
    po, got = L.alloc(int(np.prod(out_shape)) * 4), []
    try:
        for e in (-105, 0, 40):
            ps = [_to_dev(inputs[0] * np.float32(2.0 ** e))] + [_to_dev(a) for a in inputs[1:]]
            try:
                call(*[L.tensor(q, "float32", a.shape) for q, a in zip(ps, inputs)], L.tensor(po, "float32", out_shape))
                got.append((L.d2h(po, out_shape, np.float32) * np.float32(2.0 ** -e), L.last_kernel()))
            finally:
                for q in ps:
                    L.free(q)
    finally:
        L.free(po)
    return got


@pytest.mark.parametrize("what", ["128x64", "128x128", "slices", "conv", "conv wgrad", "stem", "stem wgrad"])
def test_float32_parts_take_powers_of_two_out(gpu, what):
    """Operands of any size run on their parts and no bit depends on their common power of two.  (The float32 MFMAs, to which tiles with values
    below 2^-100 went, round more often.)"""
    lib, rng, ref = L.load(), np.random.default_rng(9), ctypes.byref
    draw = lambda *s: rng.standard_normal(s).astype(np.float32)
    if what in ("128x64", "128x128", "slices"):
        M, K, N = {"128x64": (2048, 1024, 1024), "128x128": (1916, 256, 2100), "slices": (512, 1376, 512)}[what]
        got = _scaled_runs(lambda a, b, c: L.check(lib.mjt_matmul(ref(a), ref(b), ref(c), 0, 1)), [draw(M, K), draw(N, K)], (M, N))
    else:
        xs, k, R, p, o = ((2, 3, 224, 224), 32, 7, L.ConvParams(2, 2, 3, 3, 1, 1), 112) if "stem" in what else ((32, 64, 56, 56), 128, 3, L.ConvParams(2, 2, 1, 1, 1, 1), 28)
        if what == "stem wgrad":
            xs = (8,) + xs[1:]
        x, w, dy = draw(*xs), draw(k, xs[1], R, R), draw(xs[0], k, o, o)
        if "wgrad" in what:
            got = _scaled_runs(lambda a, b, c: L.check(lib.mjt_conv2d_meta_wgrad(ref(a), ref(b), ref(c), ref(p))), [x, dy], w.shape)
        else:
            got = _scaled_runs(lambda a, b, c: L.check(lib.mjt_conv2d_meta(ref(a), ref(b), ref(c), ref(p))), [x, w], dy.shape)
    for g, kern in got:
        assert ("_stem_" if "stem" in what else what if "128" in what else "_parts") in kern, kern
        assert np.array_equal(g, got[1][0]), (what, np.abs(g - got[1][0]).max())


def _columns(x, R, stride, pad):
    n, c, h, w = x.shape
    xp = np.pad(x, ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    v = np.lib.stride_tricks.sliding_window_view(xp, (R, R), axis=(2, 3))[:, :, ::stride, ::stride]       # n c oh ow r s
    return np.ascontiguousarray(v.transpose(0, 2, 3, 1, 4, 5)).reshape(n * v.shape[2] * v.shape[3], c * R * R), v.shape[2]


@pytest.mark.parametrize("xs,k,R,stride,tiny", [((16, 40, 27, 27), 200, 3, 1, False), ((16, 39, 27, 27), 100, 3, 1, False), ((32, 64, 56, 56), 128, 3, 2, False),
                                                ((16, 40, 27, 27), 200, 3, 1, True), ((32, 64, 56, 56), 128, 3, 2, True)])
def test_conv_float32_parts(gpu, xs, k, R, stride, tiny):
    """The gathering forward and weight-gradient products on bfloat16 parts; with tiny values and an infinity among the operands too."""
    lib = L.load()
    rng = np.random.default_rng(k)
    x, w = rng.standard_normal(xs).astype(np.float32), rng.standard_normal((k, xs[1], R, R)).astype(np.float32)
    if tiny:
        x[3, 5] *= np.float32(1e-34)
        x[4, 6, 2, 2] = np.inf
    cols, o = _columns(x.astype(np.float64), R, stride, R // 2)
    dy = rng.standard_normal((xs[0], k, o, o)).astype(np.float32)
    px, pw, pdy, py, pdw = _to_dev(x), _to_dev(w), _to_dev(dy), L.alloc(dy.nbytes), L.alloc(w.nbytes)
    try:
        tx, tw, tdy, ty, tdw = L.tensor(px, "float32", xs), L.tensor(pw, "float32", w.shape), L.tensor(pdy, "float32", dy.shape), L.tensor(py, "float32", dy.shape), L.tensor(pdw, "float32", w.shape)
        p = L.ConvParams(stride, stride, R // 2, R // 2, 1, 1)
        L.check(lib.mjt_conv2d_meta(ctypes.byref(tx), ctypes.byref(tw), ctypes.byref(ty), ctypes.byref(p)))
        assert L.last_kernel().startswith("mjt_conv_igemm_float32") and "_parts_" in L.last_kernel(), L.last_kernel()
        y = L.d2h(py, dy.shape, np.float32).astype(np.float64).transpose(0, 2, 3, 1).reshape(-1, k)
        L.check(lib.mjt_conv2d_meta_wgrad_grouped(ctypes.byref(tx), ctypes.byref(tdy), ctypes.byref(tdw), ctypes.byref(p), 1))
        split = "_parts_" in L.last_kernel()
        dw = L.d2h(pdw, w.shape, np.float32).astype(np.float64).reshape(k, -1)
    finally:
        for q in (px, pw, pdy, py, pdw):
            L.free(q)
    assert split or stride == 1
    w2, d2 = w.astype(np.float64).reshape(k, -1), dy.astype(np.float64).transpose(0, 2, 3, 1).reshape(-1, k).T
    with np.errstate(all="ignore"):
        for got, a, b in ((y, cols, w2.T), (dw, d2, cols)):
            want, bound = a @ b, _parts_bound(a, b, a.shape[1])
            assert np.array_equal(np.isfinite(got), np.isfinite(want))
            ok = np.isfinite(want)
            assert (np.abs(got[ok] - want[ok]) <= bound[ok]).all()
