"""Each HIP kernel alone against its plain reference (tests/torch_backend.py), at sizes
other than the engine's tiny models: widths and vocabularies that are no power of two,
head sizes in steps of 16, odd head counts and groups, scattered pages.

Vectors taken from the reference's own kernel tests (tests/test_kernels.py:14-59 there):
RMSNorm rows {1, 7, 256, 2048} x widths {2048, 4096, 896} at eps 1e-5 with the bfloat16
tolerance atol 2e-2 / rtol 1e-2; decode attention at 32 query heads on 4 kv heads of 64,
page 16, context lengths [1], [17], [1000], [2048], [5, 300, 1, 2047, 64, 65] and
range(1, 200, 7), pages scattered by a random permutation, tolerance 2e-2.
"""
import math
from types import SimpleNamespace

import pytest
import torch

import torch_backend as ref
from native_calls import counted

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from mini_inference_engine_amd.kernels.hip_backend import HipBackend
    return {torch.float32: HipBackend(torch.float32, DEV), torch.bfloat16: HipBackend(torch.bfloat16, DEV)}


def tol(dtype):
    return dict(atol=2e-2, rtol=1e-2) if dtype == torch.bfloat16 else dict(atol=2e-6, rtol=1e-5)


# ------------------------------------------------------------------ embedding
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding(ops, dtype):
    torch.manual_seed(0)
    table = torch.randn(331, 120, device=DEV).to(dtype)
    ids = torch.randint(0, 331, (77,), device=DEV, dtype=torch.int32)
    out = ops[dtype].embedding(ids, table)
    assert out.dtype == torch.float32
    assert torch.equal(out, ref.ref_embedding(ids, table))


# -------------------------------------------------------------------- rmsnorm
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [2048, 4096, 896, 120, 5000])
@pytest.mark.parametrize("rows", [1, 7, 256, 2048])
def test_add_rmsnorm(ops, dtype, rows, width):
    if rows == 2048 and width == 5000:
        rows = 300
    torch.manual_seed(rows * 7 + width)
    x = torch.randn(rows, width, device=DEV).to(dtype)
    stream = torch.randn(rows, width, device=DEV)
    w = torch.randn(width, device=DEV).to(dtype)
    s_ref = stream.clone()
    y_ref = ref.ref_add_rmsnorm(x, s_ref, w, 1e-5, dtype)
    s = stream.clone()
    y = ops[dtype].add_rmsnorm(x, s, w, 1e-5)
    assert torch.equal(s, s_ref), "the updated stream must be bit-equal to stream + x"
    torch.testing.assert_close(y.float(), y_ref.float(), **tol(dtype))
    # nothing to add: the stream is left as it is
    s2 = stream.clone()
    y2 = ops[dtype].add_rmsnorm(None, s2, w, 1e-5)
    assert torch.equal(s2, stream)
    torch.testing.assert_close(y2.float(), ref.ref_add_rmsnorm(None, stream.clone(), w, 1e-5, dtype).float(), **tol(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_add_rmsnorm_rows_and_weight_dtype(ops, dtype):
    torch.manual_seed(3)
    x = torch.randn(50, 4700, device=DEV).to(dtype)
    stream = torch.randn(50, 4700, device=DEV)
    w32 = torch.randn(4700, device=DEV)            # a weight stored in 32-bit stays so
    rows = torch.tensor([49, 0, 7, 7, 13], device=DEV, dtype=torch.int32)
    before = stream.clone()
    y = ops[dtype].add_rmsnorm(x, stream, w32, 1e-6, out_dtype=dtype, rows=rows)
    assert torch.equal(stream, before), "gathered rows must not touch the stream"
    y_ref = ref.ref_add_rmsnorm(x, before.clone(), w32, 1e-6, dtype, rows)
    torch.testing.assert_close(y.float(), y_ref.float(), **tol(dtype))


def test_rmsnorm_against_library(ops):
    """float32: equals torch's rms_norm; a wrong eps placement or a mean over the wrong size fails it."""
    torch.manual_seed(4)
    x = torch.randn(9, 300, device=DEV) * 1e-3      # small values: eps matters
    w = torch.randn(300, device=DEV)
    y = ops[torch.float32].add_rmsnorm(None, x.clone(), w, 1e-5)
    torch.testing.assert_close(y, torch.nn.functional.rms_norm(x, (300,), w, 1e-5), atol=1e-6, rtol=1e-5)


# ----------------------------------------------------------------------- gemm
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 64, 176), (7, 200, 331), (130, 96, 120), (65, 1030, 77), (300, 512, 640)])
def test_linear(ops, dtype, shape):
    M, K, N = shape
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=DEV).to(dtype)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(dtype)
    y = ops[dtype].linear(x, w)
    torch.testing.assert_close(y.float(), ref.ref_linear(x, w, None, dtype).float(), **tol(dtype))
    y32 = ops[dtype].linear(x, w, out_dtype=torch.float32)
    assert y32.dtype == torch.float32
    torch.testing.assert_close(y32, ref.ref_linear(x, w, None, torch.float32), **tol(dtype))


def test_linear_float32_is_batch_invariant(ops):
    torch.manual_seed(1)
    x = torch.randn(200, 333, device=DEV)
    w = torch.randn(150, 333, device=DEV)
    whole = ops[torch.float32].linear(x, w)
    for a, b in ((0, 1), (63, 130), (199, 200), (17, 19)):
        assert torch.equal(ops[torch.float32].linear(x[a:b].contiguous(), w), whole[a:b])

# (rows, K, N): few rows and many, K with quarters and eighths missing (4, 64, 176: steps of 32, then quarters, then eighths), a step
# cut short, tile edges
F32_SHAPES = [(1, 2048, 2048), (16, 176, 64), (5, 4, 36), (17, 64, 132), (64, 1040, 260), (65, 528, 4100), (128, 2048, 96),
              (300, 332, 640), (513, 256, 8196)]


@pytest.mark.parametrize("shape", F32_SHAPES)
def test_linear_float32_matrix_unit(ops, shape):
    """The float32 products on the matrix unit: against 64 bits within K / 16 + 32 half ulps of the sum of magnitudes (half the worst
    case of an eighth's chain of K / 8 products; the joins, the small products' chain and the products left out, 2^-24 together), a row the
    same bits in any cut (few-row kernel, tiles, units of K), the added and the gated form the same bits as the product and a step of its own."""
    M, K, N = shape
    o = ops[torch.float32]
    torch.manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) / math.sqrt(K)
    with counted(o, "gemm_f32", "mie_gemm_f32") as calls:
        y = o.linear(x, w)
    assert len(calls) == 1
    bound = (K / 16 + 32) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30
    assert bool(((y.double() - x.double() @ w.double().T).abs() <= bound).all())
    for a, b in ((0, 1), (M // 2, M // 2 + 1), (max(0, M - 17), M), (0, min(M, 16)), (0, M // 2 + 1)):
        assert torch.equal(o.linear(x[a:b].contiguous(), w), y[a:b])
    big = torch.cat([x, torch.randn(700, K, device=DEV)])
    assert torch.equal(o.linear(big, w)[:M], y)
    stream = torch.randn(M, N, device=DEV)
    expect = stream + y
    assert o.linear(x, w, add_to=stream) is None
    assert torch.equal(stream, expect)
    inter = N // 2
    if inter % 4 == 0:
        assert torch.equal(o.linear_silu_mul(x, w, inter), o.silu_mul(y, inter))
    bias = torch.randn(N, device=DEV)
    assert torch.equal(o.linear(x, w, bias=bias), y + bias)


# rows that take the few-row kernel (two steps at once, one), the tiles in eighths, whole and in quarters; K with an odd number of
# steps for a wave, without any for most, and a step cut short
F32_PARTS = [(3, 2080, 48), (12, 2080, 48), (40, 1056, 64), (20, 36, 352), (300, 2048, 2048), (1100, 96, 2304), (600, 352, 9000)]


@pytest.mark.parametrize("shape", F32_PARTS)
def test_linear_float32_in_three_parts(ops, shape):
    """The float32 product as six bfloat16 ones: its error in the 2-norm is below that of chains of 32-bit products (a quarter of
    the worst case, sqrt(terms) half ulps); numbers that bfloat16 cannot hold give the infinities, NaN and finite results that 32-bit
    arithmetic gives them, and change no bit of another row or column."""
    M, K, N = shape
    o = ops[torch.float32]
    torch.manual_seed(K + N)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) / math.sqrt(K)
    y, exact = o.linear(x, w), x.double() @ w.double().T
    assert (y.double() - exact).norm() <= 2.0 ** -24 * math.sqrt(K / 16 + 8) * exact.norm()
    for at, value in ((0, float("inf")), (K // 2, float("-inf")), (K - 1, float("nan")), (min(35, K - 1), 3.4e38)):
        x2, w2 = x.clone(), w.clone()
        x2[M // 2, at] = value
        w2[N - 3, K - 1 - at] = value
        w2[5, at] = 0.0 if at else 0.25              # an infinity times zero, and times a number bfloat16 holds whole
        if value == 3.4e38:
            w2[:, at] *= 2.0 ** -20                  # (finite results)
            x2[:, K - 1 - at] *= 2.0 ** -20
        got = o.linear(x2, w2)
        want = x2.double() @ w2.double().T
        large = want.abs() > 3.4028234663852886e38
        want[large] = torch.sign(want[large]) * float("inf")
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(torch.where(got.isinf(), got, 0.0), torch.where(want.isinf(), want, 0.0).float())
        finite = want.isfinite()
        bound = (K / 16 + 32) * 2.0 ** -24 * (x2.double().abs() @ w2.double().abs().T) + 1e-30
        assert bool(((got.double() - want).abs()[finite] <= bound[finite]).all())
        if value != 3.4e38:
            rows = torch.arange(M, device=DEV) != M // 2
            cols = (torch.arange(N, device=DEV) != N - 3) & (torch.arange(N, device=DEV) != 5)
            assert torch.equal(got[rows][:, cols], y[rows][:, cols])
            alone = o.linear(x2[M // 2:M // 2 + 1].contiguous(), w2)
            assert torch.equal(alone.nan_to_num(1e30), got[M // 2:M // 2 + 1].nan_to_num(1e30))


# (rows, K, N, parts of K that the product's plan takes): the few-row kernel (two steps at once, one), the tiles whole, in quarters
# and in eighths
F32_FORMS = [(3, 2080, 48, 0), (12, 2080, 48, 0), (600, 352, 9000, 1), (300, 2048, 2048, 4), (40, 1056, 64, 8)]


def f32_parts_of_k(o, M, K, N):
    return o.lib("gemm_f32").mie_f32_units(M, N, K, 0) if M > 16 else 0


@pytest.mark.parametrize("K", [28, 36, 60, 68, 124, 132, 252, 260, 508, 516, 1020, 1028])
def test_linear_float32_at_the_edges_of_the_cuts_of_k(ops, K):
    """A step more or less than fills K's quarters and eighths: the few-row kernel, the tiles in eighths, in quarters and
    whole give a row the same bits, as exact as K = 2,048 is asked to be."""
    o = ops[torch.float32]
    forms = [(3, 64), (12, 64), (40, 64), (300, 640), (700, 1100)]
    assert f32_parts_of_k(o, 2100, K, 4100) == 1
    assert f32_parts_of_k(o, 40, K, 64) == (1 if K < 128 else 8) and f32_parts_of_k(o, 300, K, 640) == (1 if K < 500 else 4)
    torch.manual_seed(K)
    x, w = torch.randn(2100, K, device=DEV), torch.randn(4100, K, device=DEV)
    exact = x.double() @ w.double().T
    whole = o.linear(x, w)
    assert (whole.double() - exact).norm() <= 2.0 ** -24 * math.sqrt(K / 16 + 8) * exact.norm()
    for M, N in forms:
        assert torch.equal(o.linear(x[:M].contiguous(), w[:N].contiguous()), whole[:M, :N]), (M, N)


@pytest.mark.parametrize("shape", F32_FORMS)
def test_linear_float32_just_below_the_largest_number(ops, shape):
    """Results of 3.396e38 whose operands round up where they are cut: their first parts' product is an infinity, the results are
    not, and they are the same bits in every cut, also where larger ones beside them are infinities."""
    M, K, N, parts = shape
    o = ops[torch.float32]
    assert f32_parts_of_k(o, M, K, N) == parts
    torch.manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    rows, cols = [0, M // 2, M - 1], [1, N // 2, N - 2]
    for i, (r, c) in enumerate(zip(rows, cols)):
        at = (i * K // 3 + 35) % K
        x[:, at], w[:, at] = 0.0, 0.0
        x[r, at], w[c, at] = 1.00395, 1.98829 * 2.0 ** 127 * (-1) ** i
        w[c + 1, at] = 1.995 * 2.0 ** 127                 # times x[r, at]: beyond the largest number
    y, want = o.linear(x, w), x.double() @ w.double().T
    large = want.abs() > 3.4028234663852886e38
    assert int(large.sum()) == 3 and float(want[~large].abs().max()) > 3.39e38
    assert torch.equal(y[large].double(), want[large].sign() * float("inf"))
    bound = (K / 16 + 32) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((y.double() - want).abs()[~large] <= bound[~large]).all())
    for a, b in ((0, 1), (0, min(M, 16)), (M // 2, M // 2 + 1), (M // 2, M)):
        assert torch.equal(o.linear(x[a:b].contiguous(), w), y[a:b])
    assert torch.equal(o.linear(torch.cat([x, torch.randn(700, K, device=DEV)]), w)[:M], y)
    silu = o.linear_silu_mul(x, w, N // 2)
    assert torch.equal(silu.nan_to_num(1e30), o.silu_mul(y, N // 2).nan_to_num(1e30))


@pytest.mark.parametrize("scales", [(60, -122), (-122, 60), (0, -110), (0, -118), (-118, 30), (-60, -60), (100, -140)])
@pytest.mark.parametrize("shape", F32_FORMS)
def test_linear_float32_of_tiny_operands(ops, shape, scales):
    """Operands of 2^scales: as exact as at ordinary sizes (the bound of test_linear_float32_in_three_parts), down to numbers below
    the smallest normal one (which hold the fewer bits that they hold; nothing more is lost), and the same bits in every cut."""
    M, K, N, parts = shape
    o = ops[torch.float32]
    assert f32_parts_of_k(o, M, K, N) == parts
    torch.manual_seed(K + N)
    x, w = ((torch.randn(n, K, device=DEV, dtype=torch.float64) * 2.0 ** e).float() for n, e in ((M, scales[0]), (N, scales[1])))
    y, exact = o.linear(x, w), x.double() @ w.double().T
    scale = 2.0 ** -sum(scales)          # (a norm of numbers of 2^-120 is not taken as they are)
    error, size = ((y.double() - exact) * scale).norm(), (exact * scale).norm()
    assert error <= 2.0 ** -24 * math.sqrt(K / 16 + 8) * size, (float(error / size))
    for a, b in ((0, 1), (0, min(M, 16)), (M // 2, M)):
        assert torch.equal(o.linear(x[a:b].contiguous(), w), y[a:b])


def test_linear_float32_in_parts_has_bounded_memory(ops):
    """The sums of K's parts take at most 128 MiB, at any size; what is not cut for that is computed whole with the same bits."""
    o = ops[torch.float32]
    cut = set()
    for M in (17, 100, 333, 512, 700, 1132, 1500, 2048, 4096, 8192):
        for N in (64, 2048, 5632, 11264, 28672, 57344, 128256):
            for K in (64, 2048, 5632, 14336, 28672):
                for gated in (0, 1):
                    parts = o.lib("gemm_f32").mie_f32_units(M, N, K, gated)
                    assert parts == 1 or parts * M * N * 4 <= 1 << 27, (M, N, K, gated, parts)
                    cut.add(parts)
    assert cut == {1, 4, 8}
    M, K, N = 1132, 4096, 8192
    assert f32_parts_of_k(o, M, K, N) == 1 and f32_parts_of_k(o, 700, K, N) == 4
    torch.manual_seed(0)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    y = o.linear(x, w)
    for a, b in ((0, 700), (1100, 1132), (700, 709)):
        assert torch.equal(o.linear(x[a:b].contiguous(), w), y[a:b])


def test_linear_mixed_storage(ops):
    """A matrix stored in 32-bit beside bfloat16 activations: computed, not refused."""
    torch.manual_seed(2)
    x = torch.randn(9, 120, device=DEV).to(torch.bfloat16)
    w = torch.randn(50, 120, device=DEV) / 11
    y = ops[torch.bfloat16].linear(x, w)
    assert y.dtype == torch.bfloat16
    torch.testing.assert_close(y.float(), ref.ref_linear(x, w, None, torch.bfloat16).float(), atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_silu_mul(ops, dtype):
    torch.manual_seed(5)
    inter = 176
    x = torch.randn(33, 64, device=DEV).to(dtype)
    w = (torch.randn(2 * inter, 64, device=DEV) / 8).to(dtype)
    y = ops[dtype].linear_silu_mul(x, w, inter)
    gu = ref.ref_linear(x, w, None, torch.float64)
    expect = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    torch.testing.assert_close(y.double(), expect, **tol(dtype))
    # gate first, then up: swapping the halves must change the result
    swapped = torch.nn.functional.silu(gu[:, inter:]) * gu[:, :inter]
    assert (y.double() - swapped).abs().max() > 10 * (y.double() - expect).abs().max()


# --------------------------------------------------- few-row fused products (bfloat16)
def normed(ops, stream, w_norm, eps, rows=None, pending=None):
    from mini_inference_engine_amd.kernels.api import Normed
    return Normed(ops, pending, stream, w_norm, eps, rows)


# (rows, K, N); K = 8 and 40: waves without a chunk of their own
SKINNY_SHAPES = [(1, 64, 176), (7, 200, 331), (16, 2048, 2560), (13, 120, 96), (11, 5632, 2048), (16, 2048, 640),
                 (8, 176, 64), (3, 96, 384), (5, 264, 9600), (9, 72, 12304), (16, 4104, 48), (2, 8, 32), (6, 40, 16)]


@pytest.mark.parametrize("shape", SKINNY_SHAPES)
def test_skinny_linear(ops, shape):
    M, K, N = shape
    o = ops[torch.bfloat16]
    torch.manual_seed(M * 3 + N)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    assert o._skinny_ok(x, w, None), "this shape must take the fused kernel"
    y = o.linear(x, w)
    torch.testing.assert_close(y.float(), ref.ref_linear(x, w, None, torch.bfloat16).float(), atol=2e-2, rtol=1e-2)
    y32 = o.linear(x, w, out_dtype=torch.float32)
    torch.testing.assert_close(y32, ref.ref_linear(x, w, None, torch.float32), atol=2e-3, rtol=2e-3)
    # a row's result does not depend on the rows beside it
    for a, b in ((0, 1), (M // 2, M), (M - 1, M)):
        assert torch.equal(o.linear(x[a:b].contiguous(), w, out_dtype=torch.float32), y32[a:b])
    # residual add in the epilogue
    stream = torch.randn(M, N, device=DEV)
    expect = stream + ref.ref_linear(x, w, None, torch.float32)
    assert o.linear(x, w, add_to=stream) is None
    torch.testing.assert_close(stream, expect, atol=2e-3, rtol=2e-3)


# rows, K, weight rows and the tiles a workgroup has: every number, a last workgroup with fewer and a last tile with fewer rows
@pytest.mark.parametrize("case", [(12, 136, 9605, 3), (16, 2048, 8200, 3), (9, 72, 12305, 2), (16, 72, 4813, 2), (8, 2120, 4813, 2), (3, 40, 65575, 2),
                                  (5, 264, 9605, 1), (16, 64, 4090, 1), (8, 1000, 12290, 1)])
def test_skinny_tiles_a_workgroup(ops, case):
    """Few-row products by one, two and three tiles a workgroup: plain, added, gated, with a norm in front and behind, and a row's bits by
    itself, where the tiles are others."""
    from mini_inference_engine_amd.kernels.api import Sink
    o, (M, K, N, tiles) = ops[torch.bfloat16], case
    I = (N + 1) // 2
    lib = o.lib("gemm_bf16")
    assert lib.mie_skinny_tiles(o.EPI_F32, M, N) == lib.mie_skinny_tiles(o.EPI_SWIGLU, M, I) == tiles, "the case must take the tiles it is for"
    torch.manual_seed(N)
    w, wg = ((torch.randn(n, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16) for n in (N, 2 * I))
    x, g = torch.randn(M, K, device=DEV).to(torch.bfloat16), 1 + 0.1 * torch.randn(K, device=DEV)
    y = o.linear(x, w, out_dtype=torch.float32)
    torch.testing.assert_close(y.double(), x.double() @ w.double().T, atol=1e-4, rtol=1e-4)
    assert torch.equal(o.linear(x[-1:].contiguous(), w, out_dtype=torch.float32), y[-1:])
    a = o.linear_silu_mul(x, wg, I)
    gu = x.double() @ wg.double().T
    torch.testing.assert_close(a.double(), torch.nn.functional.silu(gu[:, :I]) * gu[:, I:], atol=1e-3, rtol=1e-2)
    # added, with the norm behind it prepared
    stream, gn = torch.randn(M, N, device=DEV), 1 + 0.1 * torch.randn(N, device=DEV)
    want = stream.double() + y.double()
    behind = o.linear(x, w, add_to=Sink(stream, gn, 1e-5))
    torch.testing.assert_close(stream.double(), want, atol=1e-5, rtol=1e-5)
    squares = behind.ready["ss"][:, :behind.ready["tiles"]].double().sum(1)
    torch.testing.assert_close(squares, want.pow(2).sum(1), atol=0, rtol=1e-5)
    torch.testing.assert_close(behind.ready["x"].double(), want * gn.double(), atol=1e-2, rtol=2.0 ** -8)
    # a norm in front
    first = torch.randn(M, K, device=DEV)
    front = o.linear(x[:, :8].contiguous(), w[:K, :8].contiguous(), add_to=Sink(first, g, 1e-5))
    assert front.ready is not None
    xn = ref.ref_add_rmsnorm(None, first.clone(), g, 1e-5, torch.float64)
    torch.testing.assert_close(o.linear(front, w, out_dtype=torch.float32).double(), xn @ w.double().T, atol=2e-2, rtol=1e-2)
    gu = xn @ wg.double().T
    torch.testing.assert_close(o.linear_silu_mul(front, wg, I).double(), torch.nn.functional.silu(gu[:, :I]) * gu[:, I:], atol=3e-2, rtol=2e-2)


def test_skinny_workgroups_a_compute_unit_holds(ops):
    """The LDS of a few-row product's workgroup leaves a compute unit room for as many as its rule counts on: two of two tiles, three
    of one tile and up to 8 rows, with a norm in front as without one."""
    lib, cu = ops[torch.bfloat16].lib("gemm_bf16"), torch.cuda.get_device_properties(0).multi_processor_count
    for epi, columns in ((0, 16), (1, 16), (3, 8), (5, 8)):
        for fused in (0, 1):
            for rows in (9, 16):                      # one tile to two a compute unit, and more than three
                assert lib.mie_skinny_held(epi, rows, columns * 2 * cu, fused) >= 2
                assert lib.mie_skinny_held(epi, rows, columns * 4 * cu, fused) >= 2
            for rows in (1, 8):
                assert lib.mie_skinny_held(epi, rows, columns * 2 * cu, fused) >= 2
                assert lib.mie_skinny_held(epi, rows, columns * 4 * cu, fused) >= 3
                assert lib.mie_skinny_held(epi, rows, columns * 20 * cu, fused) >= 2


# --------------------------------------------------- products of 17 to 128 rows (bfloat16), split over K
@pytest.fixture(scope="module")
def engine_ops():
    """The backend with the engine's own thresholds between its three product paths."""
    from mini_inference_engine_amd.kernels.hip_backend import HipBackend
    return HipBackend(torch.bfloat16, DEV)


MID_SHAPES = [(33, 2048, 2048), (64, 2048, 2560), (128, 5632, 2048), (50, 2008, 1000), (37, 256, 64), (100, 4104, 4096),
              (65, 4096, 4), (40, 4096, 2048), (48, 8, 4), (17, 2048, 2048), (24, 520, 72), (128, 2048, 2560), (96, 264, 128)]


@pytest.mark.parametrize("shape", MID_SHAPES)
def test_mid_linear(engine_ops, shape):
    M, K, N = shape
    o = engine_ops
    torch.manual_seed(M * 5 + N)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    assert o._mid_ok(x, w, None) and not o._skinny_ok(x, w, None), "this shape must take the split product"
    exact = x.double() @ w.double().T
    y32 = o.linear(x, w, out_dtype=torch.float32)
    torch.testing.assert_close(y32.double(), exact, atol=1e-4, rtol=1e-4)        # float32 sums of exact products
    y = o.linear(x, w)
    assert y.dtype == torch.bfloat16
    torch.testing.assert_close(y.float(), exact.float(), atol=2e-2, rtol=1e-2)
    # a row's result does not depend on the rows beside it, nor on the number of row tiles
    for a, b in ((0, 33), (max(0, M - 33), M), (0, min(M, 64))):
        assert torch.equal(o.linear(x[a:b].contiguous(), w, out_dtype=torch.float32), y32[a:b])
    most = 128
    big = torch.cat([x, x[:most - M]]) if M < most else x
    assert torch.equal(o.linear(big, w, out_dtype=torch.float32)[:M], y32)
    # residual add
    stream = torch.randn(M, N, device=DEV)
    expect = stream.double() + exact
    assert o.linear(x, w, add_to=stream) is None
    torch.testing.assert_close(stream.double(), expect, atol=1e-4, rtol=1e-4)
    # residual add and the norm that reads the stream next, float32 and bfloat16 norm weights
    from mini_inference_engine_amd.kernels.api import Normed, Sink
    for gdt in (torch.float32, torch.bfloat16):
        stream = torch.randn(M, N, device=DEV)
        g = (1 + 0.1 * torch.randn(N, device=DEV)).to(gdt)
        r = stream.double() + exact
        want = r * torch.rsqrt(r.pow(2).mean(-1, keepdim=True) + 1e-5) * g.double()
        out = o.linear(x, w, add_to=Sink(stream, g, 1e-5))
        assert isinstance(out, Normed) and out.pending is None and out.weight is g
        torch.testing.assert_close(stream.double(), r, atol=1e-4, rtol=1e-4)
        torch.testing.assert_close(out.materialize().double(), want, atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("shape", [(129, 4096, 264), (300, 4160, 2048), (512, 5632, 136), (385, 4096, 4104), (255, 4672, 2056), (509, 4160, 5128)])
def test_tile_product_in_parts(engine_ops, shape):
    """A long K in parts on the own tiles, added into the stream with and without the norm behind it: rows and columns beyond
    the tiles, K whose stages do not divide over the parts; the float32 sums within the worst case of their additions."""
    from mini_inference_engine_amd.kernels.api import Sink
    o, (M, K, N) = engine_ops, shape
    torch.manual_seed(M)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    units = o._tile_split(x, w, None)
    assert units >= 2 and (units - 1) * -(-(K // 64) // units) < K // 64, "the case must take the path it is for"
    stream = torch.randn(M, N, device=DEV)
    expect = stream.double() + x.double() @ w.double().T
    bound = (K + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -22 * expect.abs()
    plain = stream.clone()
    with counted(o, "tile_gemm_bf16", "mie_tile_gemm_units") as calls:
        assert o.linear(x, w, add_to=plain) is None
    assert len(calls) == 1
    assert bool(((plain.double() - expect).abs() <= bound).all())
    g = torch.randn(N, device=DEV).to(torch.bfloat16)
    normed = o.linear(x, w, add_to=Sink(stream, g, 1e-5))
    assert torch.equal(stream, plain)
    torch.testing.assert_close(normed.materialize().float(), torch.nn.functional.rms_norm(plain, (N,), g.float(), 1e-5), atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("case", [(torch.float32, 5, 64, 36), (torch.float32, 70, 64, 132), (torch.bfloat16, 300, 4096, 264)])
def test_a_stream_off_16_bytes_is_added_to(engine_ops, ops, case):
    """A contiguous float32 stream (and a norm weight) that starts anywhere: what the kernels for 16-byte pieces do not take goes
    where it went without them, and the sum arrives either way."""
    from mini_inference_engine_amd.kernels.api import Normed, Sink
    dtype, M, K, N = case
    o = engine_ops if dtype == torch.bfloat16 else ops[dtype]
    torch.manual_seed(K)
    x = torch.randn(M, K, device=DEV).to(dtype)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(dtype)
    base, g = torch.randn(M, N, device=DEV), torch.randn(N + 1, device=DEV)[1:]
    want = base.double() + x.double() @ w.double().T
    for off in (0, 1):
        stream = torch.empty(M * N + off, device=DEV)[off:].view(M, N).copy_(base)
        normed = o.linear(x, w, add_to=Sink(stream, g, 1e-5))
        if torch.is_tensor(normed):                 # not added yet: the caller's to do
            stream += normed
        else:
            assert isinstance(normed, Normed)
            y = torch.nn.functional.rms_norm(want, (N,), g.double(), 1e-5)
            torch.testing.assert_close(normed.materialize().double(), y, **tol(dtype))
        torch.testing.assert_close(stream.double(), want, atol=1e-4, rtol=1e-4)


# rows, K, columns; the estimate's time of a stage, whether the product is better off on the own tiles by it, and the tile that is taken
@pytest.mark.parametrize("case", [(129, 64, 104, 0.76, True, 128128), (192, 2048, 5632, 0.76, True, 128128), (300, 192, 96, 0.76, True, 128128),
                                  (380, 64, 5512, 0.98, True, 128192), (510, 128, 5512, 0.99, True, 128192), (513, 128, 5640, 1.33, True, 192192),
                                  (1300, 2048, 2816, 1.33, False, 192192), (1020, 64, 6152, 1.57, True, 256256), (2047, 64, 1000, 0.76, True, 128128),
                                  (525, 64, 5200, 0.98, True, 192128), (1307, 128, 2272, 0.98, True, 192128), (457, 192, 8184, 0.99, True, 256128),
                                  (959, 64, 3896, 0.99, True, 256128), (690, 128, 7176, 1.33, True, 256192), (1193, 192, 3488, 1.33, True, 256192),
                                  (1169, 64, 7880, 2.35, True, 256320), (1479, 192, 5976, 2.35, True, 256320),
                                  (790, 1152, 5640, 1.33, True, 256192), (1129, 1152, 5624, 1.57, True, 256256),
                                  (250, 1152, 5640, 0.76, True, 128128), (381, 1152, 4104, 0.76, True, 128128), (505, 1152, 8152, 0.99, True, 256128),
                                  (1010, 1152, 4088, 0.99, True, 256128), (377, 1152, 5512, 0.98, True, 128192), (525, 1152, 5208, 0.98, True, 192128),
                                  (1169, 1152, 7880, 2.35, True, 256320), (513, 1152, 5640, 1.33, True, 192192),
                                  (160, 1152, 14328, 0.98, True, 192128), (383, 1152, 8184, 0.98, True, 192128), (255, 1152, 11256, 0.99, True, 128192)])
def test_tile_product_swiglu(engine_ops, case):
    """Gate and up on the own tiles (every tile size, edges in rows and columns, the shortest K and one whose stages go round the ring)
    with SwiGLU on the float32 sums, against 64 bits rounded once (2^-8 of a value for bfloat16, and the hardware's exponential beside it)."""
    from mini_inference_engine_amd.kernels import library
    (M, K, inter, stage_us, gains, tile), o = case, engine_ops
    torch.manual_seed(K + inter)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * inter, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    out = torch.full((M, inter + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    lib = o.lib("tile_gemm_bf16")
    assert lib.mie_tile_gemm_swiglu_tile(M, inter) == tile, "the case must take the tile it is for"
    library.check(lib, lib.mie_tile_gemm_swiglu(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), inter + 8, M, inter, K,
                                                torch.cuda.current_stream().cuda_stream))
    gu = x.double() @ w.double().T
    expect = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    assert bool(((out[:, :inter].double() - expect).abs() <= 2.0 ** -8 * expect.abs() + 1e-4).all())
    assert bool((out[:, inter:] == 7.0).all()), "nothing beyond the columns"
    odd = torch.full((M, inter + 4), 7.0, device=DEV, dtype=torch.bfloat16)          # rows that begin on 8 bytes
    library.check(lib, lib.mie_tile_gemm_swiglu(x.data_ptr(), K, w.data_ptr(), K, odd.data_ptr(), inter + 4, M, inter, K,
                                                torch.cuda.current_stream().cuda_stream))
    assert torch.equal(odd[:, :inter], out[:, :inter]) and bool((odd[:, inter:] == 7.0).all())
    assert abs(lib.mie_tile_gemm_swiglu_cost(M, inter, K) - 100 * stage_us * (K // 64)) <= 1
    assert o._tile_swiglu_gains(x, w, inter) == gains
    with counted(o, "tile_gemm_bf16", "mie_tile_gemm_swiglu") as calls:
        made = o.linear_silu_mul(x, w, inter)
    assert len(calls) == gains
    if gains:
        assert torch.equal(made, out[:, :inter])
    assert lib.mie_tile_gemm_swiglu(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), inter + 8, M, inter, K - 8, None) != 0
    assert lib.mie_tile_gemm_units(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), M, inter, K, K // 64 + 1, None) != 0


# rows, columns, K and the tile: every tile, edges in rows and columns, K of one stage or of no more than the ring holds, and of more than it
# holds and is read ahead at once
@pytest.mark.parametrize("case", [(137, 72, 64, 64064), (333, 2056, 320, 64064), (138, 5560, 64, 64080), (509, 2552, 576, 64080), (193, 5240, 192, 64096),
                                  (263, 4912, 256, 64128), (513, 4520, 64, 80128), (1131, 2040, 1408, 80128), (520, 4624, 192, 96128), (483, 5392, 64, 128128),
                                  (2047, 2040, 1088, 128128), (646, 5392, 1024, 128160), (642, 5488, 320, 128192), (1027, 5416, 448, 256128), (2047, 4096, 14400, 256128),
                                  (263, 3080, 1088, 64064), (395, 2552, 1088, 64080), (395, 3080, 1088, 64096), (333, 4104, 1088, 64128), (509, 5368, 1088, 96128),
                                  (771, 4912, 1088, 128160), (901, 5368, 1088, 128192), (1290, 5368, 1088, 256128)])
def test_tile_product_added(engine_ops, case):
    """A product on the own tiles added into the stream: every tile; the float32 sums within the worst case of their additions, nothing
    written beyond the last row."""
    o, (M, N, K, tile) = engine_ops, case
    lib = o.lib("tile_gemm_bf16")
    assert lib.mie_tile_gemm_tile(M, N, K) == tile, "the case must take the tile it is for"
    torch.manual_seed(M + K)
    x = torch.randn(M, K + 8, device=DEV).to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K + 16, device=DEV) / math.sqrt(K)).to(torch.bfloat16)[:, :K]
    held = torch.randn(M + 3, N, device=DEV)
    behind, expect = held[M:].clone(), held[:M].double() + x.double() @ w.double().T
    bound = (K + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -22 * expect.abs()
    with counted(o, "tile_gemm_bf16", "mie_tile_gemm_add") as calls:
        assert o.linear(x, w, add_to=held[:M]) is None
    assert len(calls) == 1
    assert bool(((held[:M].double() - expect).abs() <= bound).all()) and torch.equal(held[M:], behind)
    assert lib.mie_tile_gemm_tile(4096, 8192, K) == 0 and lib.mie_tile_gemm_add(x.data_ptr(), K + 8, w.data_ptr(), K + 16, held.data_ptr(), N, M, N, K - 8, None) != 0


# rows, q and kv heads, head size, K and the tile: every tile; pairs of tiles within a head, across heads, across q and k and across k and v, and the
# lone last one of an odd number; K of one stage, of as many as the ring holds and of many more; edges in rows and columns
@pytest.mark.parametrize("case", [(137, 2, 1, 16, 64, 64064), (333, 32, 4, 64, 320, 64064), (300, 3, 3, 80, 128, 64064), (700, 5, 2, 48, 64, 64064), (260, 2, 2, 256, 128, 64064),
                                  (512, 32, 4, 64, 192, 64080), (410, 31, 5, 64, 2048, 64080), (560, 32, 4, 64, 2048, 64096), (1500, 7, 1, 112, 64, 64128),
                                  (700, 32, 4, 64, 2048, 64128), (900, 32, 4, 64, 2048, 80128), (1131, 32, 4, 64, 64, 96128), (1131, 32, 4, 64, 1088, 96128),
                                  (520, 32, 8, 128, 64, 128128), (1500, 32, 4, 64, 2048, 128128), (2047, 32, 4, 64, 2048, 128160), (1801, 33, 3, 64, 2048, 128160),
                                  (2040, 32, 4, 64, 128, 128192), (1020, 32, 8, 128, 64, 128192), (1020, 32, 8, 128, 4096, 128192), (1100, 32, 8, 128, 4096, 256128)])
def test_tile_projection_rotary_store(engine_ops, case):
    """The q/k/v projection of many rows with rotation and cache write on the own tiles' sums: against the same kernels' float32 sums
    finished by a kernel of their own (one rounding of bfloat16 apart where the sums' order differs), other pages untouched."""
    from mini_inference_engine_amd.parts.rope import rotary_tables
    o, (M, Hq, Hkv, D, K, tile) = engine_ops, case
    torch.manual_seed(M + D)
    N, page = (Hq + 2 * Hkv) * D, 32
    assert o.lib("tile_gemm_bf16").mie_tile_gemm_tile(M, N, K) == tile, "the case must take the tile it is for"
    pages = -(-M // page) + 3
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 3000))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    pos = torch.randint(0, 3000, (M,), device=DEV, dtype=torch.int32)
    slots = (torch.randperm((pages - 1) * page, device=DEV)[:M] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.bfloat16)
    kc2, vc2 = kc.clone(), vc.clone()
    with counted(o, "tile_gemm_bf16", "mie_tile_gemm_qkv_rope") as calls:
        q = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, slots)
    assert len(calls) == 1 and tuple(q.shape) == (M, Hq * D)
    q2 = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc2, vc2, slots, for_attention=True).finish()
    for a, b in ((q, q2), (kc, kc2), (vc, vc2)):
        assert bool(((a.double() - b.double()).abs() <= 2.0 ** -7 * b.double().abs() + 1e-4).all())
    fresh = torch.ones(pages * page, dtype=torch.bool, device=DEV)
    fresh[slots.long()] = False
    assert torch.equal(kc[0], kc2[0]) and torch.equal(vc[0], vc2[0])
    at = fresh.view(pages, page)
    assert torch.equal(kc.transpose(1, 2)[at], kc2.transpose(1, 2)[at]) and torch.equal(vc.permute(0, 3, 1, 2)[at], vc2.permute(0, 3, 1, 2)[at])


# rows, K, columns and how many of them are made by uncut tiles
@pytest.mark.parametrize("case", [(512, 2048, 5632, 4096), (384, 72, 5632, 5440), (260, 72, 7000, 0), (129, 96, 8256, 8192), (600, 64, 3300, 3264), (400, 200, 4096, 4096),
                                  (520, 40, 3332, 3264), (2047, 200, 1000, 1000)])
def test_float32_gated_product_partly_uncut(ops, case):
    """Gate and up in float32 where the columns that fill the grid's rounds are uncut tiles with SwiGLU behind them and the others go in
    parts: the bits of the product and silu_mul, edges in rows, columns and K, results beyond what the parts can hold too."""
    o, (M, K, inter, whole) = ops[torch.float32], case
    lib = o.lib("gemm_f32")
    assert lib.mie_f32_whole_columns(M, inter, K) == whole, "the case must take the path it is for"
    torch.manual_seed(M + K)
    x, w = torch.randn(M, K, device=DEV), torch.randn(2 * inter, K, device=DEV) / math.sqrt(K)
    x[M // 2, 3] = 2.0e36
    with counted(o, "gemm_f32", "mie_gemm_f32_gated") as calls:
        y = o.linear_silu_mul(x, w, inter)
    assert len(calls) == (whole > 0)
    assert torch.equal(y, o.silu_mul(o.linear(x, w), inter))
    assert lib.mie_f32_whole_columns(16, inter, K) == 0
    assert lib.mie_gemm_f32_gated(x.data_ptr(), K, w.data_ptr(), K, y.data_ptr(), inter, None, 16, inter, K, None) != 0


@pytest.mark.parametrize("case", [(2047, 192, 5640), (1281, 64, 7496), (1793, 128, 6144), (2048, 2048, 5632)])
def test_wide_tile_product_swiglu(engine_ops, case):
    """Gate and up on tiles of 256 x 384 (taken where they make one round of what other tiles need two for): edges in rows and
    columns, one stage and many; against 64 bits rounded once."""
    from mini_inference_engine_amd.kernels import library
    o, (M, K, inter) = engine_ops, case
    torch.manual_seed(K + inter)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * inter, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    lib = o.lib("tile_gemm_bf16")
    assert lib.mie_tile_gemm_swiglu_tile(M, inter) == 256384, "the case must take the tile it is for"
    assert abs(lib.mie_tile_gemm_swiglu_cost(M, inter, K) - 235 * (K // 64)) <= 1
    out = torch.full((M, inter + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    library.check(lib, lib.mie_tile_gemm_swiglu(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), inter + 8, M, inter, K,
                                                torch.cuda.current_stream().cuda_stream))
    gu = x.double() @ w.double().T
    expect = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    assert bool(((out[:, :inter].double() - expect).abs() <= 2.0 ** -8 * expect.abs() + 1e-4).all())
    assert bool((out[:, inter:] == 7.0).all()), "nothing beyond the columns"


@pytest.mark.parametrize("g_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", [(1, 1024, 4, 4), (8, 2048, 2048, 4), (9, 1028, 1000, 4), (16, 5632, 516, 4), (17, 2052, 36, 8), (20, 1024, 4096, 4), (20, 1024, 4100, 0),
                                  (100, 360, 2048, 4), (40, 1536, 8192, 0), (4, 2048, 6144, 0), (300, 200, 132, 8)])
def test_float32_product_with_the_norm_behind_it(ops, case, g_dtype):
    """A float32 product added into the stream whose norm follows: parts of K that meet in the kernel that adds and norms give
    the bits of the product, the add and the norm by themselves (every width of a thread, quarters and eighths, edges of tiles);
    rows of more than 4,096 numbers keep kernels of their own for the two."""
    from mini_inference_engine_amd.kernels.api import Sink
    o, (M, K, N, units) = ops[torch.float32], case
    lib = o.lib("gemm_f32")
    assert lib.mie_f32_norm_units(M, N, K) == units, "the case must take the path it is for"
    torch.manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) / math.sqrt(K)
    x[M // 2, 3] = 3.0e38                       # results beyond what the parts can hold are computed again, here too
    g = (1 + 0.1 * torch.randn(N, device=DEV)).to(g_dtype)
    stream = torch.randn(M, N, device=DEV)
    plain = stream.clone()
    assert o.linear(x, w, add_to=plain) is None
    with counted(o, "gemm_f32", "mie_gemm_f32_add_norm") as calls:
        normed = o.linear(x, w, add_to=Sink(stream, g, 1e-5))
    assert len(calls) == (units > 0) and torch.equal(stream, plain)
    assert torch.equal(normed.materialize(), o.add_rmsnorm(None, plain, g, 1e-5))
    assert lib.mie_f32_norm_units(16, 8196, 2048) == 0 and lib.mie_f32_norm_units(4, 64, 512) == 0
    assert lib.mie_gemm_f32_add_norm(x.data_ptr(), K, w.data_ptr(), K, stream.data_ptr(), g.data_ptr(), 1, None, x.data_ptr(), M, N, K, 1e-5, None) != 0


@pytest.mark.parametrize("M", [4, 100])
def test_the_norm_behind_a_float32_product_is_of_the_wanted_type(ops, M):
    """The norm that a float32 product's last kernel makes beside the add: of the backend's type where none is asked for, of another
    where that is, the bits of the norm by itself."""
    from mini_inference_engine_amd.kernels.api import Sink
    torch.manual_seed(M)
    x, w, g = torch.randn(M, 2048, device=DEV), torch.randn(256, 2048, device=DEV) / 45, torch.randn(256, device=DEV)
    for dtype, asked in ((torch.float32, None), (torch.float32, torch.bfloat16), (torch.bfloat16, None), (torch.bfloat16, torch.float32)):
        stream = torch.randn(M, 256, device=DEV)
        y = ops[dtype].linear(x, w, out_dtype=torch.float32, add_to=Sink(stream, g, 1e-5)).materialize(asked)
        assert y.dtype == (asked or dtype)
        assert torch.equal(y, ops[dtype].add_rmsnorm(None, stream, g, 1e-5, out_dtype=y.dtype))


# rows, K, columns and the tiles of 16 weight rows a workgroup has
@pytest.mark.parametrize("case", [(17, 64, 4, 1), (33, 72, 12, 1), (64, 2008, 3000, 2), (48, 328, 5632, 3), (128, 2048, 5632, 3),
                                  (50, 8, 8188, 4), (97, 200, 8192, 4), (31, 136, 11008, 6), (64, 192, 11004, 6), (64, 256, 14336, 7)])
def test_mid_product_swiglu(engine_ops, case):
    """Gate and up of 17 to 128 rows with SwiGLU on the float32 sums: every number of tiles, edges in rows and columns, K that is
    no multiple of a chunk, fewer chunks than waves; against 64 bits rounded once, and a row's bits whatever is beside it."""
    o, (M, K, inter, tiles) = engine_ops, case
    torch.manual_seed(K + inter)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * inter, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    lib = o.lib("gemm_mid_bf16")
    assert lib.mie_mid_swiglu_tiles(M, inter) == tiles, "the case must take the tiles it is for"
    with counted(o, "gemm_mid_bf16", "mie_mid_swiglu") as calls:
        y = o.linear_silu_mul(x, w, inter)
    assert len(calls) == 1
    gu = x.double() @ w.double().T
    expect = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    assert bool(((y.double() - expect).abs() <= 2.0 ** -8 * expect.abs() + 1e-4).all())
    for a, b in ((0, 17), (max(0, M - 33), M)):
        if b - a > 16:
            assert torch.equal(o.linear_silu_mul(x[a:b].contiguous(), w, inter), y[a:b])
    out = torch.full((M, inter + 4), 7.0, device=DEV, dtype=torch.bfloat16)
    assert lib.mie_mid_swiglu(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), inter + 4, M, inter, K,
                              torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out[:, :inter], y) and bool((out[:, inter:] == 7.0).all()), "nothing beyond the columns"
    assert lib.mie_mid_swiglu(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), inter + 4, 129, inter, K, None) != 0
    assert lib.mie_mid_swiglu(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), inter + 4, M, inter, K - 4, None) != 0


def far_rows(t, stride):
    """The same matrix with its rows ``stride`` numbers apart."""
    return torch.empty((t.shape[0] - 1) * stride + t.shape[1], dtype=t.dtype, device=DEV).as_strided(t.shape, (stride, 1)).copy_(t)


# rows of x, K, weight rows and the strides of both: the largest that the kernels' 32-bit offsets reach
@pytest.mark.parametrize("case", [(16, 72, 24, 72, 1 << 28), (16, 64, 40, 1 << 24, 64), (128, 136, 100, 136, 1 << 24), (128, 64, 72, 1 << 24, 1 << 24)])
def test_products_of_rows_far_apart(engine_ops, case):
    """Few-row and split products whose rows lie as far apart as they take: the bits of compact operands; further apart is refused
    by the C entries and left to the library by the backend."""
    o, (M, K, N, ldx, ldw) = engine_ops, case
    torch.manual_seed(N)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    fx, fw = far_rows(x, ldx), far_rows(w, ldw)
    ok = o._skinny_ok if M <= 16 else o._mid_ok
    assert ok(fx, fw, None)
    assert torch.equal(o.linear(fx, fw, out_dtype=torch.float32), o.linear(x, w, out_dtype=torch.float32))
    assert torch.equal(o.linear_silu_mul(fx, fw, N // 2), o.linear_silu_mul(x, w, N // 2))
    y, s = torch.empty(M, N, device=DEV), torch.cuda.current_stream().cuda_stream
    far = max(ldx, ldw) + 8
    args = (x.data_ptr(), far if ldx > K else K, w.data_ptr(), far if ldw > K else K)
    if M <= 16:
        assert o.lib("gemm_bf16").mie_skinny_gemm(*args, y.data_ptr(), N, 1, M, N, K, None, 0, None, 0, None, None, 0, 0.0, None, s) != 0
    else:
        assert o.lib("gemm_mid_bf16").mie_mid_gemm(*args, y.data_ptr(), M, N, K, 1, None, s) != 0


@pytest.mark.parametrize("case", [(64, 64, 9220, True), (65, 64, 9216, True), (65, 64, 9220, False), (128, 64, 14336, False), (128, 2048, 5632, True),
                                  (128, 2056, 512, False)])
def test_mid_product_swiglu_is_taken_where_it_gains(engine_ops, case):
    """More than 64 rows of a weight that gives a compute unit more than four and a half tiles, or of a longer K, keep the library's
    product and silu_mul."""
    o, (M, K, inter, taken) = engine_ops, case
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    torch.manual_seed(M)
    x, w = torch.randn(M, K, device=DEV).to(torch.bfloat16), (torch.randn(2 * inter, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    with counted(o, "gemm_mid_bf16", "mie_mid_swiglu") as calls:
        y = o.linear_silu_mul(x, w, inter)
    assert len(calls) == taken
    gu = x.double() @ w.double().T
    torch.testing.assert_close(y.double(), torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:], atol=2e-2, rtol=2e-2)


def test_mid_linear_refuses_what_it_cannot_run(engine_ops):
    o = engine_ops
    lib = o.lib("gemm_mid_bf16")
    x = torch.zeros(200, 64, device=DEV, dtype=torch.bfloat16)
    w = torch.zeros(64, 64, device=DEV, dtype=torch.bfloat16)
    part = torch.zeros(1, 200, 64, device=DEV)
    z = torch.zeros(64, dtype=torch.int32, device=DEV)
    assert lib.mie_mid_gemm(x.data_ptr(), 64, w.data_ptr(), 64, part.data_ptr(), 200, 64, 64, 1, z.data_ptr(), None) != 0
    assert b"at most 128" in lib._mie_error()
    assert lib.mie_mid_gemm(x.data_ptr(), 60, w.data_ptr(), 60, part.data_ptr(), 40, 64, 60, 1, z.data_ptr(), None) != 0
    assert b"multiple of 8" in lib._mie_error()
    assert lib.mie_mid_reduce(part.data_ptr(), 1, 40, 66, 1, part.data_ptr(), 66, None, None, 0, None, 0, 0.0, None) != 0
    assert b"width" in lib._mie_error()
    assert not o._mid_ok(x[:40], torch.zeros(8192, 64, device=DEV, dtype=torch.bfloat16), None), "wide weights go to the library"


@pytest.mark.parametrize("geom", [(2, 1, 16), (3, 1, 32), (4, 2, 48), (32, 4, 64), (5, 5, 96), (8, 2, 128), (2, 1, 256)])
@pytest.mark.parametrize("M", [24, 40, 64, 128])
def test_mid_projection_rotary_store(engine_ops, geom, M):
    """Split projection, then one kernel for sum + rotary + cache write, against the separate references
    (K long enough for four splits at 24, 40 and 128 rows, one split at 64)."""
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D = geom
    o = engine_ops
    torch.manual_seed(D + M)
    K, page, pages = (264 if M == 64 else 1032), 16, 12
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 300))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    assert o._mid_ok(x, w, None)
    pos = torch.randint(0, 300, (M,), device=DEV, dtype=torch.int32)
    slots = (torch.randperm((pages - 1) * page, device=DEV)[:M] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.bfloat16)
    kc_ref, vc_ref = kc.float(), vc.float()
    qkv_ref = ref.ref_linear(x, w, None, torch.float32)
    ref.ref_rotary_kv_store(qkv_ref, pos, cos, sin, D, Hq, Hkv, D, kc_ref, vc_ref, slots)
    out = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, slots)
    assert tuple(out.shape) == (M, Hq * D), "q alone comes back"
    torch.testing.assert_close(out.float(), qkv_ref[:, :Hq * D], atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(kc.float(), kc_ref, atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(vc.float(), vc_ref, atol=2e-2, rtol=1e-2)
    assert torch.equal(kc[0].float(), kc_ref[0]) and torch.equal(vc[0].float(), vc_ref[0]), "untouched pages stay untouched"


@pytest.mark.parametrize("geom", [(2, 1, 16), (3, 1, 32), (4, 2, 48), (32, 4, 64), (5, 5, 96), (8, 2, 128), (2, 1, 256)])
@pytest.mark.parametrize("slots_kind", ["page starts", "mid page", "scattered"])
def test_many_row_projection_rotary_store(engine_ops, geom, slots_kind):
    """More than 128 rows: library product with float32 sums, then one kernel for rotary + cache write that
    reads those sums (16 tokens and 4 heads a workgroup; values turned in the LDS).  Slots in runs from a
    page's start (the 32-byte path), runs from the middle of a page, and scattered; a token count that is no
    multiple of 16; pages of 16 and of 32."""
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D = geom
    o = engine_ops
    M, K = 203, 264
    page = 32 if D == 48 else 16
    pages = 2 + -(-(M + page) // page)
    torch.manual_seed(D + len(slots_kind))
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 300))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    assert not o._mid_ok(x, w, None) and not o._skinny_ok(x, w, None)
    pos = torch.randint(0, 300, (M,), device=DEV, dtype=torch.int32)
    if slots_kind == "page starts":
        slots = torch.arange(M, device=DEV, dtype=torch.int32) + page
    elif slots_kind == "mid page":
        slots = torch.arange(M, device=DEV, dtype=torch.int32) + page + 5
    else:
        slots = (torch.randperm((pages - 1) * page, device=DEV)[:M] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.bfloat16)
    kc_ref, vc_ref = kc.float(), vc.float()
    qkv_ref = ref.ref_linear(x, w, None, torch.float32)
    ref.ref_rotary_kv_store(qkv_ref, pos, cos, sin, D, Hq, Hkv, D, kc_ref, vc_ref, slots)
    out = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, slots)
    assert tuple(out.shape) == (M, Hq * D), "q alone comes back"
    # one rounding, of the rotated float32 value
    torch.testing.assert_close(out.float(), qkv_ref[:, :Hq * D], atol=1e-2, rtol=8e-3)
    torch.testing.assert_close(kc.float(), kc_ref, atol=1e-2, rtol=8e-3)
    torch.testing.assert_close(vc.float(), vc_ref, atol=1e-2, rtol=8e-3)
    assert torch.equal(kc[0].float(), kc_ref[0]) and torch.equal(vc[0].float(), vc_ref[0]), "untouched pages stay untouched"
    written = torch.zeros(pages * page, dtype=torch.bool, device=DEV)
    written[slots.long()] = True
    keep = ~written.view(pages, page)
    assert torch.equal(kc.float().permute(0, 2, 1, 3)[keep], kc_ref.permute(0, 2, 1, 3)[keep]), "other slots' keys stay"
    assert torch.equal(vc.float().permute(0, 3, 1, 2)[keep], vc_ref.permute(0, 3, 1, 2)[keep]), "other slots' values stay"


def test_projection_kernels_refuse_what_they_cannot_run(engine_ops):
    """The entry points that take the projection's float32 sums name what is wrong instead of running."""
    o = engine_ops
    z = torch.zeros(64, device=DEV)
    zi = torch.zeros(64, device=DEV, dtype=torch.int32)
    zb = torch.zeros(4096, device=DEV, dtype=torch.bfloat16)
    p = lambda t: t.data_ptr()
    lib = o.lib("rope_kv")
    # head size 20 is no multiple of 8; a page of 24 is no multiple of 16; leading dimension too short
    assert lib.mie_rotary_kv_store_sums(p(z), 80, p(zb), 40, p(zi), p(z), p(z), p(zi), p(zb), p(zb), 2, 1, 20, 16, 1, None) != 0
    assert b"multiple of 8" in lib._mie_error()
    assert lib.mie_rotary_kv_store_sums(p(z), 64, p(zb), 32, p(zi), p(z), p(z), p(zi), p(zb), p(zb), 2, 1, 16, 24, 1, None) != 0
    assert b"page" in lib._mie_error()
    assert lib.mie_rotary_kv_store_sums(p(z), 48, p(zb), 32, p(zi), p(z), p(z), p(zi), p(zb), p(zb), 2, 1, 16, 16, 1, None) != 0
    assert b"leading dims" in lib._mie_error()
    assert lib.mie_rotary_kv_store_sums(None, 64, p(zb), 32, p(zi), p(z), p(z), p(zi), p(zb), p(zb), 2, 1, 16, 16, 1, None) != 0
    assert b"null" in lib._mie_error()
    lib = o.lib("attention_bf16", ("-DHEAD_DIM=16",))
    args = lambda Hq, Hkv, D, splits, ld: (p(z), splits, 0, ld, p(z), p(z), p(zi), p(zb), p(zb), p(zb), p(zi), 4, p(zi), 1, Hq, Hkv, D,
                                         16, 1.0, 0, lib.mie_decode_block_keys(), None)
    assert lib.mie_decode_attention_from_sums(*args(34, 2, 16, 1, 608)) != 0
    assert b"at most 16" in lib._mie_error()
    assert lib.mie_decode_attention_from_sums(*args(4, 2, 32, 1, 256)) != 0
    assert b"built for head_dim 16" in lib._mie_error()
    assert lib.mie_decode_attention_from_sums(*args(4, 2, 16, 1, 100)) != 0
    assert b"row stride" in lib._mie_error()
    assert lib.mie_decode_attention_from_sums(*args(4, 2, 16, 3, 128)) != 0      # three splits with a stride of 0
    assert b"splits" in lib._mie_error()


def test_few_row_product_refuses_what_it_cannot_run(engine_ops):
    o = engine_ops
    lib = o.lib("gemm_bf16")
    assert lib.mie_skinny_max_rows() == o.SKINNY_MAX_ROWS == 16
    x = torch.zeros(17, 64, device=DEV, dtype=torch.bfloat16)
    w = torch.zeros(32, 64, device=DEV, dtype=torch.bfloat16)
    y = torch.zeros(17, 32, device=DEV, dtype=torch.bfloat16)
    call = lambda M, K, ldx: lib.mie_skinny_gemm(x.data_ptr(), ldx, w.data_ptr(), 64, y.data_ptr(), 32, 0, M, 32, K, None, 0, None, 0,
                                                 None, None, 0, 0.0, None, None)
    assert call(17, 64, 64) != 0 and b"at most 16" in lib._mie_error()
    assert call(16, 60, 64) != 0 and b"multiple of 8" in lib._mie_error()
    assert call(16, 64, 56) != 0 and b"leading dims" in lib._mie_error()
    assert call(16, 64, 64) == 0
    assert not o._skinny_ok(x, w, None) and o._skinny_ok(x[:16], w, None)


def test_lazy_norm_input_adds_once(ops):
    """A Normed handed to linear: what is pending is added to the stream exactly once, however often it is used."""
    o = ops[torch.bfloat16]
    torch.manual_seed(0)
    stream = torch.randn(40, 96, device=DEV)
    g = torch.randn(96, device=DEV).to(torch.bfloat16)
    w = (torch.randn(331, 96, device=DEV) / 10).to(torch.bfloat16)
    rows = torch.tensor([39, 0, 7, 7, 21], device=DEV, dtype=torch.int32)
    y = o.linear(normed(o, stream, g, 1e-6, rows=rows), w, out_dtype=torch.float32)
    expect = ref.ref_add_rmsnorm(None, stream.clone(), g, 1e-6, torch.float64, rows) @ w.double().T
    torch.testing.assert_close(y.double(), expect, atol=2e-2, rtol=1e-2)
    pending = torch.randn(40, 96, device=DEV).to(torch.bfloat16)
    lazy = normed(o, stream.clone(), g, 1e-6, pending=pending)
    y2 = o.linear(lazy, w, out_dtype=torch.float32)
    y3 = o.linear(lazy, w, out_dtype=torch.float32)
    assert torch.equal(y2, y3) and lazy.pending is None
    torch.testing.assert_close(lazy.residual, stream + pending.float())


@pytest.mark.parametrize("g_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M, width, inner", [(1, 64, 176), (8, 2048, 512), (16, 96, 64), (5, 120, 328), (13, 200, 48), (3, 4160, 64)])
def test_norm_folded_into_neighbouring_products(ops, M, width, inner, g_dtype):
    """stream += x W1^T, then the RMSNorm of the stream, then a product: the norm has no kernel of its own.
    The first product prepares its input (values times weight, rounded; sums of squares per tile), the
    second applies 1 / sqrt(mean + eps) to its sums."""
    from mini_inference_engine_amd.kernels.api import Sink
    o = ops[torch.bfloat16]
    torch.manual_seed(M + width)
    x = torch.randn(M, inner, device=DEV).to(torch.bfloat16)
    w1 = (torch.randn(width, inner, device=DEV) / math.sqrt(inner)).to(torch.bfloat16)
    g = (1 + 0.1 * torch.randn(width, device=DEV)).to(g_dtype)
    stream = torch.randn(M, width, device=DEV)
    expect_stream = stream.double() + x.double() @ w1.double().T
    normed_in = o.linear(x, w1, add_to=Sink(stream, g, 1e-5))
    assert normed_in is not None and normed_in.ready is not None, "the fused kernel must have prepared the norm"
    torch.testing.assert_close(stream.double(), expect_stream, atol=2e-3, rtol=2e-3)
    xn = ref.ref_add_rmsnorm(None, stream.clone(), g, 1e-5, torch.float64)
    # consumer 1: plain product, float32 out, gathered rows (the head on wanted rows)
    w2 = (torch.randn(77, width, device=DEV) / math.sqrt(width)).to(torch.bfloat16)
    rows = torch.tensor([M - 1, 0, M // 2], device=DEV, dtype=torch.int32)
    y = o.linear(normed_in.with_rows(rows), w2, out_dtype=torch.float32)
    torch.testing.assert_close(y.double(), xn[rows.long()] @ w2.double().T, atol=2e-2, rtol=1e-2)
    # consumer 2: gate/up with SwiGLU
    w3 = (torch.randn(2 * 48, width, device=DEV) / math.sqrt(width)).to(torch.bfloat16)
    a = o.linear_silu_mul(normed_in, w3, 48)
    gu = xn @ w3.double().T
    torch.testing.assert_close(a.double(), torch.nn.functional.silu(gu[:, :48]) * gu[:, 48:], atol=3e-2, rtol=2e-2)
    # the same Normed, materialised the ordinary way, agrees
    torch.testing.assert_close(normed_in.materialize().double(), xn, atol=2e-2, rtol=1e-2)


def test_norm_folded_into_projection_rotary_store(ops):
    from mini_inference_engine_amd.kernels.api import Sink
    from mini_inference_engine_amd.parts.rope import rotary_tables
    o = ops[torch.bfloat16]
    torch.manual_seed(3)
    M, width, Hq, Hkv, D, page, pages = 8, 256, 4, 2, 64, 16, 6
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 300))
    x = torch.randn(M, 96, device=DEV).to(torch.bfloat16)
    w1 = (torch.randn(width, 96, device=DEV) / 10).to(torch.bfloat16)
    g = (1 + 0.1 * torch.randn(width, device=DEV)).to(torch.bfloat16)
    stream = torch.randn(M, width, device=DEV)
    normed_in = o.linear(x, w1, add_to=Sink(stream, g, 1e-6))
    w = (torch.randn((Hq + 2 * Hkv) * D, width, device=DEV) / 16).to(torch.bfloat16)
    pos = torch.randint(0, 300, (M,), device=DEV, dtype=torch.int32)
    slots = (torch.randperm((pages - 1) * page, device=DEV)[:M] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.bfloat16)
    kc_ref, vc_ref = kc.float(), vc.float()
    xn = ref.ref_add_rmsnorm(None, stream.clone(), g, 1e-6, torch.float32)
    qkv_ref = (xn.double() @ w.double().T).float()
    ref.ref_rotary_kv_store(qkv_ref, pos, cos, sin, D, Hq, Hkv, D, kc_ref, vc_ref, slots)
    q = o.linear_rotary_kv_store(normed_in, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, slots)
    torch.testing.assert_close(q.float(), qkv_ref[:, :Hq * D], atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(kc.float(), kc_ref, atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(vc.float(), vc_ref, atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("M, K, inter", [(1, 64, 176), (8, 2048, 5632), (12, 96, 256), (16, 120, 200), (9, 64, 48), (4, 136, 4800)])
def test_skinny_swiglu(ops, M, K, inter):
    o = ops[torch.bfloat16]
    torch.manual_seed(inter)
    w = (torch.randn(2 * inter, K, device=DEV) / math.sqrt(K) * 2).to(torch.bfloat16)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    assert o._skinny_ok(x, w, None), "this shape must take the fused kernel"
    y = o.linear_silu_mul(x, w, inter)
    gu = x.double() @ w.double().T
    # float32 sums of exact products, one rounding (2^-8 relative) at the end
    torch.testing.assert_close(y.double(), torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:], atol=1e-3, rtol=1e-2)


# ----------------------------------------------------------------- rotary + kv
def make_cache(pages, Hkv, page, D, dtype):
    k = torch.randn(pages, Hkv, page, D, device=DEV).to(dtype)
    return k, torch.randn(pages, Hkv, D, page, device=DEV).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("geom", [(4, 2, 16, 16), (3, 1, 32, 32), (5, 5, 48, 24), (32, 4, 64, 64), (7, 7, 128, 0)])
def test_rotary_kv_store(ops, dtype, geom):
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D, rot = geom
    torch.manual_seed(D)
    T, page, pages = 37, 16, 40
    cos, sin = rotary_tables(10000.0, rot, 700) if rot else (None, None)
    if rot:
        cos, sin = cos.to(DEV), sin.to(DEV)
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=DEV).to(dtype)
    pos = torch.randint(0, 700, (T,), device=DEV, dtype=torch.int32)
    slots = (torch.randperm((pages - 1) * page, device=DEV)[:T] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, dtype)
    q_ref, kc_ref, vc_ref = qkv.clone(), kc.clone(), vc.clone()
    ref.ref_rotary_kv_store(q_ref, pos, cos, sin, rot, Hq, Hkv, D, kc_ref, vc_ref, slots)
    ops[dtype].rotary_kv_store(qkv, pos, cos, sin, rot, Hq, Hkv, D, kc, vc, slots)
    torch.testing.assert_close(qkv.float(), q_ref.float(), **tol(dtype))
    torch.testing.assert_close(kc.float(), kc_ref.float(), **tol(dtype))
    assert torch.equal(vc, vc_ref), "values are copied, not computed"
    assert torch.equal(kc[0], kc_ref[0]) and torch.equal(vc[0], vc_ref[0])


@pytest.mark.parametrize("geom", [(2, 1, 16), (3, 1, 32), (4, 2, 48), (32, 4, 64), (3, 3, 80), (5, 5, 96), (8, 2, 128), (2, 1, 256),
                                  (3, 1, 112), (2, 2, 192)])
@pytest.mark.parametrize("M", [1, 8, 16, 40])
def test_fused_projection_rotary_store(ops, geom, M):
    """Projection + rotary + cache write in one kernel against the three separate references."""
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D = geom
    o = ops[torch.bfloat16]
    torch.manual_seed(D + M)
    K, page, pages = 136, 16, 12
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 300))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    pos = torch.randint(0, 300, (M,), device=DEV, dtype=torch.int32)
    slots = (torch.randperm((pages - 1) * page, device=DEV)[:M] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.bfloat16)
    kc_ref, vc_ref = kc.float(), vc.float()
    qkv_ref = ref.ref_linear(x, w, None, torch.float32)
    ref.ref_rotary_kv_store(qkv_ref, pos, cos, sin, D, Hq, Hkv, D, kc_ref, vc_ref, slots)
    out = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, slots)
    assert tuple(out.shape) == (M, Hq * D), "the fused kernel returns q alone"
    torch.testing.assert_close(out.float(), qkv_ref[:, :Hq * D], atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(kc.float(), kc_ref, atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(vc.float(), vc_ref, atol=2e-2, rtol=1e-2)
    assert torch.equal(kc[0].float(), kc_ref[0]) and torch.equal(vc[0].float(), vc_ref[0]), "untouched pages stay untouched"
    # rotary over a part of the head is not fused: separate kernels, the whole projection comes back
    if D == 32:
        cos16, sin16 = (t.to(DEV) for t in rotary_tables(10000.0, 16, 300))
        kc2, vc2 = make_cache(pages, Hkv, page, D, torch.bfloat16)
        kr, vr = kc2.float(), vc2.float()
        full = o.linear_rotary_kv_store(x, w, pos, cos16, sin16, 16, Hq, Hkv, D, kc2, vc2, slots)
        assert full.shape[1] == (Hq + 2 * Hkv) * D
        q_ref = ref.ref_linear(x, w, None, torch.float32)
        ref.ref_rotary_kv_store(q_ref, pos, cos16, sin16, 16, Hq, Hkv, D, kr, vr, slots)
        torch.testing.assert_close(kc2.float(), kr, atol=2e-2, rtol=1e-2)
        torch.testing.assert_close(full.float()[:, :Hq * D], q_ref[:, :Hq * D], atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("geom", [(2, 1, 16), (3, 3, 80), (5, 1, 112), (32, 4, 64), (2, 2, 256)])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17])
def test_float32_projection_rotary_store(ops, geom, M):
    """The float32 product that rotates and writes to the cache by itself (up to 16 rows) against the product and the
    rotary kernel in turn: the same sums, rotated with the same expression, so the same bits (17 rows: two kernels)."""
    from mini_inference_engine_amd.kernels.api import KernelBackend
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D = geom
    o = ops[torch.float32]
    torch.manual_seed(D + M)
    K, page, pages = 136, 16, 12
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 300))
    x = torch.randn(M, K, device=DEV)
    w = torch.randn((Hq + 2 * Hkv) * D, K, device=DEV) / math.sqrt(K)
    pos = torch.randint(0, 300, (M,), device=DEV, dtype=torch.int32)
    slots = (torch.randperm((pages - 1) * page, device=DEV)[:M] + page).to(torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.float32)
    kc2, vc2 = kc.clone(), vc.clone()
    want = KernelBackend.linear_rotary_kv_store(o, x, w, pos, cos, sin, D, Hq, Hkv, D, kc2, vc2, slots)
    out = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, slots)
    assert (out.shape[1] == Hq * D) == (M <= 16), "one kernel for up to 16 rows, which returns q alone"
    assert torch.equal(out[:, :Hq * D], want[:, :Hq * D]) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.parametrize("M", [5, 17])
def test_float32_projection_rotary_store_refuses_strided_weights(ops, M):
    """A weight matrix whose rows are not contiguous (or x so) is refused with any number of rows, and nothing is written."""
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D, K, page, pages = 2, 1, 16, 64, 16, 4
    o = ops[torch.float32]
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, 30))
    wide, x2 = torch.randn((Hq + 2 * Hkv) * D, 2 * K, device=DEV), torch.randn(M, 2 * K, device=DEV)
    pos = torch.arange(M, device=DEV, dtype=torch.int32)
    kc, vc = make_cache(pages, Hkv, page, D, torch.float32)
    kept = kc.clone()
    for x, w in ((x2[:, :K], wide[:, ::2]), (x2[:, ::2], wide[:, :K])):
        with pytest.raises(ValueError, match="unit inner stride"):
            o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc, vc, pos + page)
    assert torch.equal(kc, kept)


def test_rotary_q_only(ops):
    from mini_inference_engine_amd.parts.rope import rotary_tables
    cos, sin = (t.to(DEV) for t in rotary_tables(500000.0, 32, 100))
    q = torch.randn(11, 3 * 32, device=DEV)
    pos = torch.arange(11, device=DEV, dtype=torch.int32) * 9
    expect = q.clone()
    ref.ref_rotary_kv_store(expect, pos, cos, sin, 32, 3, 0, 32, None, None, None)
    ops[torch.float32].rotary_kv_store(q, pos, cos, sin, 32, 3, 0, 32, None, None, None)
    torch.testing.assert_close(q, expect, atol=1e-6, rtol=1e-5)


# ------------------------------------------------------------------ attention
def paged_setup(ctx_lens, q_lens, Hq, Hkv, D, page, dtype, num_pages=None, seed=0, spike=None):
    """Rows with ctx_lens[i] keys of which the last q_lens[i] are this step's tokens.  Pages are a
    random permutation (page 0 never used); unused block-table entries are 0.
    spike = (row, key): that key's k is made to dominate the row's last query."""
    g = torch.Generator(device="cpu").manual_seed(seed)
    rows = len(ctx_lens)
    need = sum(-(-c // page) for c in ctx_lens)
    num_pages = num_pages or need + 5
    kc = torch.randn(num_pages, Hkv, page, D, generator=g).to(dtype)
    vc = torch.randn(num_pages, Hkv, D, page, generator=g).to(dtype)
    perm = torch.randperm(num_pages - 1, generator=g) + 1
    max_blocks = max(-(-c // page) for c in ctx_lens) + 2
    bt = torch.zeros(rows, max_blocks, dtype=torch.int32)
    i = 0
    for r, c in enumerate(ctx_lens):
        n = -(-c // page)
        bt[r, :n] = perm[i:i + n]
        i += n
    T = sum(q_lens)
    q = torch.randn(T, Hq * D, generator=g).to(dtype)
    token_row = torch.repeat_interleave(torch.arange(rows), torch.tensor(q_lens)).to(torch.int32)
    positions = torch.cat([torch.arange(c - n, c) for c, n in zip(ctx_lens, q_lens)]).to(torch.int32)
    if spike is not None:
        r, key = spike
        t_last = sum(q_lens[:r + 1]) - 1
        pg, off = int(bt[r, key // page]), key % page
        direction = torch.randn(D, generator=g)
        direction = direction / direction.norm()
        kc[pg, :, off, :] = (direction * 6.0).to(dtype)
        q[t_last] = (direction * 6.0).repeat(Hq).to(dtype)
    nd = 0
    while nd < rows and q_lens[nd] == 1:
        nd += 1
    assert all(n > 1 for n in q_lens[nd:]), "single-token rows lead the batch"
    row_start = torch.tensor([0] + list(torch.tensor(q_lens).cumsum(0)), dtype=torch.int32)
    row_position = torch.tensor([c - n for c, n in zip(ctx_lens, q_lens)], dtype=torch.int32)
    step = SimpleNamespace(token_row=token_row.to(DEV), positions=positions.to(DEV), num_rows=rows,
                           max_context=max(ctx_lens), num_tokens=T, num_decode_rows=nd,
                           max_row_tokens=max(q_lens), row_start=row_start.to(DEV),
                           row_position=row_position.to(DEV))
    group = SimpleNamespace(block_tables=bt.to(DEV), max_blocks=max_blocks)
    return q.to(DEV), kc.to(DEV), vc.to(DEV), group, step


def run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, scale, window, **kw):
    out = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, scale, window, **kw)
    expect = ref.ref_paged_attention(q, Hq, Hkv, D, kc, vc, group.block_tables, step.token_row, step.positions,
                                     scale, window, torch.float64)
    return out, expect


ATT_TOL = {torch.float32: dict(atol=3e-6, rtol=1e-5), torch.bfloat16: dict(atol=2e-2, rtol=2e-2)}
# The spiked set-ups have unscaled scores up to 36 (|q| = |k| = 6, scale 1): a float32 score then carries an
# absolute rounding error of about 36 * 2^-23 * sqrt(64 terms) = 3e-5, which passes through exp() as a relative
# error of the probabilities.  Their float32 bound follows from that, not from the unit-scale bound above.
SPIKE_TOL = {torch.float32: dict(atol=4e-5, rtol=1e-4), torch.bfloat16: dict(atol=2e-2, rtol=2e-2)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ctx", [[1], [17], [1000], [2048], [5, 300, 1, 2047, 64, 65], list(range(1, 200, 7))])
def test_decode_attention_reference_vectors(ops, dtype, ctx):
    Hq, Hkv, D, page = 32, 4, 64, 16
    q, kc, vc, group, step = paged_setup(ctx, [1] * len(ctx), Hq, Hkv, D, page, dtype, num_pages=4096)
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1 / math.sqrt(D), None)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])


@pytest.mark.parametrize("splits", [None, 1, 3, 8])
@pytest.mark.parametrize("ctx", [[1], [17], [1000], [2048], [5, 300, 1, 2047, 64, 65], list(range(1, 200, 7))])
def test_decode_attention_split_count_and_static_bound(ops, ctx, splits):
    """The matrix-core decode kernel: any split count, and a looser bound on the context (as under
    graph capture, where the bound is static), give the same answer
    (the reference tests the same: tests/test_kernels.py:54-59 there)."""
    Hq, Hkv, D, page = 32, 4, 64, 16
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup(ctx, [1] * len(ctx), Hq, Hkv, D, page, dtype, num_pages=4096, seed=len(ctx))
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1 / math.sqrt(D), None, num_splits=splits)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])
    generic = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 1 / math.sqrt(D), None, force_generic=True)
    torch.testing.assert_close(out.float(), generic.float(), **ATT_TOL[dtype])
    step.max_context = 2048
    extra = max(0, 2048 // page + 1 - group.block_tables.shape[1])
    group.block_tables = torch.nn.functional.pad(group.block_tables, (0, extra)).contiguous()
    out2 = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 1 / math.sqrt(D), None, num_splits=splits)
    torch.testing.assert_close(out2.double(), expect, **ATT_TOL[dtype])


@pytest.mark.parametrize("form", ["plain", "sink", "kept", "chunk", "biased"])
@pytest.mark.parametrize("geom", [(32, 4, 64, 16), (8, 1, 128, 16), (4, 4, 256, 16), (2, 1, 48, 32)])
def test_decode_attention_weights_below_the_smallest_normal_number(ops, geom, form):
    """A key whose weight is e^-90 = 8.2e-40 beside keys of weight 1 (one, and one a block) without values: its value of 2^100 times
    the weight comes out, within half a unit of the weight's bfloat16 (2^-134 of 8.2e-40: 5.6 %).  It stands in the block
    of the largest score, and in an earlier one of the same wave (up to sixteen a workgroup, 32 keys each in turn), whose sums are
    rescaled by e^-90."""
    Hq, Hkv, D, page = geom
    dtype = torch.bfloat16
    n = 600
    q, kc, vc, group, step = paged_setup([n], [1], Hq, Hkv, D, page, dtype, seed=D)
    q.zero_()
    q.view(1, Hq, D)[:, :, 0] = 1.0
    window, kw = None, {}
    if form == "sink":
        kw = dict(sink=-100.0)
    if form == "kept":
        window, kw = n - 4, dict(keep_first=4)
    if form == "chunk":
        kw = dict(chunk=640)
    if form == "biased":
        kw = dict(distance_bias=torch.zeros(Hq, 30, device=DEV))
    for small, ones in ((3, (9,)), (3, (515,)), (100, (20, 130))):
        kc.zero_()
        vc.zero_()
        kc[..., 0] = -1000.0                             # the other keys: weights of e^-1000
        for key, score, value in ((small, -90.0, 2.0 ** 100), *((k, 0.0, 0.0) for k in ones)):
            pg, off = int(group.block_tables[0, key // page]), key % page
            kc[pg, :, off, 0] = score
            vc[pg, :, :, off] = value
        out = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 1.0, window, num_splits=1, **kw)
        want = math.exp(-90.0) * 2.0 ** 100 / len(ones)
        assert bool(((out.double() / want - 1).abs() <= 0.056 + 2.0 ** -8).all()), (small, ones, float(out.double().min()), float(out.double().max()), want)


LONG_DECODE = [  # (Hq, Hkv, D), contexts
    ((32, 4, 64), [4096]), ((32, 4, 64), [8192]), ((32, 8, 128), [8192]), ((32, 32, 128), [4096]),
    ((32, 8, 128), [8191, 5, 4097, 300, 6000, 64, 1, 2048]),
    ((32, 8, 128), [8192] + [40 + 3 * i for i in range(63)]),        # 64 rows: rows x kv heads fill the GPU, no split
]


@pytest.mark.parametrize("spiked", [False, True], ids=["random", "far key"])
@pytest.mark.parametrize("splits", [None, 1, 64])
@pytest.mark.parametrize("case", LONG_DECODE, ids=[f"{g[0]}on{g[1]}x{g[2]}-{len(c)}rows-{max(c)}" for g, c in LONG_DECODE])
def test_decode_attention_past_4096_keys(ops, case, splits, spiked):
    """Contexts of 4,096 and 8,192 keys (block tables of 256 and 512 pages) at the head sizes and groupings of the
    benchmark configurations: with the split the engine chooses (up to 64 partial results a head for one row,
    none for 64 rows), unsplit, and split 64 ways; with random keys, and with one key among the first 64 made to
    dominate the longest row's query, 8,000 keys away."""
    (Hq, Hkv, D), ctx = case
    dtype = torch.bfloat16
    spike = (0, 37) if spiked else None
    q, kc, vc, group, step = paged_setup(ctx, [1] * len(ctx), Hq, Hkv, D, 16, dtype, seed=len(ctx) + D, spike=spike)
    scale = 1.0 if spiked else 1 / math.sqrt(D)
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, scale, None, num_splits=splits)
    torch.testing.assert_close(out.double(), expect, **(SPIKE_TOL if spiked else ATT_TOL)[dtype])
    if spiked:          # the far key's value is what comes out
        pg = int(group.block_tables[0, 37 // 16])
        v_far = vc[pg, :, :, 37 % 16].float().repeat_interleave(Hq // Hkv, dim=0).reshape(-1)
        torch.testing.assert_close(out[0].float(), v_far, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("edge", [None, "first key inside", "last key outside"])
@pytest.mark.parametrize("window", [1024, 4000])
@pytest.mark.parametrize("geom", [(32, 8, 128), (32, 4, 64)])
def test_windowed_attention_at_long_contexts(ops, geom, window, edge):
    """A window of 1,024 or 4,000 keys at contexts of thousands, at the head sizes and groupings of the benchmark
    configurations (no registered architecture has a window: the part and the kernels do): single-token rows,
    where the context bound a kernel is given shrinks to the window, and a portion of 300 tokens behind 5,000
    earlier ones.  With ``edge``, the key just inside (or just outside) the window of the first row's last query
    is made to dominate it: inside, its value is what comes out; outside, it must leave no trace."""
    Hq, Hkv, D = geom
    dtype = torch.bfloat16
    for ctx, qn in (([6000, 700, 4096, 1025, 1024, 33], [1] * 6), ([5300, 2100], [300, 40])):
        spike = None
        if edge is not None:
            last = ctx[0] - 1                                        # position of the first row's last query
            key = last - window + 1 if edge == "first key inside" else last - window
            spike = (0, key)
        q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, 16, dtype, seed=D + window + len(ctx), spike=spike)
        scale = 1 / math.sqrt(D) if edge is None else 1.0
        out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, scale, window)
        torch.testing.assert_close(out.double(), expect, **(ATT_TOL if edge is None else SPIKE_TOL)[dtype])
        if edge is not None:
            t_last = qn[0] - 1
            pg = int(group.block_tables[0, spike[1] // 16])
            v_key = vc[pg, :, :, spike[1] % 16].float().repeat_interleave(Hq // Hkv, dim=0).reshape(-1)
            gap = (out[t_last].float() - v_key).abs().max()
            if edge == "first key inside":
                assert float(gap) < 3e-2, f"the key at the window's edge should dominate (off by {float(gap):.2e})"
            else:
                assert float(gap) > 0.5, "a key one past the window was seen"


@pytest.mark.parametrize("key", [None, 5, 6143, 6144, 8100])
@pytest.mark.parametrize("geom", [(32, 8, 128), (32, 4, 64)])
def test_prefill_attention_with_6144_earlier_tokens(ops, geom, key):
    """A portion of 2,048 tokens behind 6,144 earlier ones (and a short portion behind 6,144 beside it): the walk
    over a block table of 512 pages, 128 blocks of 64 keys a query tile.  A sample of the queries against the
    token-by-token reference; with ``key``, that key is made to dominate the last query."""
    Hq, Hkv, D = geom
    dtype = torch.bfloat16
    ctx, qn = [8192, 6200], [2048, 56]
    q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, 16, dtype, seed=D + (key or 0),
                                         spike=None if key is None else (0, key))
    scale = 1 / math.sqrt(D) if key is None else 1.0
    out = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, scale, None)
    idx = torch.tensor([0, 1, 15, 16, 31, 32, 63, 64, 65, 1000, 1023, 1024, 2046, 2047, 2048, 2049, 2103], device=DEV)
    expect = ref.ref_paged_attention(q[idx], Hq, Hkv, D, kc, vc, group.block_tables, step.token_row[idx],
                                     step.positions[idx], scale, None, torch.float64)
    torch.testing.assert_close(out[idx].double(), expect, **(ATT_TOL if key is None else SPIKE_TOL)[dtype])
    assert bool(torch.isfinite(out.float()).all())


@pytest.mark.parametrize("D", [112, 192])
def test_head_sizes_outside_the_prebuilt_list(ops, D):
    """Head sizes that are a multiple of 16 but not in kernels/variants.py: the attention modules for them are
    compiled at first use (unless an earlier run left them built) and must give what the others give: decode
    attention split and unsplit, prefill attention behind earlier portions and with a window, a far key, against
    the references.  (The projection kernels take the head size at run time: 112 and 192 are among the geometries
    of test_fused_projection_rotary_store and test_decode_attention_finishes_the_projection.)"""
    from mini_inference_engine_amd.kernels.variants import HEAD_DIMS
    assert D not in HEAD_DIMS and D % 16 == 0
    dtype = torch.bfloat16
    Hq, Hkv, page = 6, 2, 16
    for splits in (None, 1, 5):
        q, kc, vc, group, step = paged_setup([1, 17, 700, 64, 65, 1500], [1] * 6, Hq, Hkv, D, page, dtype, seed=D)
        out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1 / math.sqrt(D), None,
                                    num_splits=splits)
        torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])
    for window in (None, 24):
        q, kc, vc, group, step = paged_setup([9, 300, 2, 64, 65, 200, 1000], [1, 1, 2, 64, 65, 3, 489], Hq, Hkv, D, page,
                                             dtype, seed=D + 1)
        out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.1 / math.sqrt(D), window)
        torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])
    q, kc, vc, group, step = paged_setup([600], [600], Hq, Hkv, D, page, dtype, seed=D + 2, spike=(0, 3))
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.0, None)
    torch.testing.assert_close(out.double(), expect, **SPIKE_TOL[dtype])


@pytest.mark.parametrize("geom", [(32, 4, 64, 16, 64), (8, 8, 128, 16, 40), (6, 2, 32, 32, 130), (16, 1, 16, 16, 257),
                                  (10, 5, 48, 16, 52), (4, 4, 256, 16, 64), (16, 8, 64, 16, 64), (4, 4, 32, 16, 150),
                                  (4, 2, 112, 16, 130), (4, 4, 192, 16, 64)])
@pytest.mark.parametrize("window", [None, 40])
def test_decode_attention_finishes_the_projection(engine_ops, geom, window):
    """Steps of single-token rows whose rows x kv heads are 256 workgroups or more: the decode kernel takes the
    q/k/v projection's float32 sums (partial sums of the split product up to 128 rows, the library's sums above)
    and does rotary, cache write and attention itself.  Against the same step done by the kernels that are each
    checked against their references elsewhere: sum + rotary + cache write, then attention over the cache.
    Contexts of 1 key, around the kernel's first blocks (which it asks for before the new key is written),
    at page edges, and long ones; fewer and more workgroups than those up to which one is eight waves."""
    from mini_inference_engine_amd.kernels.hip_backend import ProjectionSums
    from mini_inference_engine_amd.parts.rope import rotary_tables
    Hq, Hkv, D, page, M = geom
    o = engine_ops
    assert M * Hkv >= o.DECODE_WHOLE_WORKGROUPS
    ctx = [1, 2, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 255, 256, 257, 300, 1000, 48]
    ctx = (ctx * (M // len(ctx) + 1))[:M]
    K = 1032 if window else 264          # four splits of K or one (where the product splits at all)
    torch.manual_seed(D + M)
    _, kc, vc, group, step = paged_setup(ctx, [1] * M, Hq, Hkv, D, page, torch.bfloat16, seed=D + Hkv)
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, max(ctx) + 1))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    pos = step.positions
    bt = group.block_tables
    slots = (bt[torch.arange(M, device=DEV), (pos // page).long()] * page + pos % page).to(torch.int32)
    group.slot_mapping = slots
    scale = 0.9 / math.sqrt(D)

    kc1, vc1 = kc.clone(), vc.clone()
    pending = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc1, vc1, slots, for_attention=True)
    assert isinstance(pending, ProjectionSums), "this many rows must leave the projection unfinished"
    assert torch.equal(kc1, kc) and torch.equal(vc1, vc), "nothing is written before the attention runs"
    out1 = o.paged_attention(pending, Hq, Hkv, D, kc1, vc1, group, step, scale, window)

    kc2, vc2 = kc.clone(), vc.clone()
    q2 = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc2, vc2, slots)
    assert torch.is_tensor(q2)
    out2 = o.paged_attention(q2, Hq, Hkv, D, kc2, vc2, group, step, scale, window)
    # the same sums in the same order, the same expressions: the new keys and values are the same numbers
    assert torch.equal(vc1, vc2), f"{int((vc1 != vc2).sum())} values differ, by up to {float((vc1.float() - vc2.float()).abs().max())}"
    assert torch.equal(kc1, kc2), f"{int((kc1 != kc2).sum())} keys differ, by up to {float((kc1.float() - kc2.float()).abs().max())}"
    assert not torch.equal(kc1, kc), "the step's keys were written"
    torch.testing.assert_close(out1.float(), out2.float(), atol=2e-3, rtol=2e-3)
    # and against the exact attention over that cache
    expect = ref.ref_paged_attention(q2, Hq, Hkv, D, kc2, vc2, bt, step.token_row, pos, scale, window, torch.float64)
    torch.testing.assert_close(out1.double(), expect, **ATT_TOL[torch.bfloat16])
    # a projection that was made for other positions or slots than the step's is finished in a kernel of its own
    # (with its own positions and slots), not by the attention kernel (which would use the step's)
    kc4, vc4 = kc.clone(), vc.clone()
    pending = o.linear_rotary_kv_store(x, w, pos.clone(), cos, sin, D, Hq, Hkv, D, kc4, vc4, slots, for_attention=True)
    assert o._decode_attention_from_sums(pending, Hq, Hkv, D, kc4, vc4, group, step, scale, window, False) is None
    pending = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc4, vc4, slots.clone(), for_attention=True)
    assert o._decode_attention_from_sums(pending, Hq, Hkv, D, kc4, vc4, group, step, scale, window, False) is None
    assert torch.equal(kc4, kc), "a refused step writes nothing"
    # a step that is not of this kind finishes the projection in a kernel of its own
    kc3, vc3 = kc.clone(), vc.clone()
    pending = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, kc3, vc3, slots, for_attention=True)
    out3 = o.paged_attention(pending, Hq, Hkv, D, kc3, vc3, group, step, scale, window, num_splits=2)
    assert torch.equal(kc3, kc2) and torch.equal(vc3, vc2)
    torch.testing.assert_close(out3.double(), expect, **ATT_TOL[torch.bfloat16])


@pytest.mark.parametrize("geom", [(4, 2, 16, 16), (3, 1, 32, 16), (5, 5, 48, 16), (40, 2, 80, 32), (8, 1, 128, 64),
                                  (2, 2, 256, 16), (12, 4, 96, 48), (17, 1, 64, 16)])
@pytest.mark.parametrize("window", [None, 40])
def test_decode_attention_geometries(ops, geom, window):
    """Other head sizes (steps of 16), groups beyond 16 heads, odd counts, page sizes, a window."""
    Hq, Hkv, D, page = geom
    ctx = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 500, 96]
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup(ctx, [1] * len(ctx), Hq, Hkv, D, page, dtype, seed=D + Hq)
    for splits in (None, 1, 4):
        out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 0.9 / math.sqrt(D), window,
                                    num_splits=splits)
        torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])


def test_decode_attention_ignores_stale_pages_bf16(ops):
    Hq, Hkv, D, page = 8, 2, 64, 16
    ctx = [37, 5, 64, 1, 130, 33]
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup(ctx, [1] * len(ctx), Hq, Hkv, D, page, dtype, seed=4)
    owned = torch.zeros(kc.shape[0], page, dtype=torch.bool, device=DEV)
    for r, c in enumerate(ctx):
        for p in range(c):
            owned[int(group.block_tables[r, p // page]), p % page] = True
    kc2, vc2 = kc.clone(), vc.clone()
    kc2.permute(0, 2, 1, 3)[~owned] = float("nan")
    vc2.permute(0, 3, 1, 2)[~owned] = float("nan")
    for splits in (1, 2):
        clean = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.2, None, num_splits=splits)
        dirty = ops[dtype].paged_attention(q, Hq, Hkv, D, kc2, vc2, group, step, 0.2, None, num_splits=splits)
        assert torch.equal(clean, dirty)
    for window in (3, 20):
        clean = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.2, window)
        lo_owned = owned.clone()
        for r, c in enumerate(ctx):
            for p in range(max(0, c - window)):
                lo_owned[int(group.block_tables[r, p // page]), p % page] = False
        kc3, vc3 = kc.clone(), vc.clone()
        kc3.permute(0, 2, 1, 3)[~lo_owned] = float("nan")
        vc3.permute(0, 3, 1, 2)[~lo_owned] = float("nan")
        dirty = ops[dtype].paged_attention(q, Hq, Hkv, D, kc3, vc3, group, step, 0.2, window)
        assert torch.equal(clean, dirty)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("geom", [(4, 2, 16, 16), (3, 1, 32, 16), (5, 5, 48, 16), (6, 2, 80, 32), (8, 1, 128, 64),
                                  (2, 2, 256, 16), (12, 4, 96, 16)])
def test_attention_mixed_rows(ops, dtype, geom):
    """Single tokens beside portions that start anywhere, other head sizes, groups and page sizes."""
    Hq, Hkv, D, page = geom
    ctx = [40, 1, 16, 17, 130, 64, 33, 2]
    qn = [1, 1, 1, 1, 50, 64, 2, 2]
    q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, page, dtype, seed=D)
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 0.7 / math.sqrt(D), None)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])


# single tokens' contexts; portions (tokens, tokens before them); heads; window; sink: one and many single tokens, contexts of one key, of whole
# and broken blocks and pages, contexts cut at 2,048 keys, every grid of the portions, groups of more than 16 heads, as many workgroups as
# compute units, and one single token more (two kernels)
@pytest.mark.parametrize("case", [([1], [(2, 0)], (4, 1), 0, None), ([700, 64, 3], [(33, 0), (150, 77)], (32, 4), 0, None), ([900] * 32, [(701, 0), (399, 0)], (32, 4), 0, None),
                                  ([2500, 31], [(65, 9)], (32, 4), 0, 0.7), ([4200], [(40, 300)], (8, 8), 0, None), ([2500, 800, 17], [(130, 1500)], (16, 4), 256, None),
                                  ([333, 5000], [(70, 0), (2, 4000)], (40, 2), 1000, -0.5), ([50] * 64, [(1300, 0), (1290, 3)], (32, 4), 0, None),
                                  ([50] * 65, [(40, 0)], (32, 4), 0, None)])
@pytest.mark.parametrize("page", [16, 48])
def test_attention_of_singles_beside_portions(ops, case, page):
    """A step's single tokens and portions in one launch (head size 64): against 64 bits at the bound of the kernels alone, the single
    tokens as near to their own kernel's, and no key that is not a request's reaches a result."""
    contexts, portions, (Hq, Hkv), window, sink = case
    o, D, n = ops[torch.bfloat16], 64, len(contexts)
    ctx, new = contexts + [a + b for a, b in portions], [1] * n + [a for a, _ in portions]
    q, kc, vc, group, step = paged_setup(ctx, new, Hq, Hkv, D, page, torch.bfloat16, seed=n + len(portions))
    used = torch.zeros(kc.shape[0], dtype=torch.bool, device=DEV)
    for r, c in enumerate(ctx):
        pages = group.block_tables[r, :-(-c // page)].long()
        used[pages] = True
        if c % page:                            # behind a request's last key: numbers that must not reach a sum
            kc[pages[-1], :, c % page:] = vc[pages[-1], :, :, c % page:] = float("nan")
    kc[~used] = vc[~used] = float("nan")
    fused = n * Hkv * -(-(Hq // Hkv) // 16) <= 256
    with counted(o, "prefill_attention_bf16", "mie_step_attention", defines=("-DHEAD_DIM=64",)) as calls:
        out = o.paged_attention(q, Hq, Hkv, D, kc, vc, group, step, D ** -0.5, window or None, sink=sink)
    assert len(calls) == (1 if fused else 0)
    plain_k, plain_v = kc.nan_to_num(0.0), vc.nan_to_num(0.0)
    expect = ref.ref_paged_attention(q, Hq, Hkv, D, plain_k, plain_v, group.block_tables, step.token_row, step.positions, D ** -0.5, window or None,
                                     torch.float64, **({} if sink is None else {"sink": sink}))
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[torch.bfloat16])
    # the same by two kernels: the single tokens alone, then the portions
    one = SimpleNamespace(token_row=step.token_row[:n], positions=step.positions[:n], num_rows=n, max_context=max(contexts), num_tokens=n, num_decode_rows=n,
                          max_row_tokens=1, row_start=None, row_position=None)
    alone = o.paged_attention(q[:n], Hq, Hkv, D, kc, vc, group, one, D ** -0.5, window or None, sink=sink)
    # on either side the weights, their sum's share in them and the result are rounded to bfloat16, 2^-9 of sum p |v| each at most; one
    # more for the float32 sums of scores and weights
    weighed = ref.ref_paged_attention(q[:n], Hq, Hkv, D, plain_k, plain_v.abs(), group.block_tables, step.token_row[:n], step.positions[:n], D ** -0.5,
                                      window or None, torch.float64, **({} if sink is None else {"sink": sink}))
    assert bool(((alone.double() - out[:n].double()).abs() <= 7 * 2.0 ** -9 * weighed).all())


@pytest.mark.parametrize("key", [0, 31, 2047, 2048, 4095, 4096, 4490, 4499])
def test_attention_of_singles_beside_portions_finds_a_far_key(ops, key):
    """One key among 4,500 dominates a single token beside a portion, whose context is cut into three parts of 2,048 keys: a part that is
    dropped or joined wrongly shows."""
    o, Hq, Hkv, D, page = ops[torch.bfloat16], 8, 2, 64, 16
    q, kc, vc, group, step = paged_setup([4500, 700], [1, 130], Hq, Hkv, D, page, torch.bfloat16, seed=key, spike=(0, key))
    with counted(o, "prefill_attention_bf16", "mie_step_attention", defines=("-DHEAD_DIM=64",)) as calls:
        out, expect = run_attention(ops, torch.bfloat16, q, kc, vc, group, step, Hq, Hkv, D, 1.0, None)
    partition, splits = o.decode_splits(1, Hq, Hkv, 4500, None, o.lib("attention_bf16", ("-DHEAD_DIM=64",)).mie_decode_block_keys(), D)
    assert len(calls) == 1 and splits > 1 and partition <= o.STEP_SPLIT_KEYS == 2048, "one launch, parts of 2,048 keys"
    pg, off = int(group.block_tables[0, key // page]), key % page
    v_key = vc[pg, :, :, off].double().repeat_interleave(Hq // Hkv, 0).reshape(-1)
    assert (expect[0] - v_key).abs().max() < 5e-3, "the set-up must make that key dominate"
    torch.testing.assert_close(out.double(), expect, **SPIKE_TOL[torch.bfloat16])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("key", [0, 15, 16, 31, 255, 256, 700, 1022])
def test_attention_finds_a_far_key(ops, dtype, key):
    """One key among a thousand dominates: the output must be (nearly) that key's value, so a
    kernel that skips a page edge, the first key or a split's last key fails by a wide margin."""
    Hq, Hkv, D, page = 8, 2, 64, 16
    ctx = [1023, 300]
    q, kc, vc, group, step = paged_setup(ctx, [1, 1], Hq, Hkv, D, page, dtype, seed=key, spike=(0, key))
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.0, None)
    pg, off = int(group.block_tables[0, key // page]), key % page
    v_key = vc[pg, :, :, off].double().repeat_interleave(Hq // Hkv, 0).reshape(-1)
    assert (expect[0] - v_key).abs().max() < 1e-3, "the set-up must make that key dominate"
    torch.testing.assert_close(out.double(), expect, **SPIKE_TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("window", [1, 5, 16, 17, 100])
def test_attention_window_edge(ops, dtype, window):
    """The key just outside the window dominates if it is (wrongly) seen; the one just inside must be."""
    Hq, Hkv, D, page = 4, 2, 32, 16
    ctx, qn = [200, 90], [1, 30]
    for inside in (True, False):
        key = 199 - window + 1 if inside else 199 - window
        if key < 0:
            continue
        q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, page, dtype, seed=window, spike=(0, key))
        out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.0, window)
        torch.testing.assert_close(out.double(), expect, **SPIKE_TOL[dtype])


@pytest.mark.parametrize("key", [0, 15, 16, 31, 32, 63, 64, 127, 128, 569, 570, 571, 575, 576, 698, 699])
def test_prefill_attention_finds_a_far_key(ops, key):
    """The same inside a row of many tokens, which the matrix-core prefill kernel computes: a portion that
    starts in the middle of a page (position 570), keys at page and 64-key block edges, the first key of the
    request, the portion's own first keys, the last query's own key.  Beside it a two-token row."""
    Hq, Hkv, D, page = 8, 2, 64, 16
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup([700, 41], [130, 2], Hq, Hkv, D, page, dtype, seed=key, spike=(0, key))
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.0, None)
    pg, off = int(group.block_tables[0, key // page]), key % page
    v_key = vc[pg, :, :, off].double().repeat_interleave(Hq // Hkv, 0).reshape(-1)
    # (a property of the set-up, not of the kernel: the exact result is that key's value up to the other keys' share)
    assert (expect[129] - v_key).abs().max() < 5e-3, "the set-up must make that key dominate the row's last query"
    torch.testing.assert_close(out.double(), expect, **SPIKE_TOL[dtype])


@pytest.mark.parametrize("window", [1, 5, 16, 17, 64, 65, 100])
def test_prefill_attention_window_edge(ops, window):
    """A many-token row with a window: the key just inside the last query's window must be seen, the one just
    outside must not (it dominates if it is)."""
    Hq, Hkv, D, page = 4, 2, 32, 16
    dtype = torch.bfloat16
    for inside in (True, False):
        key = 299 - window + 1 if inside else 299 - window
        q, kc, vc, group, step = paged_setup([300, 9], [75, 2], Hq, Hkv, D, page, dtype, seed=window, spike=(0, key))
        out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.0, window)
        torch.testing.assert_close(out.double(), expect, **SPIKE_TOL[dtype])


@pytest.mark.parametrize("geom", [(4, 2, 16, 16), (3, 1, 32, 16), (5, 5, 48, 16), (6, 2, 80, 32), (8, 1, 128, 64),
                                  (2, 2, 256, 16), (12, 4, 96, 16), (32, 4, 64, 16), (8, 8, 128, 16),
                                  (20, 2, 64, 16), (16, 1, 256, 32), (6, 2, 64, 48), (5, 1, 32, 48)])
@pytest.mark.parametrize("window", [None, 24])
def test_prefill_attention_geometries(ops, geom, window):
    """The matrix-core prefill kernel: portions that start anywhere (page edges, mid page), tails that
    do not fill a tile, two-token rows, every head-size step, beside single-token rows."""
    Hq, Hkv, D, page = geom
    ctx = [9, 300, 2, 64, 65, 17, 200, 131, 48, 1000]
    qn = [1, 1, 2, 64, 65, 17, 3, 100, 31, 489]
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, page, dtype, seed=D * 3 + Hq)
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.1 / math.sqrt(D), window)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])
    generic = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 1.1 / math.sqrt(D), window,
                                         force_generic=True)
    torch.testing.assert_close(out.float(), generic.float(), **ATT_TOL[dtype])


@pytest.mark.parametrize("geom", [(32, 32, 16, 16), (32, 32, 128, 16), (64, 8, 64, 32)])
def test_prefill_attention_many_workgroups(ops, geom):
    """Rows and heads enough for the kernel's other way of spending eight waves (over twice the queries of a
    workgroup instead of over two halves of the keys): the launcher picks it from the size of the grid."""
    Hq, Hkv, D, page = geom
    ctx = [700, 600, 650, 603]
    qn = [600, 600, 600, 603]
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, page, dtype, seed=D + Hkv)
    out, expect = run_attention(ops, dtype, q, kc, vc, group, step, Hq, Hkv, D, 1.1 / math.sqrt(D), None)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[dtype])


def test_prefill_attention_ignores_stale_pages_bf16(ops):
    Hq, Hkv, D, page = 8, 2, 64, 16
    ctx, qn = [37, 5, 64, 130, 33], [30, 5, 2, 67, 33]
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, page, dtype, seed=4)
    owned = torch.zeros(kc.shape[0], page, dtype=torch.bool, device=DEV)
    for r, c in enumerate(ctx):
        for p in range(c):
            owned[int(group.block_tables[r, p // page]), p % page] = True
    kc2, vc2 = kc.clone(), vc.clone()
    kc2.permute(0, 2, 1, 3)[~owned] = float("nan")
    vc2.permute(0, 3, 1, 2)[~owned] = float("nan")
    clean = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.2, None)
    dirty = ops[dtype].paged_attention(q, Hq, Hkv, D, kc2, vc2, group, step, 0.2, None)
    assert torch.equal(clean, dirty)


# (heads, kv heads, head size, page, context, tokens of the step that are the row's own, with padding) and the kernel that each takes
PREFILL_KINDS = {
    "four waves, in pairs": (4, 4, 256, 16, 90, 35, 64), "four waves of size 128, two workgroups a compute unit": (32, 8, 128, 16, 1500, 1200, 1300),
    "four waves, pages of 48": (32, 32, 128, 48, 1300, 1100, 1200),
    "keys in halves": (8, 2, 64, 16, 170, 29, 48), "keys in halves, pages of 48": (32, 4, 64, 48, 600, 333, 512),
    "keys in halves, size 128": (16, 8, 128, 16, 1500, 1025, 1400), "keys in halves, in pairs": (128, 128, 64, 48, 450, 300, 400),
    "twice the queries": (96, 96, 80, 16, 640, 500, 512),
    "twice the queries, in pairs": (128, 128, 64, 16, 700, 600, 650), "twice the queries, in pairs, size 128": (128, 128, 128, 16, 700, 600, 650)}
PREFILL_KIND = {"four waves": 0, "four waves, in pairs": 3, "keys in halves": 2, "keys in halves, in pairs": 5, "twice the queries": 1,
                "twice the queries, in pairs": 4}
PREFILL_FORMS = ["plain", "window", "kept", "chunk", "sigmoid", "sigmoid chunk", "biased"]


def prefill_case(ops, name):
    """The geometry, after a look at whether its step takes the kernel that it is here for."""
    geom = PREFILL_KINDS[name]
    Hq, Hkv, D, _, _, _, padded = geom
    what = max((k for k in PREFILL_KIND if name.startswith(k)), key=len)
    lib = ops[torch.bfloat16].lib("prefill_attention_bf16", (f"-DHEAD_DIM={D}",))
    assert lib.mie_prefill_attention_kind(1, padded, Hq, Hkv) == PREFILL_KIND[what], name
    return geom


@pytest.mark.parametrize("form", PREFILL_FORMS)
@pytest.mark.parametrize("name", PREFILL_KINDS)
def test_prefill_attention_kinds(ops, name, form):
    """Every kernel that a portion can take, in every form, behind earlier keys: tokens at the edges of tiles and stretches and some
    between, against 64 bits.  Half an ulp of bfloat16 each for a weight, for what their rounding adds to the denominator and for the
    result is 3 * 2^-9 of a head's result in the 2-norm; 2^-7 allows for a token's values being few."""
    Hq, Hkv, D, page, n, real, padded = prefill_case(ops, name)
    n, real = n + padded - real, padded                # the whole length is the row's own
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup([n], [real], Hq, Hkv, D, page, dtype, seed=D + n)
    window, kw = {"window": (45, {}), "kept": (70, dict(keep_first=5)), "chunk": (None, dict(chunk=72)), "sigmoid": (None, dict(weights="sigmoid")),
                  "sigmoid chunk": (None, dict(weights="sigmoid", chunk=72)),
                  "biased": (None, dict(distance_bias=torch.randn(Hq, 200, device=DEV)))}.get(form, (None, {}))
    out = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 1.1 / math.sqrt(D), window, **kw)
    at = sorted({t for e in (0, 32, 64, 128, 256, real // 2, real) for t in (e - 1, e, e + 1) if 0 <= t < real} | set(range(7, real, real // 12)))
    want = ref.ref_paged_attention(q[at], Hq, Hkv, D, kc, vc, group.block_tables, step.token_row[at], step.positions[at], 1.1 / math.sqrt(D),
                                   window, torch.float64, **kw).view(len(at), Hq, D)
    error = (out[at].double().view(len(at), Hq, D) - want).norm(dim=-1) / want.norm(dim=-1)
    assert float(error.max()) <= 2.0 ** -7, (at[int(error.max(1).values.argmax())], float(error.max()))


# every kernel that a portion can take; (kept keys, window, chunk) of the forms that hide a row's first keys
@pytest.mark.parametrize("form", PREFILL_FORMS)
@pytest.mark.parametrize("geom", PREFILL_KINDS)
def test_prefill_attention_looks_at_no_slot_its_row_did_not_write(ops, geom, form):
    """A row lengthened with padding tokens, whose keys are not in its pages, with NaN in every slot the row did not write and in
    the pages whose keys lie before all its queries' first: its own tokens get the bits they get from a cache of zeros there."""
    Hq, Hkv, D, page, n, real, padded = prefill_case(ops, geom)
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup([n], [real], Hq, Hkv, D, page, dtype, seed=D + n)
    window, kw, first = None, {}, 0
    if form in ("window", "kept"):
        window, first = 21, n - real - 20
    if form == "kept":
        kw = dict(keep_first=5)
    if form.endswith("chunk"):
        kw, first = dict(chunk=40), (n - real) // 40 * 40
    if form.startswith("sigmoid"):
        kw["weights"] = "sigmoid"
    if form == "biased":
        kw = dict(distance_bias=torch.randn(Hq, 30, device=DEV))
    own = torch.zeros(kc.shape[0], page, dtype=torch.bool, device=DEV)
    for p in [*range(kw.get("keep_first", 0)), *range(first, n)]:
        own[int(group.block_tables[0, p // page]), p % page] = True
    more = padded - real
    longer = SimpleNamespace(token_row=torch.zeros(padded, dtype=torch.int32, device=DEV), num_rows=1, num_tokens=padded,
                             positions=torch.arange(n - real, n + more, dtype=torch.int32, device=DEV),
                             max_context=n + more, num_decode_rows=0, max_row_tokens=padded, row_position=step.row_position,
                             row_start=torch.tensor([0, padded], dtype=torch.int32, device=DEV),
                             row_written=torch.tensor([n], dtype=torch.int32, device=DEV))
    bt = torch.nn.functional.pad(group.block_tables, (0, more // page + 2))
    wide = SimpleNamespace(block_tables=bt, max_blocks=bt.shape[1])
    seen = []
    for fill in (0.0, float("nan")):
        kd, vd = kc.clone(), vc.clone()
        kd.permute(0, 2, 1, 3)[~own] = fill
        vd.permute(0, 3, 1, 2)[~own] = fill
        qd = torch.cat([q, torch.full_like(q[:1], fill).expand(more, -1)])
        seen.append(ops[dtype].paged_attention(qd, Hq, Hkv, D, kd, vd, wide, longer, 0.2, window, **kw)[:real])
    assert bool(torch.isfinite(seen[0]).all()) and torch.equal(seen[0], seen[1])


def test_prefill_last_row_equals_decode(ops):
    """The last token of a portion, computed by the prefill kernel, equals the same token computed as a
    single-token row by the decode kernel (same keys, same cache), within bfloat16 rounding."""
    Hq, Hkv, D, page = 8, 2, 64, 16
    dtype = torch.bfloat16
    q, kc, vc, group, step = paged_setup([150], [40], Hq, Hkv, D, page, dtype, seed=12)
    whole = ops[dtype].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.125, None)
    q1, _, _, g1, s1 = paged_setup([150], [1], Hq, Hkv, D, page, dtype, seed=12)
    g1.block_tables = group.block_tables
    last = ops[dtype].paged_attention(q[-1:].contiguous(), Hq, Hkv, D, kc, vc, g1, s1, 0.125, None)
    torch.testing.assert_close(whole[-1:].float(), last.float(), **ATT_TOL[dtype])


def test_attention_one_key_is_its_value(ops):
    q, kc, vc, group, step = paged_setup([1, 1, 1], [1, 1, 1], 6, 3, 48, 16, torch.float32, seed=9)
    out = ops[torch.float32].paged_attention(q, 6, 3, 48, kc, vc, group, step, 0.3, None)
    for r in range(3):
        v = vc[int(group.block_tables[r, 0]), :, :, 0].repeat_interleave(2, 0).reshape(-1)
        torch.testing.assert_close(out[r], v, atol=1e-6, rtol=1e-6)


def test_attention_ignores_stale_pages(ops):
    """NaN in every slot beyond a row's context, and in pages it does not own, changes nothing."""
    Hq, Hkv, D, page = 4, 2, 32, 16
    ctx, qn = [37, 5, 64], [1, 5, 20]
    q, kc, vc, group, step = paged_setup(ctx, qn, Hq, Hkv, D, page, torch.float32, seed=2)
    clean = ops[torch.float32].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.2, None)
    owned = torch.zeros(kc.shape[0], page, dtype=torch.bool, device=DEV)
    for r, c in enumerate(ctx):
        for p in range(c):
            owned[int(group.block_tables[r, p // page]), p % page] = True
    kc2, vc2 = kc.clone(), vc.clone()
    kc2.permute(0, 2, 1, 3)[~owned] = float("nan")
    vc2.permute(0, 3, 1, 2)[~owned] = float("nan")
    dirty = ops[torch.float32].paged_attention(q, Hq, Hkv, D, kc2, vc2, group, step, 0.2, None)
    assert torch.equal(clean, dirty)


# heads, kv heads, head size, page: groups that fill 16 queries, leave some of them empty, and take several tiles
@pytest.mark.parametrize("window", [None, 1, 100, 128, 300])
@pytest.mark.parametrize("geom", [(32, 4, 64, 16), (3, 1, 32, 16), (5, 5, 48, 32), (40, 2, 16, 16), (16, 1, 128, 16), (10, 2, 112, 48)])
def test_attention_float32_matrix_unit(ops, geom, window):
    """The 32-bit attention on the matrix unit, against 64 bits and against itself: a request's tokens as one portion, as
    portions cut in the middle of a segment of 128 keys, and one by one give the same bits."""
    Hq, Hkv, D, page = geom
    o, n = ops[torch.float32], 389
    q, kc, vc, group, step = paged_setup([n, 131], [n, 131], Hq, Hkv, D, page, torch.float32, seed=D)
    with counted(o, "attention_f32", "mie_attention_f32_single", "mie_attention_f32_portions") as calls:
        whole, expect = run_attention(ops, torch.float32, q, kc, vc, group, step, Hq, Hkv, D, 1 / math.sqrt(D), window)
    assert calls == ["mie_attention_f32_portions"]
    torch.testing.assert_close(whole.double(), expect, **ATT_TOL[torch.float32])
    for a, b in ((0, 2), (2, 129), (129, 256), (256, n)):
        part = SimpleNamespace(token_row=step.token_row[a:b], positions=step.positions[a:b], num_rows=1, max_context=b, num_tokens=b - a,
                               num_decode_rows=0, max_row_tokens=b - a, row_start=torch.tensor([0, b - a], dtype=torch.int32, device=DEV),
                               row_position=torch.tensor([a], dtype=torch.int32, device=DEV))
        assert torch.equal(o.paged_attention(q[a:b], Hq, Hkv, D, kc, vc, group, part, 1 / math.sqrt(D), window), whole[a:b])
    for bound in (n, 2000):                     # a static bound on the context, as under capture
        wide = SimpleNamespace(block_tables=torch.nn.functional.pad(group.block_tables, (0, 2000 // page + 1 - group.block_tables.shape[1])))
        wide.max_blocks = wide.block_tables.shape[1]
        single = SimpleNamespace(token_row=step.token_row, positions=step.positions, num_rows=2, max_context=bound, num_tokens=n + 131,
                                 num_decode_rows=n + 131, max_row_tokens=1, row_start=None, row_position=None)
        with counted(o, "attention_f32", "mie_attention_f32_single", "mie_attention_f32_portions") as calls:
            out = o.paged_attention(q, Hq, Hkv, D, kc, vc, wide, single, 1 / math.sqrt(D), window)
        assert calls == ["mie_attention_f32_single"] and torch.equal(out, whole)


@pytest.mark.parametrize("D", [64, 96, 128])
def test_decode_attention_of_caches_off_16_bytes(ops, D):
    """Contiguous caches that begin 8 bytes into memory: the same result as of ones that begin on 16."""
    q, kc, vc, group, step = paged_setup([70, 33, 200], [1, 1, 1], 8, 2, D, 16, torch.bfloat16, seed=D)
    o = ops[torch.bfloat16]
    want = o.paged_attention(q, 8, 2, D, kc, vc, group, step, D ** -0.5, None)
    off = [torch.empty(t.numel() + 4, dtype=t.dtype, device=DEV)[4:].view(t.shape).copy_(t) for t in (kc, vc)]
    assert all(t.data_ptr() % 16 for t in off)
    assert torch.equal(o.paged_attention(q, 8, 2, D, *off, group, step, D ** -0.5, None), want)


def off_16_bytes(*caches):
    off = [torch.empty(t.numel() + 4, dtype=t.dtype, device=DEV)[4:].view(t.shape).copy_(t) for t in caches]
    assert all(t.data_ptr() % 16 for t in off)
    return off


@pytest.mark.parametrize("D", [64, 80, 96, 128])
def test_attention_of_caches_off_16_bytes_keeps_bits_and_memory(ops, D):
    """Caches that begin 8 bytes into memory, every kind of attention, split and whole contexts, eight and four waves, prompts: the
    bits of caches that begin on 16, and never a copy of the caches."""
    o, Hq, Hkv = ops[torch.bfloat16], 8, 2
    table = torch.randn(Hq, 40, device=DEV)
    kinds = [{}, dict(window=50), dict(weights="sigmoid", softcap=5.0), dict(weights="sigmoid", chunk=64), dict(distance_bias=table),
             dict(window=40, keep_first=5), dict(chunk=48), dict(sink=0.5)]
    for ctx, new in (([70, 33, 200], [1, 1, 1]), ([1, 16, 31, 33, 200] * 20, [1] * 100), ([100, 65] * 80, [1] * 160), ([90, 33, 200, 130], [1, 1, 64, 130])):
        q, kc, vc, group, step = paged_setup(ctx, new, Hq, Hkv, D, 16, torch.bfloat16, num_pages=4096, seed=D)
        off = off_16_bytes(kc, vc)
        for kind in kinds:
            kw = dict(kind)
            window = kw.pop("window", None)
            want = o.paged_attention(q, Hq, Hkv, D, kc, vc, group, step, D ** -0.5, window, **kw)
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            got = o.paged_attention(q, Hq, Hkv, D, *off, group, step, D ** -0.5, window, **kw)
            torch.cuda.synchronize()
            assert torch.cuda.max_memory_allocated() - before < kc.numel()
            assert torch.equal(got, want), (len(ctx), kind)


@pytest.mark.parametrize("M", [64, 140])
def test_decode_attention_from_sums_into_caches_off_16_bytes(engine_ops, M):
    """The decode kernel that finishes the projection, on caches 8 bytes into memory: results and caches as on 16."""
    from mini_inference_engine_amd.kernels.hip_backend import ProjectionSums
    from mini_inference_engine_amd.parts.rope import rotary_tables
    o, Hq, Hkv, D, page, K = engine_ops, 16, 4, 64, 16, 264
    ctx = ([1, 16, 17, 33, 128, 300, 48] * 20)[:M]
    _, kc, vc, group, step = paged_setup(ctx, [1] * M, Hq, Hkv, D, page, torch.bfloat16, seed=M)
    cos, sin = (t.to(DEV) for t in rotary_tables(10000.0, D, max(ctx) + 1))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    pos = step.positions
    group.slot_mapping = (group.block_tables[torch.arange(M, device=DEV), (pos // page).long()] * page + pos % page).to(torch.int32)
    made = []
    for caches in (off_16_bytes(kc, vc), (kc, vc)):
        pending = o.linear_rotary_kv_store(x, w, pos, cos, sin, D, Hq, Hkv, D, *caches, group.slot_mapping, for_attention=True)
        assert isinstance(pending, ProjectionSums)
        with counted(o, "attention_bf16", "mie_decode_attention_from_sums", defines=("-DHEAD_DIM=64",)) as calls:
            out = o.paged_attention(pending, Hq, Hkv, D, *caches, group, step, D ** -0.5, None)
        assert len(calls) == 1
        made.append((out, *caches))
    assert all(torch.equal(a, b) for a, b in zip(*made))


@pytest.mark.parametrize("window", [None, 1, 130])
@pytest.mark.parametrize("geom", [(32, 4, 64, 16), (3, 1, 32, 16), (5, 5, 48, 32), (40, 2, 16, 16), (16, 1, 128, 16), (10, 2, 112, 48), (6, 2, 80, 16)])
def test_attention_float32_few_single_tokens(ops, geom, window):
    """Few single tokens (four waves a segment) beside the same ones among many (one wave): the same bits, for every head size's
    number of value tiles a wave, segments that are begun, full and single keys."""
    Hq, Hkv, D, page = geom
    o, ctx = ops[torch.float32], [1, 127, 128, 129, 300]
    many = ctx + [500] * 1100
    q, kc, vc, group, step = paged_setup(many, [1] * len(many), Hq, Hkv, D, page, torch.float32, seed=D)
    splits = -(-500 // 128)
    heads = Hkv * -(-(Hq // Hkv) // 16)
    assert splits * heads * len(ctx) <= 1024 < heads * len(many)
    whole = o.paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 1 / math.sqrt(D), window)
    n = len(ctx)
    few = SimpleNamespace(token_row=step.token_row[:n], positions=step.positions[:n], num_rows=n, max_context=500, num_tokens=n,
                          num_decode_rows=n, max_row_tokens=1, row_start=None, row_position=None)
    out = o.paged_attention(q[:n], Hq, Hkv, D, kc, vc, SimpleNamespace(block_tables=group.block_tables[:n].contiguous(), max_blocks=group.max_blocks),
                            few, 1 / math.sqrt(D), window)
    assert torch.equal(out, whole[:n])
    expect = ref.ref_paged_attention(q[:n], Hq, Hkv, D, kc, vc, group.block_tables[:n], few.token_row, few.positions, 1 / math.sqrt(D), window, torch.float64)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[torch.float32])


# head size and the segments a compute unit up to which they are four waves' work, of several segments a token and of one
@pytest.mark.parametrize("case", [(16, 1, 1), (32, 2, 2), (48, 4, 3), (64, 4, 4), (80, 3, 2), (96, 3, 2), (112, 4, 4), (128, 4, 4)])
def test_attention_float32_of_as_many_single_tokens_as_four_waves_take(ops, case):
    """Single tokens at the line between the two kernels and one token beyond it: the same bits."""
    o, (D, several, one), cu = ops[torch.float32], case, torch.cuda.get_device_properties(0).multi_processor_count
    four = o.lib("attention_f32").mie_attention_f32_four_waves
    for ctx, splits, most in ((17, 1, one), (140, 2, several)):
        n = most * cu // splits
        assert four(n, 3, 1, D, splits) == 1 and four(n + 1, 3, 1, D, splits) == 0
        q, kc, vc, group, step = paged_setup([ctx - r % 16 for r in range(n + 1)], [1] * (n + 1), 3, 1, D, 16, torch.float32, seed=D)
        beyond, expect = run_attention(ops, torch.float32, q, kc, vc, group, step, 3, 1, D, D ** -0.5, None)
        torch.testing.assert_close(beyond.double(), expect, **ATT_TOL[torch.float32])
        few = SimpleNamespace(token_row=step.token_row[:n], positions=step.positions[:n], num_rows=n, max_context=ctx, num_tokens=n, num_decode_rows=n,
                              max_row_tokens=1, row_start=None, row_position=None)
        tables = SimpleNamespace(block_tables=group.block_tables[:n].contiguous(), max_blocks=group.max_blocks)
        assert torch.equal(o.paged_attention(q[:n], 3, 1, D, kc, vc, tables, few, D ** -0.5, None), beyond[:n])


# heads, kv heads, head size, page, rows, their tokens, keys before them: one segment at most; rows of one, two and a half and three tiles a
# workgroup in more workgroups than there are compute units; many workgroups of heads of 16, and of 48 and 80 with two segments
@pytest.mark.parametrize("window", [None, 37])
@pytest.mark.parametrize("case", [(32, 4, 64, 16, 1, 128, 0), (40, 2, 16, 16, 3, 100, 28), (16, 1, 128, 16, 2, 33, 50), (12, 12, 64, 16, 32, 16, 250),
                                  (32, 8, 128, 16, 40, 20, 300), (6, 2, 112, 16, 129, 5, 200), (3, 1, 32, 16, 300, 13, 130), (8, 2, 48, 48, 260, 9, 0),
                                  (40, 2, 16, 16, 16, 60, 300), (8, 2, 48, 16, 80, 30, 200), (16, 2, 80, 16, 64, 30, 0), (12, 12, 64, 16, 16, 75, 0)])
def test_attention_float32_portions_by_single_waves(ops, case, window):
    """Portions that single waves take against the same ones by workgroups of four tiles (a few of the rows, the context not said): the
    same bits, also beside a later token's keys and values that are not finite; and against 64 bits."""
    Hq, Hkv, D, page, rows, new, have = case
    o, few, scale = ops[torch.float32], min(rows, 4), 1 / math.sqrt(D)
    q, kc, vc, group, step = paged_setup([have + new] * rows, [new] * rows, Hq, Hkv, D, page, torch.float32, seed=D)
    alone = o.lib("attention_f32").mie_attention_f32_alone
    assert alone(rows, new, Hq, Hkv, D, page, have + new) == 1 and alone(few, new, Hq, Hkv, D, page, 0) == 0
    part = SimpleNamespace(token_row=step.token_row[:few * new], positions=step.positions[:few * new], num_rows=few, max_context=0, num_tokens=few * new,
                           num_decode_rows=0, max_row_tokens=new, row_start=step.row_start[:few + 1], row_position=step.row_position[:few])
    tables = SimpleNamespace(block_tables=group.block_tables[:few].contiguous(), max_blocks=group.max_blocks)
    out, expect = run_attention(ops, torch.float32, q, kc, vc, group, step, Hq, Hkv, D, scale, window)
    torch.testing.assert_close(out.double(), expect, **ATT_TOL[torch.float32])
    last = have + new - 1
    for spoilt in (False, True):
        if spoilt:
            pages = group.block_tables[:, last // page].long()
            kc[pages, :, last % page] = float("inf")
            vc[pages, :, :, last % page] = float("nan")
        a = o.paged_attention(q, Hq, Hkv, D, kc, vc, group, step, scale, window)[:few * new]
        b = o.paged_attention(q[:few * new], Hq, Hkv, D, kc, vc, tables, part, scale, window)
        assert torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(b, 7.0))
        assert spoilt or torch.equal(a, out[:few * new])
        seen = a.view(few, new, -1)[:, :-1]
        assert bool(torch.isfinite(seen).all()) and (not spoilt or torch.equal(seen, out.view(rows, new, -1)[:few, :-1]))


def test_attention_float32_of_pages_beyond_32_bit_offsets(ops):
    """A page of more than 2^24 tokens (one holds a whole cache): the bits of the same keys in small pages."""
    Hq, Hkv, D, ctx, page = 4, 1, 16, 300, (1 << 24) + 16
    q, kc, vc, group, step = paged_setup([ctx], [140], Hq, Hkv, D, 16, torch.float32, seed=5)
    want = ops[torch.float32].paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.25, None)
    named = group.block_tables[0, :-(-ctx // 16)].long()
    k, v = torch.zeros(1, Hkv, page, D, device=DEV), torch.zeros(1, Hkv, D, page, device=DEV)
    k[0, 0, :16 * named.numel()] = kc[named, 0].reshape(-1, D)
    v[0, 0, :, :16 * named.numel()] = vc[named, 0].permute(1, 0, 2).reshape(D, -1)
    one = SimpleNamespace(block_tables=torch.zeros(1, 1, dtype=torch.int32, device=DEV), max_blocks=1)
    with counted(ops[torch.float32], "attention_f32", "mie_attention_f32_portions") as calls:
        got = ops[torch.float32].paged_attention(q, Hq, Hkv, D, k, v, one, step, 0.25, None)
    assert len(calls) == 1 and torch.equal(got, want)


def test_attention_float32_of_a_step_that_does_not_describe_its_rows(ops):
    """What the float32 attention reads of a step beyond its tokens is only there to choose a faster kernel: without the longest
    row's length or the largest context, or with row arrays of another type, the result is the same."""
    Hq, Hkv, D, page = 4, 2, 32, 16
    q, kc, vc, group, step = paged_setup([37, 64, 20], [1, 64, 5], Hq, Hkv, D, page, torch.float32, seed=2)
    expect = ref.ref_paged_attention(q, Hq, Hkv, D, kc, vc, group.block_tables, step.token_row, step.positions, 0.2, None, torch.float64)
    torch.full((70, Hq * D), float("nan"), device=DEV)          # what an unwritten result would be made of
    for change in (dict(max_row_tokens=0), dict(max_context=0), dict(row_start=step.row_start.long()), dict(row_position=None), dict(row_start=None)):
        out = ops[torch.float32].paged_attention(q, Hq, Hkv, D, kc, vc, group, SimpleNamespace(**{**vars(step), **change}), 0.2, None)
        torch.testing.assert_close(out.double(), expect, **ATT_TOL[torch.float32])


def test_attention_float32_single_tokens_in_bounded_memory(ops):
    """Single tokens under a static bound on the context that makes their segments' results too many to lie side by side: the
    same bits as under a tight bound, and no more memory than is set aside for them."""
    Hq, Hkv, D, page, rows, bound = 32, 4, 64, 16, 37, 65536
    o = ops[torch.float32]
    q, kc, vc, group, step = paged_setup([(37 * r) % 700 + 1 for r in range(rows)], [1] * rows, Hq, Hkv, D, page, torch.float32, seed=4)
    tight = o.paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.125, None)
    assert rows * Hq * (bound // 128) * (D + 2) * 4 > o.F32_SEGMENT_BYTES
    bt = torch.nn.functional.pad(group.block_tables, (0, bound // page - group.block_tables.shape[1]))
    wide = SimpleNamespace(block_tables=bt, max_blocks=bt.shape[1])
    bounded = SimpleNamespace(**{**vars(step), "max_context": bound})
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    loose = o.paged_attention(q, Hq, Hkv, D, kc, vc, wide, bounded, 0.125, None)
    assert torch.cuda.max_memory_allocated() - before <= o.F32_SEGMENT_BYTES + (4 << 20)
    assert torch.equal(loose, tight)


# 16 queries of a wave: 16, 2, 5 and 1 neighbouring tokens; a window whose first key lies inside a tile of 16 keys
@pytest.mark.parametrize("window", [None, 21])
@pytest.mark.parametrize("geom", [(4, 4, 64, 16), (32, 4, 64, 16), (3, 1, 32, 48), (32, 2, 16, 16)])
def test_attention_float32_looks_at_no_other_querys_keys(ops, geom, window):
    """A row lengthened with padding tokens whose keys lie in the scratch page, with NaN in every slot the row did not write:
    the row's own tokens get the bits of the step without padding.  And what is not a number in a value of the row itself
    reaches the tokens that see it, in the dimension it stands in, and no others."""
    Hq, Hkv, D, page = geom
    o, n, real, padded = ops[torch.float32], 170, 29, 48
    q, kc, vc, group, step = paged_setup([n], [real], Hq, Hkv, D, page, torch.float32, seed=D + Hq)
    clean = o.paged_attention(q, Hq, Hkv, D, kc, vc, group, step, 0.2, window)
    bt = torch.nn.functional.pad(group.block_tables, (0, 4))
    lo = 0 if window is None else n - real - window + 1
    own = torch.zeros(kc.shape[0], page, dtype=torch.bool, device=DEV)
    for p in range(lo, n):
        own[int(bt[0, p // page]), p % page] = True
    kd, vd = kc.clone(), vc.clone()
    kd.permute(0, 2, 1, 3)[~own] = float("nan")
    vd.permute(0, 3, 1, 2)[~own] = float("nan")
    longer = SimpleNamespace(token_row=torch.zeros(padded, dtype=torch.int32, device=DEV), num_rows=1, num_tokens=padded,
                             positions=torch.arange(n - real, n - real + padded, dtype=torch.int32, device=DEV),
                             max_context=n - real + padded, num_decode_rows=0, max_row_tokens=padded,
                             row_start=torch.tensor([0, padded], dtype=torch.int32, device=DEV), row_position=step.row_position)
    wide = SimpleNamespace(block_tables=bt, max_blocks=bt.shape[1])
    got = o.paged_attention(torch.cat([q, torch.full_like(q[:1], float("nan")).expand(padded - real, -1)]), Hq, Hkv, D, kd, vd, wide,
                            longer, 0.2, window)
    assert torch.equal(got[:real], clean)
    for at, what in ((n - 3, float("inf")), (n - real + 1, float("-inf")), (n - 20, float("nan"))):
        ve = vd.clone()
        ve[int(bt[0, at // page]), 0, 5, at % page] = what
        odd = o.paged_attention(q, Hq, Hkv, D, kc, ve, group, step, 0.2, window).view(real, Hkv, Hq // Hkv, D)
        sees = torch.arange(n - real, n, device=DEV)
        sees = (sees >= at) & (sees - at < (window or n))
        want = clean.clone().view(real, Hkv, Hq // Hkv, D)
        want[sees, 0, :, 5] = what
        assert torch.equal(torch.nan_to_num(odd, 1e6, 2e6, 3e6), torch.nan_to_num(want, 1e6, 2e6, 3e6))


# ------------------------------------------------------------------- sampling
def test_sample_greedy_and_ties(ops):
    torch.manual_seed(0)
    logits = torch.randn(9, 331, device=DEV)
    logits[3, 100] = logits[3, 200] = 50.0          # equal maxima: the lowest index wins
    logits[4] = 0.0
    zeros = torch.zeros(9, device=DEV)
    out = ops[torch.float32].sample(logits, zeros, torch.zeros(9, dtype=torch.int64, device=DEV),
                                    torch.zeros(9, dtype=torch.int32, device=DEV))
    expect = logits.argmax(-1)
    expect[3], expect[4] = 100, 0
    assert out.tolist() == expect.tolist()


@pytest.mark.parametrize("V, ld", [(4099, 4100), (8192, 8192), (4097, 4097), (5, 8)])
def test_sample_wide_rows(ops, V, ld):
    """Rows read four values at a time and one at a time, with a tail: the winner may sit anywhere."""
    torch.manual_seed(V)
    full = torch.randn(6, ld, device=DEV)
    full[:, V:] = 100.0                                  # beyond the vocabulary: never looked at
    logits = full[:, :V]
    places = [0, V - 1, max(V - 2, 0), V // 2, min(V & ~3, V - 1), min(V - 1, 4095)]
    for r, v in enumerate(places):
        logits[r, v] = 30.0
    zeros = torch.zeros(6, device=DEV)
    out = ops[torch.float32].sample(logits, zeros, torch.zeros(6, dtype=torch.int64, device=DEV),
                                    torch.zeros(6, dtype=torch.int32, device=DEV))
    assert out.tolist() == places
    temps = torch.full((6,), 0.9, device=DEV)
    seeds = torch.arange(6, dtype=torch.int64, device=DEV) + 11
    ctrs = torch.arange(6, dtype=torch.int32, device=DEV)
    noisy = (torch.randn(6, ld, device=DEV) * 2)[:, :V]
    out = ops[torch.float32].sample(noisy, temps, seeds, ctrs).tolist()
    for r in range(6):
        z = ref.ref_perturbed(noisy[r], 0.9, int(seeds[r]), int(ctrs[r]))
        assert float(z.max() - z[out[r]]) <= 1e-4, f"row {r}: chose {out[r]}, best {int(z.argmax())}"


def test_sample_noise_matches_specification(ops):
    torch.manual_seed(1)
    V = 1000
    logits = torch.randn(6, V, device=DEV) * 2
    temps = torch.tensor([0.8, 0.0, 1.5, 0.8, 0.3, 1.0], device=DEV)
    seeds = torch.tensor([1, 2, 2**40 + 3, 1, -5, 2**62], dtype=torch.int64, device=DEV)
    ctrs = torch.tensor([0, 5, 7, 1, 2**31 - 1, 3], dtype=torch.int32, device=DEV)
    out = ops[torch.float32].sample(logits, temps, seeds, ctrs).tolist()
    for r in range(6):
        z = ref.ref_perturbed(logits[r], float(temps[r]), int(seeds[r]), int(ctrs[r]))
        # the kernel's float32 noise may differ from the float64 one in the last digits
        assert float(z.max() - z[out[r]]) <= 1e-4, f"row {r}: chose {out[r]}, best {int(z.argmax())}"
    # the noise depends on the counter: on flat logits the draw is the noise's argmax, so 16 counters of one
    # seed give (nearly) 16 different tokens out of 1000, and a repeated counter repeats its token
    flat = torch.zeros(17, V, device=DEV)
    counters = torch.tensor(list(range(16)) + [3], dtype=torch.int32, device=DEV)
    drawn = ops[torch.float32].sample(flat, torch.ones(17, device=DEV), torch.full((17,), 9, dtype=torch.int64, device=DEV),
                                      counters).tolist()
    assert len(set(drawn[:16])) >= 14 and drawn[16] == drawn[3]


def test_sample_distribution(ops):
    """Frequencies of the draw follow softmax(logits / t): chi-square on a small vocabulary."""
    V, n, t = 7, 4000, 0.7
    logits_row = torch.tensor([0.1, 1.0, -0.5, 2.0, 0.0, 1.5, -2.0], device=DEV)
    logits = logits_row.repeat(n, 1).contiguous()
    out = ops[torch.float32].sample(logits, torch.full((n,), t, device=DEV),
                                    torch.full((n,), 1234, dtype=torch.int64, device=DEV),
                                    torch.arange(n, dtype=torch.int32, device=DEV))
    counts = torch.bincount(out.long().cpu(), minlength=V).double()
    p = torch.softmax(logits_row.double().cpu() / t, 0)
    chi2 = float(((counts - n * p) ** 2 / (n * p)).sum())
    assert chi2 < 22.46, f"chi-square {chi2:.1f} with 6 degrees of freedom (p < 0.001 above 22.46)"
