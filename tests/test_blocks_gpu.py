"""Parity of every instruction block, called through the C ABI (via the block
mirror of webgpt_amd/blocks.py), against the CPU oracle on the same seeded inputs.
fp32 bar: |got - want| <= 1e-5 + 1e-4 |want|; copies, gathers and the int8
dequantisation are bit-exact."""
import math
import time

import numpy as np
import pytest

from oracle import ref
from webgpt_amd import WgptError, blocks
from webgpt_amd.blocks import (AttentionBlock, DeEmbedBlock, EmbedBlock, FastMatMulBlock, GeluBlock, LayerNormBlock,
                               ResidualBlock, SoftmaxBlock, init_tensor, run_passes)

from helpers import close, pack_words, worst

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(99)


def rnd(*shape, scale=1.0):
    return (RNG.standard_normal(shape) * scale).astype(np.float32)


def run(inst, shape):
    run_passes(inst["passes"])
    out = inst["resultBuffer"].download().reshape(shape)
    blocks.clearOperationCache()
    return out


@pytest.mark.parametrize("M,N,K", [(1, 8, 4), (1, 768, 768), (1, 2304, 768), (1, 768, 3072), (1, 72, 100), (2, 64, 64),
                                   (3, 1600, 1600), (4, 384, 1536), (5, 8, 12), (7, 200, 36), (16, 768, 768),
                                   (128, 2304, 768), (65, 136, 260), (200, 768, 3072), (2048, 4096, 64), (2050, 4104, 40),
                                   # short prompts: K split over the waves of a workgroup (32x32 and 16x16 blocks, ragged M,
                                   # K steps that do not divide by the eight waves)
                                   (17, 32, 128), (100, 1600, 1600), (250, 96, 3200), (33, 6400, 1600), (256, 384, 384), (31, 64, 144),
                                   # the two-group kernel: K split four ways, one tile per compute unit, ragged M and N
                                   # with an odd number of K steps, and the same shape with a ragged K (other kernel)
                                   (512, 1024, 1024), (512, 4096, 1024), (950, 2056, 96), (950, 2056, 100)])
def test_fast_matmul(device, M, N, K):
    A, W, b = rnd(M, K), rnd(K, N, scale=0.05), rnd(N)
    inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(W, [K, N]), init_tensor(b, [N]))
    got = run(inst, (M, N))
    want = ref.matmul_bias(A, W, b)
    assert close(got, want), worst(got, want)


def _dispatch_edge_shapes():
    """Seeded shapes around the tile counts at which the matmul changes kernel or K split (64x128 tiles in whole
    rounds of 256 workgroups, 64x64 tiles otherwise), with ragged M, N and K among them."""
    rng = np.random.default_rng(20240607)
    shapes = []
    for tiles in (63, 64, 65, 127, 128, 218, 255, 256, 257, 435, 512, 513, 1023, 1024, 1025):
        mt = int(rng.integers(2, 17))                      # rows of 64
        nt = max(1, tiles // mt)                           # columns of 128
        M = 64 * mt - int(rng.integers(0, 40))
        N = 128 * nt - 8 * int(rng.integers(0, 8))
        K = int(rng.choice([32, 96, 100, 128, 256, 260, 512, 1024]))
        shapes.append((max(M, 5), max(N, 8), K))
    return shapes


@pytest.mark.parametrize("M,N,K", [(128, 2304, 768), (64, 1536, 640), (128, 768, 672), (100, 768, 576), (448, 512, 768),
                                   (449, 512, 768), (128, 1600, 6400), (33, 4800, 1600)])
def test_fast_matmul_with_few_rows_and_odd_slice_counts(device, M, N, K):
    # up to 448 rows the K range is cut into any number of slices that leaves whole steps of 32 (here 3, 5, 7, 6, ...),
    # not only powers of two; 449 rows fall back to doubling. (Weights scaled with K: near a zero of the output the
    # rounding of 6400 fp32 additions, in whatever order, is otherwise larger than the absolute tolerance.)
    A, W, b = rnd(M, K), rnd(K, N, scale=0.05 * min(1.0, 1024.0 / K)), rnd(N)
    inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(W, [K, N]), init_tensor(b, [N]))
    got = run(inst, (M, N))
    want = ref.matmul_bias(A, W, b)
    assert close(got, want), worst(got, want)


@pytest.mark.parametrize("M,N,K", _dispatch_edge_shapes())
def test_fast_matmul_around_kernel_choices(device, M, N, K):
    A, W, b = rnd(M, K), rnd(K, N, scale=0.05), rnd(N)
    inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(W, [K, N]), init_tensor(b, [N]))
    got = run(inst, (M, N))
    want = ref.matmul_bias(A, W, b)
    assert close(got, want), worst(got, want)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [(5, 8, 4), (16, 24, 32), (17, 40, 36), (16, 4800, 1600), (31, 104, 900), (33, 2304, 768),
                                   (65, 72, 100), (128, 2304, 768), (128, 3080, 772), (129, 136, 4096), (500, 1032, 96),
                                   (943, 768, 768), (1000, 3072, 1060)])
def test_split_matmul_error_bound(device, int8, M, N, K):
    """The products on the bf16 matrix cores against 64-bit ones: the edges of every tile that rows of W have (16, 32, 64
    and 128 rows; the 64x128 one is for a model's order of the weights), partial steps of 32 k and sliced K. The parts of a
    value of 2**-110 and more add up to it exactly and all six products kept are exact, so the error
    is that of the fp32 sums: at most six roundings per sixteen k, a few for the slices and waves, each at most 2**-24 of
    the sum of magnitudes, and 2**-24 of it for the products left out (a value's second and third parts are at most 2**-8
    and 2**-17 of it, and two such products are left out)."""
    rng = np.random.default_rng(M * N + K)
    A = rng.standard_normal((M, K)).astype(np.float32) * np.exp(rng.standard_normal((M, 1))).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    if int8:
        q = rng.integers(-128, 128, (K, N))
        scale = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
        W = q.astype(np.float64) * (scale / np.float32(127.0)).astype(np.float64)
        inst = FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(A, [M, K]), init_tensor(pack_words(q), [K, N // 4]),
                                               init_tensor(scale, [N]), init_tensor(bias, [N]))
    else:
        w = (rng.standard_normal((K, N)) * np.exp2(rng.integers(-8, 8, (K, N)))).astype(np.float32)
        W = w.astype(np.float64)
        inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(w, [K, N]), init_tensor(bias, [N]))
    got = run(inst, (M, N)).astype(np.float64)
    want = A.astype(np.float64) @ W + bias
    size = np.abs(A).astype(np.float64) @ np.abs(W) + np.abs(bias)
    bound = 2.0 ** -24 * (6 * K / 16 + 20) * size
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))
    # and in practice no worse than sums of a few products at a time in fp32
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * max(4.0, K ** 0.5) * np.linalg.norm(size)


@pytest.mark.parametrize("M,N,K", [(16, 64, 4), (33, 72, 64), (65, 136, 1024), (130, 264, 260)])
def test_split_matmul_largest_part_left_out(device, M, N, K):
    """Every value 1 + 2**-8 - 2**-17, whose parts are 1, 2**-8 and -2**-17: the products left out are 1.98 * 2**-25 of each
    product, all of one sign. Bound of test_split_matmul_error_bound."""
    x = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(np.full((M, K), x), [M, K]), init_tensor(np.full((K, N), x), [K, N]),
                                       init_tensor(np.zeros(N, np.float32), [N]))
    got = run(inst, (M, N)).astype(np.float64)
    want = K * np.float64(x) ** 2
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * (6 * K / 16 + 2) * want), float(np.abs(got / want - 1).max()) * 2.0 ** 24


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [(5, 8, 4), (17, 40, 100), (33, 768, 3072), (130, 136, 256)])
def test_split_matmul_not_finite(device, int8, M, N, K):
    """Operands without a three-way bf16 split (infinite ones, and those within half a bf16 ulp of the largest float) give
    what fp32 products give; all other values stay small integers, whose sums are exact."""
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(1, 5, (M, K)).astype(np.float32)
    q = rng.integers(1, 5, (K, N)) * rng.choice([-1, 1], (1, N))
    q[1], q[:, 5] = np.sign(q[1]), np.abs(q[:, 5])  # the large values meet ones, and each other with one sign: one reading
    A[:, K - 1] = 1
    w = q.astype(np.float32)
    A[0, K - 1], A[1, 0], A[2, K // 2], A[3, 1] = np.inf, -np.inf, np.nan, np.float32(3.4e38)
    if int8:
        q[0, 3] = 0  # inf times zero
        w = q.astype(np.float32)
        inst = FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(A, [M, K]), init_tensor(pack_words(q), [K, N // 4]),
                                               init_tensor(np.full(N, 127, np.float32), [N]), init_tensor(np.zeros(N, np.float32), [N]))
    else:
        w[1, 2], w[K - 1, 5] = -np.inf, np.float32(3.4e38)
        inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(w, [K, N]), init_tensor(np.zeros(N, np.float32), [N]))
    got = run(inst, (M, N))
    with np.errstate(all="ignore"):
        want = np.zeros((M, N), np.float32)  # products and sums rounded to fp32, as far as infinities go
        for k in range(K):
            want = (want + A[:, k:k + 1] * w[k:k + 1]).astype(np.float32)
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    assert np.allclose(got[fin], want[fin], rtol=1e-6, atol=0)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [(17, 568, 1872), (100, 4440, 8), (33, 4200, 1048), (33, 2816, 1836), (33, 4216, 1296), (33, 2744, 2148),
                                   (100, 3240, 4), (17, 4280, 2068), (300, 3400, 648), (300, 3528, 900), (943, 544, 4), (449, 4552, 36)])
def test_split_matmul_not_finite_in_every_kernel(device, int8, M, N, K):
    """Shapes that take each of the kernels (16, 32, 64 and 128 rows to a tile), with and without slices, most of them with a
    partial step of 32 k: the rows and columns of infinities and NaN, and only they, come out so; all other values are small
    integers, whose sums are exact."""
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(-4, 5, (M, K)).astype(np.float32)
    q = rng.integers(1, 5, (K, N)) * rng.choice([-1, 1], (1, N))
    w = q.astype(np.float32)
    A[3, 0], A[M - 1, K - 1], A[M // 2, K // 2] = np.inf, -np.inf, np.nan
    if int8:
        inst = FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(A, [M, K]), init_tensor(pack_words(q), [K, N // 4]),
                                               init_tensor(np.full(N, 127, np.float32), [N]), init_tensor(np.zeros(N, np.float32), [N]))
    else:
        A[:, K - 1][A[:, K - 1] == 0] = 1  # (no infinity times zero)
        w[K - 1, N - 3] = np.inf
        inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(w, [K, N]), init_tensor(np.zeros(N, np.float32), [N]))
    got = run(inst, (M, N))
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ w.astype(np.float64)
    assert np.array_equal(got, want.astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("big", ["all", "row", "value"])
@pytest.mark.parametrize("M,N,K", [(5, 8, 100), (17, 568, 1872), (33, 2816, 1836), (33, 2744, 2148), (17, 4280, 2068), (100, 3240, 40), (300, 3528, 900),
                                   (449, 4552, 260)])
def test_int8_matmul_large_activations(device, M, N, K, big):
    """Activations whose product with the bare int8 weights leaves the range of fp32, while that with scaled weights does not:
    everywhere, in one row and in one value (whose wave's sums are then scaled apart from the others'). Error: that of
    test_split_matmul_error_bound, and two roundings for the scaled weights."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    if big == "all":
        A *= np.float32(3e36)
    elif big == "row":
        A[M // 2] *= np.float32(3e36)
    else:
        A[M // 2, K // 3] = 3e37
    q = rng.integers(-128, 128, (K, N))
    scale = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    got = run(FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(A, [M, K]), init_tensor(pack_words(q), [K, N // 4]), init_tensor(scale, [N]),
                                              init_tensor(bias, [N])), (M, N)).astype(np.float64)
    W = q * (scale / np.float32(127.0)).astype(np.float64)
    want = A.astype(np.float64) @ W + bias
    size = np.abs(A).astype(np.float64) @ np.abs(W) + np.abs(bias)
    assert np.abs(size).max() < 1e38
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * (K + 24) * size), float(np.max(np.abs(got - want) / size))


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("small", ["A", "row", "W", "column", "value"])
@pytest.mark.parametrize("M,N,K", [(5, 8, 100), (17, 568, 1872), (33, 4200, 1048), (33, 2744, 2148), (100, 3240, 40), (300, 3400, 648), (449, 4552, 36)])
def test_split_matmul_tiny_values(device, int8, M, N, K, small):
    """Operands around 2**-119, whose third bf16 part is too small for bf16: the same relative error as at any other size, also
    where a single row, column or output is that small. The fp32 sums have a quantum of 2**-149."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    tiny = np.float32(2.0 ** -119)
    if small == "A" or (int8 and small == "W"):
        A *= tiny
    elif small in ("row", "value"):
        A[M // 2] *= tiny
        if small == "value":  # (the first column of W takes that row's only value that is not tiny)
            A[M // 2, 0] = 1
    if int8:
        q = rng.integers(-128, 128, (K, N))
        if small == "value":
            q[0, 1:] = 1
            q[0, 0] = 0
        scale = rng.uniform(100, 200, N).astype(np.float32)
        inst = FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(A, [M, K]), init_tensor(pack_words(q), [K, N // 4]), init_tensor(scale, [N]),
                                               init_tensor(np.zeros(N, np.float32), [N]))
        W = q * (scale / np.float32(127.0)).astype(np.float64)
    else:
        w = rng.standard_normal((K, N)).astype(np.float32) * (tiny if small == "W" else np.float32(1))
        if small == "column":
            w[:, N // 3] *= tiny
        elif small == "value":
            w[0, 0] = 0
        inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(w, [K, N]), init_tensor(np.zeros(N, np.float32), [N]))
        W = w.astype(np.float64)
    got = run(inst, (M, N)).astype(np.float64)
    want = A.astype(np.float64) @ W
    bound = 2.0 ** -24 * (K + 24) * (np.abs(A).astype(np.float64) @ np.abs(W)) + K * 2.0 ** -149
    if small == "value":
        got, want, bound = got[M // 2, :1], want[M // 2, :1], bound[M // 2, :1]
    assert np.linalg.norm((got - want) / bound) <= 0.25 * math.sqrt(got.size), float(np.linalg.norm((got - want) / bound) / math.sqrt(got.size))
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))


@pytest.mark.parametrize("M,N,K", [(5, 8, 100), (17, 568, 1872), (33, 4200, 1048), (33, 2744, 2148), (100, 3240, 40), (300, 3400, 648), (449, 4552, 36)])
@pytest.mark.parametrize("small", ["A", "W"])
def test_split_matmul_tiny_times_large(device, small, M, N, K):
    """One operand around 2**-119, the other around 2**30: the outputs are not tiny themselves. Independent roundings of K
    additions, each 2**-25 of a partial sum in the mean square and none larger than the outputs: sqrt(K) 2**-25 in norm, of
    which four times is allowed (2**-15.7 with the third parts lost)."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32) * np.float32(2.0 ** (-119 if small == "A" else 30))
    w = rng.standard_normal((K, N)).astype(np.float32) * np.float32(2.0 ** (30 if small == "A" else -119))
    inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(A, [M, K]), init_tensor(w, [K, N]), init_tensor(np.zeros(N, np.float32), [N]))
    got = run(inst, (M, N)).astype(np.float64)
    want = A.astype(np.float64) @ w.astype(np.float64)
    assert np.linalg.norm(got - want) <= 4 * math.sqrt(K) * 2.0 ** -25 * np.linalg.norm(want), float(np.linalg.norm(got - want) / np.linalg.norm(want))


def _launch_ms(inst, launches=40):
    """Milliseconds of a launch, the best of three runs of them (the copy of the result that ends a run is in it)."""
    best = math.inf
    for _ in range(4):
        t = time.perf_counter()
        for _ in range(launches):
            run_passes(inst["passes"])
        inst["resultBuffer"].download()
        best = min(best, time.perf_counter() - t)
    return 1e3 * best / launches


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [(16, 2304, 768), (128, 3072, 768), (943, 3072, 768)])
def test_split_matmul_not_finite_in_time(device, int8, M, N, K):
    """Sums that are taken again cost fp32 matrix instructions (2.7 times, int8 5.3 times the time of the split ones), not one
    product after the other: a launch with nothing but NaN takes less than five times a launch with none (measured: 1.2 to
    2.5; 9 to 30 one after the other)."""
    rng = np.random.default_rng(M)
    A = rng.standard_normal((M, K)).astype(np.float32)
    ms = []
    for a in (A, np.full_like(A, np.nan)):
        if int8:
            inst = FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(a, [M, K]), init_tensor(pack_words(rng.integers(-127, 128, (K, N))), [K, N // 4]),
                                                   init_tensor(np.ones(N, np.float32), [N]), init_tensor(np.zeros(N, np.float32), [N]))
        else:
            inst = FastMatMulBlock.newInstance(M, N, K, init_tensor(a, [M, K]), init_tensor(rnd(K, N), [K, N]), init_tensor(np.zeros(N, np.float32), [N]))
        ms.append(_launch_ms(inst))
        blocks.clearOperationCache()
    assert ms[1] < 5 * ms[0], ms


@pytest.mark.parametrize("M,N,K,int8", [(5, 2 ** 20 + 8, 516, False), (17, 2 ** 22 + 32, 516, True), (530000, 8, 1024, False), (5, 2 ** 27 + 8, 4, False)])
def test_matmul_beyond_two_gib(device, M, N, K, int8):
    """Operands beyond the reach of 32-bit offsets: W in runs of rows (fp32 and int8), A in runs of rows, and rows of W of which
    not even four are in reach. Small integers, repeated with a prime period: every sum is exact."""
    rng = np.random.default_rng(N)
    A = np.tile(rng.integers(-3, 4, (min(M, 4099), K)).astype(np.float32), ((M + 4098) // 4099, 1))[:M]
    base = rng.integers(-3, 4, (K, min(N, 4099))).astype(np.int8 if int8 else np.float32)
    W = np.tile(base, (1, (N + 4098) // 4099))[:, :N]
    bias = np.tile(rng.integers(-3, 4, base.shape[1]).astype(np.float32), (N + 4098) // 4099)[:N]
    if int8:
        W = np.ascontiguousarray(W).view(np.int32)
    bufs = [init_tensor(A, [M, K]), init_tensor(W, W.shape), init_tensor(bias, [N])]
    try:
        if int8:
            bufs.append(init_tensor(np.full(N, 127, np.float32), [N]))
            inst = FastMatMulBlock.newInt8Instance(M, N, K, bufs[0], bufs[1], bufs[3], bufs[2])
        else:
            inst = FastMatMulBlock.newInstance(M, N, K, *bufs)
        got = run(inst, (M, N))
    finally:
        for b in bufs:
            b.destroy()
        FastMatMulBlock.destroyBuffers()  # (up to 2.7 GB of result)
    want = A[:4099] @ base.astype(np.float32) + bias[:base.shape[1]]
    for m in range(0, M, len(want)):
        for n in range(0, N, want.shape[1]):
            part = got[m:m + len(want), n:n + want.shape[1]]
            assert np.array_equal(part, want[:part.shape[0], :part.shape[1]]), (m, n)


def test_fast_matmul_exact_and_preconditions(device):
    A = RNG.integers(-8, 9, (3, 12)).astype(np.float32)
    W = RNG.integers(-8, 9, (12, 16)).astype(np.float32)
    b = RNG.integers(-8, 9, 16).astype(np.float32)
    bufs = init_tensor(A, [3, 12]), init_tensor(W, [12, 16]), init_tensor(b, [16])
    assert np.array_equal(run(FastMatMulBlock.newInstance(3, 16, 12, *bufs), (3, 16)), A @ W + b)
    with pytest.raises(ValueError, match="Cols must be divisible by 16."):
        FastMatMulBlock.newInstance(3, 12, 12, *bufs)
    # the library checks shapes against buffer sizes before any launch
    with pytest.raises(WgptError, match="buffer holds"):
        run_passes(FastMatMulBlock.newInstance(4, 16, 12, *bufs)["passes"])
    blocks.clearOperationCache()


@pytest.mark.parametrize("M,N", [(1, 4), (1, 768), (3, 384), (130, 1600)])
def test_residual_and_gelu(device, M, N):
    a, b = rnd(M, N, scale=3.0), rnd(M, N)
    got = run(ResidualBlock.newInstance(M, N, init_tensor(a, [M, N]), init_tensor(b, [M, N])), (M, N))
    assert np.array_equal(got, a + b)
    a[0, :4] = [-10.5, 10.5, -10.0, 10.0]
    got = run(GeluBlock.newInstance(M, N, init_tensor(a, [M, N])), (M, N))
    want = ref.gelu(a)
    assert close(got, want), worst(got, want)
    assert got[0, 0] == 0.0 and got[0, 1] == np.float32(10.5)


@pytest.mark.parametrize("M,N", [(1, 4), (1, 768), (5, 384), (64, 1600), (2, 4100), (3, 1024)])
def test_layernorm(device, M, N):
    x, g, b = rnd(M, N, scale=2.0) + 0.5, rnd(N), rnd(N)
    got = run(LayerNormBlock.newInstance(M, N, init_tensor(x, [M, N]), init_tensor(g, [N]), init_tensor(b, [N])), (M, N))
    want = ref.layernorm(x, g, b)
    assert close(got, want), worst(got, want)


@pytest.mark.parametrize("M,N", [(1, 1), (3, 7), (12, 64), (24, 129), (6, 1024), (2, 5000)])
def test_softmax(device, M, N):
    x = rnd(M, N, scale=3.0)
    if N > 2:
        x[0, 2:] = -1e9
    got = run(SoftmaxBlock.newInstance(M, N, init_tensor(x, [M, N])), (M, N))
    want = ref.softmax(x)
    assert close(got, want, atol=1e-7), worst(got, want, atol=1e-7)
    if N > 2:
        assert np.count_nonzero(got[0, 2:]) == 0


@pytest.mark.parametrize("M,N", [(1, 1), (3, 7), (24, 129), (65, 64)])
def test_softmax_transposed_store(device, M, N):
    # SoftmaxBlock.newInstance(rows, cols, in, transpose=true): out[i * M + row] (instructions.js:594)
    x = rnd(M, N, scale=3.0)
    inst = SoftmaxBlock.newInstance(M, N, init_tensor(x, [M, N]), True)
    assert tuple(inst["resultBuffer"].dims) == (N, M)
    got = run(inst, (N, M))
    plain = run(SoftmaxBlock.newInstance(M, N, init_tensor(x, [M, N])), (M, N))
    assert np.array_equal(got, plain.T)
    want = ref.softmax(x).T
    assert close(got, want, atol=1e-7), worst(got, want, atol=1e-7)


def test_chunked_vocabulary_buffers_as_the_reference_builds_them(device):
    """The reference holds the table as zero-padded chunks: [chunk, d] copies for the gather and host-transposed
    [d, chunk] copies for the de-embedding (model.js:298-364; 50257 rows -> two chunks of 25132). Both blocks accept
    such lists and give the single-table results bit for bit."""
    V, d, T, ctx, chunk = 50257, 768, 9, 32, 25132
    wte, wpe = rnd(V, d, scale=0.02), rnd(ctx, d, scale=0.02)
    padded = np.zeros((2 * chunk, d), np.float32)
    padded[:V] = wte
    gather = [init_tensor(padded[i * chunk:(i + 1) * chunk], [chunk, d]) for i in range(2)]
    transposed = [init_tensor(np.ascontiguousarray(padded[i * chunk:(i + 1) * chunk].T), [d, chunk]) for i in range(2)]
    idx = np.array([0, V - 1, 17, 17, 25131, 25132, 40000, 3, 50256], np.int32)
    wte_b, wpe_b = init_tensor(wte, [V, d]), init_tensor(wpe, [ctx, d])
    inst = EmbedBlock.newInstance(idx, T, d, chunk, gather, wpe_b, ResidualBlock)
    assert sum(p["flag"] == "copy" for p in inst["passes"]) == T + 1          # instructions.js:795-819
    got = run(inst, (T, d))
    assert np.array_equal(got, ref.embed(idx, wte, wpe))
    assert np.array_equal(got, run(EmbedBlock.newInstance(idx, T, d, V, [wte_b], wpe_b, ResidualBlock), (T, d)))
    x = rnd(T, d)
    x_b = init_tensor(x, [T, d])
    single = run(DeEmbedBlock.newInstance(d, V, V, T, V, x_b, [wte_b]), (V,))
    for _ in range(2):   # the second instance finds the chunks' row form already made
        inst = DeEmbedBlock.newInstance(d, V, 2 * chunk, T, chunk, x_b, transposed)
        assert [p["flag"] for p in inst["passes"]] == ["compute", "copy"] * 2      # instructions.js:858-882
        got = run(inst, (V,))
        assert np.array_equal(got, single)
    want = ref.deembed(x, wte)
    assert close(got, want), worst(got, want)
    with pytest.raises(ValueError, match="outside"):
        EmbedBlock.newInstance(np.array([2 * chunk], np.int32), 1, d, chunk, gather, wpe_b, ResidualBlock)
    for b in gather + transposed + [wte_b, wpe_b, x_b]:
        b.destroy()
    blocks.clearOperationCache()


def test_embed_and_deembed(device):
    V, d, T, ctx = 50257, 768, 9, 32
    wte, wpe = rnd(V, d, scale=0.02), rnd(ctx, d, scale=0.02)
    idx = np.array([0, V - 1, 17, 17, 25131, 25132, 40000, 3, 50256], np.int32)
    wte_b, wpe_b = init_tensor(wte, [V, d]), init_tensor(wpe, [ctx, d])
    got = run(EmbedBlock.newInstance(idx, T, d, V, [wte_b], wpe_b, ResidualBlock), (T, d))
    assert np.array_equal(got, ref.embed(idx, wte, wpe))
    x = rnd(T, d)
    got = run(DeEmbedBlock.newInstance(d, V, V, T, V, init_tensor(x, [T, d]), [wte_b]), (V,))
    want = ref.deembed(x, wte)
    assert close(got, want), worst(got, want)
    with pytest.raises(WgptError, match="outside"):
        run_passes(EmbedBlock.newInstance(np.array([V], np.int32), 1, d, V, [wte_b], wpe_b, ResidualBlock)["passes"])
    blocks.clearOperationCache()


def test_deembed_ragged_vocab(device):
    V, d, T = 65, 384, 3
    wte, x = rnd(V, d), rnd(T, d)
    got = run(DeEmbedBlock.newInstance(d, V, 68, T, 68, init_tensor(x, [T, d]), [init_tensor(wte, [V, d])]), (V,))
    want = ref.deembed(x, wte)
    assert close(got, want), worst(got, want)


@pytest.mark.parametrize("T,H,hs", [(1, 2, 8), (15, 4, 32), (64, 6, 64), (130, 12, 64), (5, 2, 4), (33, 25, 64), (20, 3, 64), (300, 2, 64)])
def test_attention(device, T, H, hs):
    d = H * hs
    x = rnd(T, d)
    W = [rnd(d, d, scale=0.5 / math.sqrt(d)) for _ in range(4)]
    b = [rnd(d, scale=0.1) for _ in range(4)]
    scale = 1 / math.sqrt(hs)
    bufs = [init_tensor(x, [T, d])]
    for i in range(4):
        bufs += [init_tensor(W[i], [d, d]), init_tensor(b[i], [d])]
    got = run(AttentionBlock.newFusedInstance(T, d, scale, H, hs, *bufs, FastMatMulBlock, SoftmaxBlock), (T, d))
    want = ref.attention(x, W[0], b[0], W[1], b[1], W[2], b[2], W[3], b[3], H)
    assert close(got, want), worst(got, want)


@pytest.mark.parametrize("T,H,hs", [(192, 2, 4), (192, 12, 4), (191, 14, 8), (1152, 2, 16), (193, 2, 20), (320, 5, 32), (257, 2, 36), (700, 2, 64), (225, 2, 68), (331, 4, 96),
                                    (256, 2, 100), (1023, 2, 128)])
def test_attention_split_operands(device, T, H, hs):
    """Prompts long enough for the split operands: the edges of a block of 32 queries, keys or dimensions. With the identity as
    every weight, q = k = v = x; scores reach 20 (the diagonal), so that maxima move from tile to tile. Products and sums of
    the scores are rounded like fp32 ones: an error of a few ulp of the largest score, 2**-20 of the weights at most, and
    2**-23 for each of the few roundings behind them. Infinite and other special values reach the rows that see them, and no others."""
    d = H * hs
    rng = np.random.default_rng(T + d)
    x = rng.standard_normal((T, d)).astype(np.float32)
    special = x.copy()
    special[T - 2, 0], special[T - 1, 1] = np.inf, np.nan
    eye, zero = np.eye(d, dtype=np.float32), np.zeros(d, np.float32)
    scale = 1 / math.sqrt(hs)
    got = []
    for values in (x, special):
        bufs = [init_tensor(values, [T, d])]
        for i in range(4):
            bufs += [init_tensor(eye, [d, d]), init_tensor(zero, [d])]
        got.append(run(AttentionBlock.newFusedInstance(T, d, scale, H, hs, *bufs, FastMatMulBlock, SoftmaxBlock), (T, d)))
    v = x.astype(np.float64).reshape(T, H, hs).transpose(1, 0, 2)
    s = v @ v.transpose(0, 2, 1) * np.float64(np.float32(scale))
    s[:, np.triu(np.ones((T, T), bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want = (p @ v).transpose(1, 0, 2).reshape(T, d)
    size = (p @ np.abs(v)).transpose(1, 0, 2).reshape(T, d)
    bound = (2.0 ** -20 * max(1.0, np.abs(s[np.isfinite(s)]).max() / 16) + 2.0 ** -21) * size
    assert np.all(np.abs(got[0] - want) <= bound)
    assert np.all(np.abs(got[1] - want)[:T - 2] <= bound[:T - 2])  # (a block with such rows is taken again without splits: other roundings)
    assert not np.isfinite(got[1][T - 2]).any() and not np.isfinite(got[1][T - 1]).any()


@pytest.mark.parametrize("T,H,hs,where", [(943, 12, 48, "key"), (943, 12, 48, "value"), (300, 8, 128, "key"), (943, 4, 32, "last")])
def test_attention_split_not_finite_in_time(device, T, H, hs, where):
    """A NaN in the first key, an infinity in the first value (every query takes its output again, to the end) and a NaN in the
    last key: less than eight times the time of a call without (measured: 2.0 to 3.2; 100 to 710 with a loop over the keys
    for each output)."""
    d = H * hs
    x = rnd(T, d)
    eye, zero = np.eye(d, dtype=np.float32), np.zeros(d, np.float32)
    ms = []
    for special in (False, True):
        v = x.copy()
        bias = zero
        if special and where == "value":  # (scores stay finite: the infinity comes in with the values' bias)
            bias = zero.copy()
            bias[::hs] = np.inf
        elif special:
            v[0 if where == "key" else T - 1, 0] = np.nan
        bufs = [init_tensor(v, [T, d])]
        for b in (zero, zero, bias, zero):
            bufs += [init_tensor(eye, [d, d]), init_tensor(b, [d])]
        inst = AttentionBlock.newFusedInstance(T, d, 1 / math.sqrt(hs), H, hs, *bufs, FastMatMulBlock, SoftmaxBlock)
        ms.append(_launch_ms(inst, 10))
        blocks.clearOperationCache()
    assert ms[1] < 8 * ms[0], ms


@pytest.mark.parametrize("T,H,hs", [(300, 4, 20), (2200, 3, 64), (2300, 4, 36), (400, 3, 96), (400, 2, 128)])
def test_attention_split_infinite_values(device, T, H, hs):
    """Operands that have no split although the outputs are finite: a key whose scores are -inf (its weight is zero), values next
    to the largest float; and an infinite value, for the queries from its own on. Context of more than 2048 keys among
    them. They come out of the projections: the last three columns of x are zero but for one row each, and meet 2**70."""
    d = H * hs
    rng = np.random.default_rng(T + d)
    x = rng.standard_normal((T, d)).astype(np.float32)
    x[:, 0] = np.abs(x[:, 0]) + 0.1
    x[:, d - 3:] = 0
    x[5, d - 3], x[9, d - 2], x[T - 2, d - 1] = 2.0 ** 70, np.float32(3.4e38) * np.float32(2.0 ** -70), 2.0 ** 70
    wq, wo, zero = np.eye(d, dtype=np.float32), np.eye(d, dtype=np.float32), np.zeros(d, np.float32)
    wq[d - 3:] = 0
    wk, wv = wq.copy(), wq.copy()
    wk[d - 3, 0] = -2.0 ** 70       # key 5 of head 0: -inf in dimension 0
    wv[d - 2, hs + 2] = 2.0 ** 70   # value 9 of head 1: 3.4e38 in dimension 2
    wv[d - 1, hs + 3] = 2.0 ** 70   # value T - 2 of head 1: inf in dimension 3
    bufs = [init_tensor(x, [T, d])]
    for w in (wq, wk, wv, wo):
        bufs += [init_tensor(w, [d, d]), init_tensor(zero, [d])]
    scale = 1 / math.sqrt(hs)
    got = run(AttentionBlock.newFusedInstance(T, d, scale, H, hs, *bufs, FastMatMulBlock, SoftmaxBlock), (T, d))
    with np.errstate(all="ignore"):
        heads = lambda w: (x.astype(np.float64) @ w).reshape(T, H, hs).transpose(1, 0, 2)
        q, k, v = heads(wq), heads(wk), heads(wv)
        v[1, 9, 2] = np.float32(3.4e38)
        k[0, 5, 0] = 0
        s = q @ k.transpose(0, 2, 1) * np.float64(np.float32(scale))
        s[0, :, 5] = -np.inf
        s[:, np.triu(np.ones((T, T), bool), 1)] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        v[1, T - 2, 3] = 0
        want = (p @ v).transpose(1, 0, 2).reshape(T, d)
        size = (p @ np.abs(v)).transpose(1, 0, 2).reshape(T, d)
        # a score is a sum of hs products in any order of up to eight roundings, and is rounded once more with the scale and the
        # maximum: an absolute error e, which is the relative one of its weight; value 9 makes single weights visible. The
        # sums over the keys: a run of at most T / 32 additions in a lane, and a few between lanes.
        e = 2.0 ** -24 * (8 * (np.abs(q) @ np.abs(k).transpose(0, 2, 1)) * scale + 2 * np.abs(np.where(np.isfinite(s), s, 0)) + 8)
        pe = p * e
        bound = (pe @ np.abs(v) + pe.sum(-1, keepdims=True) * (p @ np.abs(v))).transpose(1, 0, 2).reshape(T, d) + 2.0 ** -24 * (T / 32 + 16) * size + 1e-30
    ratio = (np.abs(got - want) / bound)[:T - 2]
    assert np.all(ratio <= 1), (float(ratio.max()), np.unravel_index(ratio.argmax(), ratio.shape))
    assert not np.isfinite(got[T - 2:]).any()  # (the projection behind it spreads an infinite output over its row)


@pytest.mark.parametrize("small", ["all", "dimension"])
@pytest.mark.parametrize("T,H,hs", [(193, 2, 20), (700, 2, 64), (331, 4, 96), (1023, 2, 128)])
def test_attention_split_tiny_values(device, T, H, hs, small):
    """Values around 2**-119, all of them or those of one dimension, whose third bf16 part is too small for bf16: the relative
    error of test_attention_split_operands, and for each key a quantum of 2**-149."""
    d = H * hs
    rng = np.random.default_rng(T + d)
    x = rng.standard_normal((T, d)).astype(np.float32)
    eye, zero = np.eye(d, dtype=np.float32), np.zeros(d, np.float32)
    wv = eye.copy()
    if small == "all":
        wv *= np.float32(2.0 ** -119)
    else:
        wv[hs + 3, hs + 3] = 2.0 ** -119
    bufs = [init_tensor(x, [T, d])]
    for w in (eye, eye, wv, eye):
        bufs += [init_tensor(w, [d, d]), init_tensor(zero, [d])]
    scale = 1 / math.sqrt(hs)
    got = run(AttentionBlock.newFusedInstance(T, d, scale, H, hs, *bufs, FastMatMulBlock, SoftmaxBlock), (T, d)).astype(np.float64)
    k = x.astype(np.float64).reshape(T, H, hs).transpose(1, 0, 2)
    v = (x.astype(np.float64) * np.diag(wv)).reshape(T, H, hs).transpose(1, 0, 2)
    s = k @ k.transpose(0, 2, 1) * np.float64(np.float32(scale))
    s[:, np.triu(np.ones((T, T), bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want = (p @ v).transpose(1, 0, 2).reshape(T, d)
    size = (p @ np.abs(v)).transpose(1, 0, 2).reshape(T, d)
    bound = (2.0 ** -20 * max(1.0, np.abs(s[np.isfinite(s)]).max() / 16) + 2.0 ** -21) * size + T * 2.0 ** -149
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))


@pytest.mark.parametrize("below,exponent", [(83, 30), (83, 80), (88, 40), (88, 100)])
@pytest.mark.parametrize("T,H,hs", [(193, 2, 20), (700, 2, 64), (331, 4, 96), (1023, 2, 128)])
def test_attention_split_tiny_weights(device, T, H, hs, below, exponent):
    """Weights of 2**-124 to 2**-119 (scores 83 to 86 below the first key's, whose value is zero), whose third bf16 part is too
    small for bf16, on values around 2**30 and 2**80: the outputs are not tiny themselves. Scores are exact here and all terms
    positive: a few roundings for a weight and the quotient, and one for each of the at most T / 8 keys that are added up in a row
    (2**-12 with the third parts lost). Scores 88 to 91 below: weights are subnormal, within 2**-149 (2**-17 of them), and not zero."""
    d = H * hs
    rng = np.random.default_rng(T + d)
    x = (rng.uniform(1, 2, (T, d)) * 2.0 ** exponent).astype(np.float32)
    x[0] = 0
    x[1:, ::hs] = -rng.integers(below * 64, (below + 3) * 64, (T - 1, H)) / np.float32(64)  # the scores: q is 1 in the first dimension, else 0
    eye, none, zero = np.eye(d, dtype=np.float32), np.zeros((d, d), np.float32), np.zeros(d, np.float32)
    bq = zero.copy()
    bq[::hs] = 1
    bufs = [init_tensor(x, [T, d])]
    for w, b in ((none, bq), (eye, zero), (eye, zero), (eye, zero)):
        bufs += [init_tensor(w, [d, d]), init_tensor(b, [d])]
    got = run(AttentionBlock.newFusedInstance(T, d, 1.0, H, hs, *bufs, FastMatMulBlock, SoftmaxBlock), (T, d)).astype(np.float64)
    weights = np.exp(x[:, ::hs].astype(np.float64))
    for h in range(H):
        want = np.cumsum(weights[:, h:h + 1] * x[:, h * hs + 1:(h + 1) * hs], 0) / np.cumsum(weights[:, h:h + 1], 0)
        error = np.abs(got[:, h * hs + 1:(h + 1) * hs] - want)
        assert np.all(error <= (2.0 ** -24 * (T / 8 + 16) + (2.0 ** -17 if below > 87 else 0)) * want), float(np.max(error[1:] / want[1:]))


def test_attention_values_known_answer(device):
    # other/test.js:370-388 through the attention block: with Wq = Wk = 0 every score is 0, so the
    # softmax is uniform over j <= i: P = 1/(i+1). V = c // hs + 1 (via bv, Wv = 0), Wo = I:
    # O[i, c] = sum_{j<=i} (1/(i+1)) * (c // hs + 1) = c // hs + 1.
    T, d, H = 15, 128, 4
    hs = d // H
    z = np.zeros((d, d), np.float32)
    zb = np.zeros(d, np.float32)
    vrow = (np.arange(d) // hs + 1).astype(np.float32)
    bufs = [init_tensor(rnd(T, d), [T, d]), init_tensor(z, [d, d]), init_tensor(zb, [d]), init_tensor(z, [d, d]),
            init_tensor(zb, [d]), init_tensor(z, [d, d]), init_tensor(vrow, [d]),
            init_tensor(np.eye(d, dtype=np.float32), [d, d]), init_tensor(zb, [d])]
    got = run(AttentionBlock.newFusedInstance(T, d, 1 / math.sqrt(hs), H, hs, *bufs), (T, d))
    assert np.allclose(got, np.tile(vrow, (T, 1)), rtol=1e-6)


@pytest.mark.parametrize("M,N,K", [(1, 8, 4), (1, 1600, 1600), (1, 4800, 1600), (1, 1600, 6400), (3, 264, 100), (40, 136, 64), (130, 264, 100), (300, 4800, 1600), (512, 1600, 6400)])
def test_int8_matmul_and_bit_exact_dequant(device, M, N, K):
    A = rnd(M, K)
    q = RNG.integers(-127, 128, (K, N))
    q[0, :4] = [-128, 127, -1, 0]
    packed = pack_words(q)
    scale = RNG.uniform(1e-3, 1e-2, N).astype(np.float32)
    bias = rnd(N)
    pk, sc = init_tensor(packed, [K, N // 4]), init_tensor(scale, [N])
    # dequantised weights: bit-exact
    wbuf = blocks.Buffer([K, N])
    from webgpt_amd import _lib
    _lib.call("wgpt_dequant_i8", K, N, pk.handle, sc.handle, wbuf.handle)
    W = wbuf.download().reshape(K, N)
    wbuf.destroy()
    want_w = ref.dequant_i8(packed, scale, N)
    assert np.array_equal(W.view(np.uint32), want_w.view(np.uint32))
    inst = FastMatMulBlock.newInt8Instance(M, N, K, init_tensor(A, [M, K]), pk, sc, init_tensor(bias, [N]))
    got = run(inst, (M, N))
    want = ref.matmul_i8(A, packed, scale, bias)
    assert close(got, want), worst(got, want)


def test_int8_dequant_all_bytes(device):
    from webgpt_amd import _lib
    scales = np.array([1e-3, 9.999e-3, 0.0123456, 1.0, 3.1415927, 1e-8, 127.0, 5.5e-3], np.float32)
    q = np.repeat(np.arange(-128, 128)[:, None], 8, axis=1)
    packed = pack_words(q)
    pk, sc, out = init_tensor(packed, [256, 2]), init_tensor(scales, [8]), blocks.Buffer([256, 8])
    _lib.call("wgpt_dequant_i8", 256, 8, pk.handle, sc.handle, out.handle)
    got = out.download().reshape(256, 8)
    want = (q.astype(np.float32) / np.float32(127.0)) * scales[None, :]
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(got.view(np.uint32), ref.dequant_i8(packed, scales, 8).view(np.uint32))
