"""chatnet_matmul with several columns against float64 products of the oracle's
dequantized weights, at the edges of each path: a few columns in one launch
(multi-column GEMV), the matrix-core paths from 8 columns on, non-finite
values, a capturing stream and the no-allocation variant."""
import threading

import numpy as np
import pytest

import oracle
from chatnet_amd import _native, hiprt, ops, synth
from gpu_util import announce, gpu_matmul, normwise, run_with_failing_malloc

pytestmark = pytest.mark.gpu

F32, F16 = 0, 1


def float_weights(qtype, M, K, seed):
    w = synth.normal(seed, f"fc{M}x{K}", M * K, 0.05).reshape(M, K)
    return w.astype(np.float16) if qtype == F16 else w


# Groups of columns whose fp32 x fits in LDS: 8 up to K = 4864, 3 at 11008, 2 at
# 16384; tiles of 32 and 64 columns and ragged rows for the F16 product.
@pytest.mark.parametrize("M,K,N", [
    (1, 64, 2), (3, 192, 7), (130, 4096, 5), (37, 11008, 7), (65, 16384, 3), (5, 64, 8), (129, 4096, 33), (200, 320, 64),
    (4096, 4096, 24), (66, 16384, 12), (1000, 2048, 300),
])
@pytest.mark.parametrize("qtype", [F32, F16])
def test_float_columns_match_float64(qtype, M, K, N):
    """Bar: 32-bit sums in any order, |error| <= K * 2^-24 of sum |w x| at worst
    (the F16 product's x is exact down to 2^-28 of its column's largest); measured
    about 1e-7 of the largest output."""
    announce(f"float columns type={qtype} M={M} K={K} N={N}")
    w = float_weights(qtype, M, K, 5)
    x = synth.normal(6, f"fcx{N}x{K}", N * K, 1.0).reshape(N, K)
    x[:, 0] *= 300.0
    y = gpu_matmul(qtype, w.view(np.uint8).ravel(), x, M, K)
    r = x.astype(np.float64) @ w.astype(np.float64).T
    scale = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert np.all(np.abs(y - r) <= 2e-6 * scale), float(np.max(np.abs(y - r) / scale))
    if qtype == F32 or N * K * 4 <= 152 * 1024 and N <= 8:  # one GEMV launch: each column the single-column result
        for n in range(N):
            assert np.array_equal(y[n], gpu_matmul(qtype, w.view(np.uint8).ravel(), x[n], M, K)[0])


def test_f16_columns_of_other_magnitudes_and_non_finite_values():
    """Columns far outside fp16's range keep their accuracy; infinities and NaN in
    x or W give what the single-column product gives."""
    M, K, N = 70, 256, 12
    w = float_weights(F16, M, K, 7)
    w[3, 5], w[4, 6], w[5, 7] = np.inf, -np.inf, np.nan
    x = synth.normal(8, "fcx-mag", N * K, 1.0).reshape(N, K).astype(np.float64)
    x *= np.array([1e-30, 1e-12, 3e-5, 1e-3, 0.5, 1.0, 7.0, 6e4, 1e8, 1e20, 1e30, 0.0])[:, None]
    x = x.astype(np.float32)
    x[5, 9], x[6, 10], x[7, 11] = np.inf, -np.inf, np.nan
    x[4, 5] = 0.25  # an exact fp16 value against the infinite weight: its low part is zero
    announce("f16 columns, magnitudes and non-finite values")
    y = gpu_matmul(F16, w.view(np.uint8).ravel(), x, M, K)
    for n in range(N):
        one = gpu_matmul(F16, w.view(np.uint8).ravel(), x[n], M, K)[0]
        fin = np.isfinite(one)
        assert np.array_equal(fin, np.isfinite(y[n])), n
        assert np.array_equal(np.isnan(one), np.isnan(y[n])), n
        assert np.array_equal(one[~fin & ~np.isnan(one)], y[n][~fin & ~np.isnan(one)]), n
        if fin.any():
            assert normwise(y[n][fin], one[fin]) <= 2e-6, n


@pytest.mark.parametrize("M,K,N", [(512, 512, 12), (100, 4096, 40), (64, 11008, 5), (4096, 4096, 70)])
def test_f16_columns_hold_x_in_fp32(M, K, N):
    """Against single ones the product is x itself, all 24 bits, also beside an
    element 2^20 times larger under zero weights; beside one 2^30 times larger, to
    2^-50 of it (the matrix cores align the terms of a sum to about 2^-52 of the
    largest operand there)."""
    announce(f"f16 columns, x exact M={M} K={K} N={N}")
    at = (np.arange(M) * 7 + 1) % (K - 1) + 1
    w = np.zeros((M, K), np.float16)
    w[np.arange(M), at] = 1.0
    x = synth.normal(57, f"exx{N}x{K}", N * K, 1.0).reshape(N, K)
    x += np.copysign(np.float32(0.125), x)
    for big, tol in ((1.0, 0.0), (2.0 ** 20, 0.0), (2.0 ** 30, 2.0 ** -20)):
        x[:, 0] = big
        assert np.max(np.abs(gpu_matmul(F16, w.view(np.uint8).ravel(), x, M, K) - x[:, at])) <= tol, big


@pytest.mark.parametrize("M,K,N", [(96, 512, 16), (96, 512, 3)])
def test_f16_columns_captured_without_a_workspace_and_noalloc(M, K, N):
    """F16 rows take no workspace they cannot have: a captured call on a stream
    with or without a workspace, and the no-allocation variant, run the
    multi-column GEMV, each column the single-column result."""
    announce(f"f16 captured M={M} K={K} N={N}")
    w = float_weights(F16, M, K, 9)
    x = synth.normal(9, "fcx-cap", N * K, 1.0).reshape(N, K)
    ref = np.stack([gpu_matmul(F16, w.view(np.uint8).ravel(), x[n], M, K)[0] for n in range(N)])
    w_d = hiprt.DeviceBuffer.from_numpy(w.view(np.uint8).ravel(), pad=256)
    x_d, y_d = hiprt.DeviceBuffer.from_numpy(x), hiprt.DeviceBuffer(4 * N * M)
    stream = hiprt.Stream()
    ops.matmul_ptr(F16, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, stream.h)  # the stream has a workspace
    stream.synchronize()
    graph = hiprt.Graph(stream, lambda: ops.matmul_ptr(F16, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, stream.h))
    for _ in range(2):
        y_d.fill(0xFF)
        hiprt.synchronize()
        graph.launch()
        stream.synchronize()
        assert np.array_equal(y_d.to_numpy(np.float32, N * M).reshape(N, M), ref)
    y_d.fill(0xFF)
    hiprt.synchronize()
    lib = _native.hip_lib()
    _native.check(lib.chatnet_matmul_noalloc(F16, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, stream.h))
    stream.synchronize()
    assert np.array_equal(y_d.to_numpy(np.float32, N * M).reshape(N, M), ref)
    del graph
    for b in (w_d, x_d, y_d):
        b.free()


BLOCK_TYPES = {3: "q4_1", 6: "q5_0", 7: "q5_1", 8: "q8_0", 10: "q2_k", 11: "q3_k", 12: "q4_k", 13: "q5_k", 14: "q6_k",
               20: "iq4_nl", 23: "iq4_xs"}
FINE_TYPES = (3, 6, 7, 10, 20, 23)  # up to 7 columns: x in fp32


def digit_bound(qtype, x, w):
    """32 roundings of 2^-24 of sum |w x| for the 32-bit sums and, where x is held
    in digits, half a step of them in every element: a step is at most 2^-29 of
    its 32-element block's maximum in the matrix-core product (from 2 columns on,
    fine types 8), 2^-18 of its group's (of 16 or 32 elements) in the GEMV."""
    N = x.shape[0]
    ax = np.abs(x).astype(np.float64)
    bound = 32 * 2.0 ** -24 * (ax @ np.abs(w).T)
    if qtype in FINE_TYPES and N < 8:
        return bound
    g = np.repeat(ax.reshape(N, -1, 32).max(2), 32, axis=1)
    return bound + 0.5 * (2.0 ** -18 if N == 1 else 2.0 ** -29) * (g @ np.abs(w).T)


# One column (the GEMV), then one to four tiles of digit rows (4 columns each), one
# and two row tiles per wave (from 4097 rows), several
# row groups per workgroup (over 16384 rows), rows whose x is staged in several
# rounds, ahead of the launch or in the workgroup, and ragged last row tiles.
@pytest.mark.parametrize("M,K,N", [
    (1, 256, 1), (3, 512, 2), (130, 4096, 7), (37, 11008, 1), (37, 11008, 5), (65, 16384, 3), (8200, 768, 4),
    (4100, 5120, 2), (5, 2304, 1), (17, 256, 6), (70, 1024, 10), (4200, 512, 8), (130, 2304, 16), (33, 7936, 11),
    (17000, 256, 3),
])
@pytest.mark.parametrize("qtype", sorted(BLOCK_TYPES))
def test_block_types_few_columns_match_float64(qtype, M, K, N):
    """Every column against the float64 product of the dequantized weights, within
    digit_bound; from two columns on also 6e-7 in the 2-norm (1e-7 to 3e-7 from the
    32-bit sums; x at 19 bits gave 4e-6)."""
    announce(f"few columns {BLOCK_TYPES[qtype]} M={M} K={K} N={N}")
    t = synth.tensor(qtype, 31, f"few{qtype}-{M}x{K}", M, K)
    x = synth.normal(32, f"fewx{N}x{K}", N * K, 1.0).reshape(N, K)
    x[:, K // 2] *= 20.0
    y = gpu_matmul(qtype, t.data, x, M, K)
    w = oracle.dequant(qtype, t.data, M * K).reshape(M, K).astype(np.float64)
    r = x.astype(np.float64) @ w.T
    bound = digit_bound(qtype, x, w)
    assert np.all(np.abs(y - r) <= bound), float(np.max(np.abs(y - r) / bound))
    if N >= 2:
        assert np.linalg.norm(y - r) <= 6e-7 * np.linalg.norm(r), float(np.linalg.norm(y - r) / np.linalg.norm(r))


@pytest.mark.parametrize("qtype", sorted(BLOCK_TYPES))
def test_up_to_sixteen_columns_of_any_length_keep_their_precision(qtype):
    """10 and 11 columns, K = 8192 and beyond, K shared over workgroups and not:
    digit_bound and 6e-7 in the 2-norm up to 16 columns (fp16 operands, from 17 on,
    give 3e-4)."""
    for (M, K, N) in [(33, 8192, 16), (33, 8448, 10), (33, 8448, 11), (2100, 8448, 16), (37, 11008, 11), (20, 16384, 16)]:
        announce(f"long rows {BLOCK_TYPES[qtype]} M={M} K={K} N={N}")
        t = synth.tensor(qtype, 55, f"long{qtype}-{M}x{K}", M, K)
        x = synth.normal(56, f"longx{N}x{K}", N * K, 1.0).reshape(N, K)
        y = gpu_matmul(qtype, t.data, x, M, K)
        w = oracle.dequant(qtype, t.data, M * K).reshape(M, K).astype(np.float64)
        r = x.astype(np.float64) @ w.T
        assert np.all(np.abs(y - r) <= digit_bound(qtype, x, w))
        assert np.linalg.norm(y - r) <= 6e-7 * np.linalg.norm(r)


def test_odd_rows_of_short_k_match_float64():
    """K = 64 and 192: one pair of blocks, and rows whose records end mid-unit."""
    for qtype in (3, 6, 7, 8, 20):
        for (M, K, N) in [(1, 64, 1), (70, 64, 3), (33, 192, 5), (64, 960, 2)]:
            announce(f"short rows {BLOCK_TYPES[qtype]} M={M} K={K} N={N}")
            t = synth.tensor(qtype, 33, f"short{qtype}-{M}x{K}", M, K)
            x = synth.normal(34, f"shortx{N}x{K}", N * K, 1.0).reshape(N, K)
            y = gpu_matmul(qtype, t.data, x, M, K)
            w = oracle.dequant(qtype, t.data, M * K).reshape(M, K).astype(np.float64)
            assert np.all(np.abs(y - x.astype(np.float64) @ w.T) <= digit_bound(qtype, x, w))


@pytest.mark.parametrize("qtype", [3, 6, 7, 10, 20, 23])
@pytest.mark.parametrize("N", [1, 3])
def test_non_finite_x_and_wide_magnitudes(qtype, N):
    """A column with an infinity or NaN gives no finite output (the packed-unit
    product these types ran before met it in fp32); columns of 1e30 and 1e-30
    keep their accuracy."""
    M, K = 40, 512
    t = synth.tensor(qtype, 35, f"nf{qtype}", M, K)
    w = oracle.dequant(qtype, t.data, M * K).reshape(M, K).astype(np.float64)
    for bad in (np.inf, -np.inf, np.nan):
        x = synth.normal(36, "nfx", N * K, 1.0).reshape(N, K)
        x[N - 1, 77] = bad
        y = gpu_matmul(qtype, t.data, x, M, K)
        assert not np.any(np.isfinite(y[N - 1]))
        assert np.all(np.isfinite(y[: N - 1]))
    for mag in (1e30, 1e-30):
        x = (synth.normal(37, "nfy", N * K, 1.0) * mag).reshape(N, K).astype(np.float32)
        y = gpu_matmul(qtype, t.data, x, M, K)
        r = x.astype(np.float64) @ w.T
        assert max(normwise(y[n], r[n]) for n in range(N)) <= 2e-6


def smallest_weights_at(qtype, t, M, K, k):
    """The tensor's bytes with the weight of column k (5, 15 or 10 in its block: a
    low nibble, or Q2_K's lowest field) of every row at its type's smallest
    magnitude: 0, or the table's 1 (IQ4)."""
    n, size = (256, {10: 84, 23: 136}[qtype]) if qtype in (10, 23) else (32, {3: 20, 6: 22, 7: 24, 20: 18}[qtype])
    b = t.data.reshape(M, K // n, size).copy()
    j, blk = k % n, b[:, k // n]
    if qtype == 3:
        b[:, :, 2:4] = 0
        blk[:, 4 + j] &= 0xF0
    elif qtype == 6:
        blk[:, 6 + j] &= 0xF0
        blk[:, 2 + j // 8] |= 1 << (j % 8)
    elif qtype == 7:
        b[:, :, 2:4] = 0
        blk[:, 8 + j] &= 0xF0
        blk[:, 4 + j // 8] &= 0xFF ^ (1 << (j % 8))
    elif qtype == 20:
        blk[:, 2 + j] = (blk[:, 2 + j] & 0xF0) | 8
    elif qtype == 10:
        b[:, :, 82:84] = 0
        blk[:, 16 + j] &= 0xFC
    else:
        blk[:, 8 + j] = (blk[:, 8 + j] & 0xF0) | 8
    return b.reshape(-1)


# One column and several: 16, 32 and 64 lanes a row, one to four units a lane, rows
# past the grid's first turn, groups of columns (3 and 2 at 11008 and 16384); the
# outlier in a group's first and last quarter.
@pytest.mark.parametrize("M,K,k,N", [
    (40, 512, 5, 1), (9, 11008, 10 + 512, 1), (6, 16384, 5, 1), (33, 768, 256 + 15, 2), (40, 512, 5, 7), (9, 11008, 10, 4),
    (6, 16384, 5, 3), (9000, 2304, 256 + 15, 7), (70, 4096, 5, 5), (33, 8192, 5, 2),
])
@pytest.mark.parametrize("qtype", FINE_TYPES)
def test_fp32_types_keep_the_neighbours_of_a_large_element(qtype, M, K, k, N):
    """x is fp32 for these types: an element of 1e5 under a zero (or the smallest)
    weight leaves its neighbours' bits alone.  digit_bound's 32 roundings: a group's
    16 products, the groups of a lane, the lanes."""
    announce(f"large element {BLOCK_TYPES[qtype]} M={M} K={K} N={N}")
    data = smallest_weights_at(qtype, synth.tensor(qtype, 51, f"out{qtype}-{M}x{K}", M, K), M, K, k)
    x = synth.normal(52, f"outx{N}x{K}", N * K, 1.0).reshape(N, K)
    x[:, k] = 1e5
    w = oracle.dequant(qtype, data, M * K).reshape(M, K).astype(np.float64)
    y = gpu_matmul(qtype, data, x, M, K)
    bound = digit_bound(qtype, x, w)
    err = np.abs(y - x.astype(np.float64) @ w.T)
    assert np.all(err <= bound), float(np.max(err / bound))


@pytest.mark.parametrize("N", [2, 5, 12, 16])
@pytest.mark.parametrize("qtype", [8, 11, 12, 13, 14])
def test_a_large_element_leaves_the_other_half_of_its_block(qtype, N):
    """An element of 1e5 whose 16-element group has zero weights: the other group of
    the 32-element block keeps at least the single-column GEMV's 19 bits of its own
    16 elements."""
    M, K = 40, 512
    announce(f"large element, other half {BLOCK_TYPES[qtype]} N={N}")
    t = synth.tensor(qtype, 53, f"half{qtype}", M, K)
    n, size = (32, 34) if qtype == 8 else (256, {11: 110, 12: 144, 13: 176, 14: 210}[qtype])
    b = t.data.reshape(M, K // n, size).copy()
    if qtype == 8:
        b[:, 0, 2:18] = 0
    elif qtype == 11:  # 6-bit scale 32 (zero) of group 0
        b[:, 0, 96] &= 0xF0
        b[:, 0, 104] = (b[:, 0, 104] & 0xFC) | 2
    elif qtype == 14:
        b[:, 0, 192] = 0
    else:
        b[:, 0, 2:4] = 0  # dmin
        qs = 16 if qtype == 12 else 48
        b[:, 0, qs:qs + 16] &= 0xF0
        if qtype == 13:
            b[:, 0, 16:18] = 0
    x = synth.normal(54, f"halfx{N}", N * K, 1.0).reshape(N, K)
    x[:, 5] = 1e5
    w = oracle.dequant(qtype, b.reshape(-1), M * K).reshape(M, K).astype(np.float64)
    assert not w[:, :16].any()
    y = gpu_matmul(qtype, b.reshape(-1), x, M, K)
    g = np.repeat(np.abs(x).astype(np.float64).reshape(N, -1, 16).max(2), 16, axis=1)
    bound = (2.0 ** -18 * g + 32 * 2.0 ** -24 * np.abs(x)) @ np.abs(w).T
    err = np.abs(y - x.astype(np.float64) @ w.T)
    assert np.all(err <= bound), float(np.max(err / bound))


@pytest.mark.parametrize("M,same_order", [(2100, True), (96, False)])
@pytest.mark.parametrize("qtype", [12, 6])
def test_few_columns_captured_without_a_workspace_and_noalloc(qtype, M, same_order):
    """x staged ahead, and K shared over workgroups (few rows), need the stream's
    workspace: a capturing stream, whether it has one or not, and the no-allocation
    variant stage x in every workgroup, to the same bits, and sum K in one
    workgroup."""
    K, N = 4096, 9
    announce(f"few columns captured {BLOCK_TYPES[qtype]}")
    t = synth.tensor(qtype, 38, f"cap{qtype}", M, K)
    x = synth.normal(39, "capx", N * K, 1.0).reshape(N, K)
    ref = gpu_matmul(qtype, t.data, x, M, K)
    bound = np.zeros(ref.shape)
    if not same_order:  # 32-bit sums in another order
        w = oracle.dequant(qtype, t.data, M * K).reshape(M, K).astype(np.float64)
        bound = 16 * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    w_d = hiprt.DeviceBuffer.from_numpy(t.data, pad=256)
    x_d, y_d = hiprt.DeviceBuffer.from_numpy(x), hiprt.DeviceBuffer(4 * N * M)
    stream = hiprt.Stream()
    _native.check(_native.hip_lib().chatnet_matmul_noalloc(qtype, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, stream.h))
    stream.synchronize()
    alone = y_d.to_numpy(np.float32, N * M).reshape(N, M)
    assert np.all(np.abs(alone - ref) <= bound)
    y_d.fill(0xFF)
    ops.matmul_ptr(qtype, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, 2)  # hipStreamPerThread: one handle, many streams
    hiprt.synchronize()
    assert np.array_equal(y_d.to_numpy(np.float32, N * M).reshape(N, M), alone)
    y_d.fill(0xFF)
    ops.matmul_ptr(qtype, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, stream.h)  # the stream has a workspace
    stream.synchronize()
    assert np.array_equal(y_d.to_numpy(np.float32, N * M).reshape(N, M), ref)
    graph = hiprt.Graph(stream, lambda: ops.matmul_ptr(qtype, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, stream.h))
    for _ in range(2):
        y_d.fill(0xFF)
        hiprt.synchronize()
        graph.launch()
        stream.synchronize()
        assert np.array_equal(y_d.to_numpy(np.float32, N * M).reshape(N, M), alone)
    del graph
    for b in (w_d, x_d, y_d):
        b.free()


WITHOUT_MEMORY = """
import numpy as np
from chatnet_amd import _native, hiprt, ops, synth
lib = _native.hip_lib()
malloc_limit(1024)
for qtype, M, K, N in [(1, 96, 512, 16), (12, 96, 4096, 9), (8, 2100, 4096, 12), (12, 96, 512, 40)]:
    print("[gpu-case] no memory for a workspace", qtype, M, K, N, flush=True)
    w = (synth.normal(70, "w", M * K, 0.05).astype(np.float16).view(np.uint8) if qtype == 1
         else synth.tensor(qtype, 70, "w", M, K).data)
    w_d = hiprt.DeviceBuffer.from_numpy(w, pad=256)
    x_d = hiprt.DeviceBuffer.from_numpy(synth.normal(71, "x", N * K, 1.0))
    y, z = hiprt.DeviceBuffer(4 * N * M), hiprt.DeviceBuffer(4 * N * M)
    y.fill(0xFF)
    rc = lib.chatnet_matmul(qtype, w_d.ptr, x_d.ptr, y.ptr, M, K, N, None)
    assert rc == (0 if N <= 16 else _native.ERR_OUT_OF_MEMORY), rc  # the GEMM has no other path
    if rc == 0:
        _native.check(lib.chatnet_matmul_noalloc(qtype, w_d.ptr, x_d.ptr, z.ptr, M, K, N, None))
        hiprt.synchronize()
        assert np.array_equal(y.to_numpy(np.uint32, N * M), z.to_numpy(np.uint32, N * M))
"""


def test_without_memory_for_a_workspace(tmp_path):
    """Products that only gain by a workspace run without one where its allocation
    fails, with the no-allocation variant's bits; the GEMM reports the failure."""
    run_with_failing_malloc(tmp_path, WITHOUT_MEMORY)


def test_threads_on_shared_and_own_streams():
    """Four threads, two of them on one stream, each with products that use and grow
    the stream's workspace (a packing pass, K splits, F16 planes, K shares, x staged
    ahead): every result is the single call's."""
    announce("threads, shared and own streams")
    work = []
    for i, (qtype, M, K, N) in enumerate([(14, 300, 2048, 40), (F16, 512, 512, 24), (12, 96, 4096, 9), (8, 2100, 4096, 12),
                                          (12, 1000, 4096, 100), (18, 200, 512, 3)]):
        w = float_weights(qtype, M, K, 60).view(np.uint8).ravel() if qtype == F16 else synth.tensor(qtype, 60 + i, "thr", M, K).data
        x = synth.normal(61 + i, "thrx", N * K, 1.0).reshape(N, K)
        work.append((qtype, M, K, N, gpu_matmul(qtype, w, x, M, K), hiprt.DeviceBuffer.from_numpy(w, pad=256),
                     hiprt.DeviceBuffer.from_numpy(x)))
    shared = hiprt.Stream()
    streams = [shared, shared, hiprt.Stream(), hiprt.Stream()]
    outs = [[[hiprt.DeviceBuffer(4 * c[1] * c[3]) for c in work] for _ in range(3)] for _ in streams]
    errors = []

    def run(t):
        try:
            for r in range(3):
                for i in range(len(work)):
                    j = (i + t) % len(work)
                    qtype, M, K, N, _, w_d, x_d = work[j]
                    ops.matmul_ptr(qtype, w_d.ptr, x_d.ptr, outs[t][r][j].ptr, M, K, N, streams[t].h)
        except Exception as e:  # reported below, in the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(t,)) for t in range(len(streams))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    hiprt.synchronize()
    assert not errors, errors
    for per_thread in outs:
        for per_round in per_thread:
            for c, y in zip(work, per_round):
                assert np.array_equal(y.to_numpy(np.float32, c[1] * c[3]).reshape(c[3], c[1]), c[4])
                y.free()
    for c in work:
        c[5].free()
        c[6].free()


# Types whose GEMM reads the stored blocks: 32-, 64- and 128-column tiles, one
# chunk and odd chunk counts, K split and whole, single and ragged rows.
@pytest.mark.parametrize("M,K,N", [(1, 256, 17), (130, 768, 40), (67, 2304, 129), (300, 4096, 65), (2050, 512, 300)])
@pytest.mark.parametrize("qtype", [3, 6, 7, 8, 10, 12, 13, 20, 23])
def test_stored_block_gemm_edges(qtype, M, K, N):
    """Both operands meet in fp16, each rounded once: |error| <= 2 * 2^-11 (1 +
    2^-11) of sum |w x|, and the 32-bit sums' part far below."""
    announce(f"stored gemm {BLOCK_TYPES[qtype]} M={M} K={K} N={N}")
    t = synth.tensor(qtype, 41, f"sg{qtype}-{M}x{K}", M, K)
    x = synth.normal(42, f"sgx{N}x{K}", N * K, 1.0).reshape(N, K)
    y = gpu_matmul(qtype, t.data, x, M, K)
    w = oracle.dequant(qtype, t.data, M * K).reshape(M, K).astype(np.float64)
    r = x.astype(np.float64) @ w.T
    scale = np.abs(x).astype(np.float64) @ np.abs(w).T
    assert np.all(np.abs(y - r) <= 2.0 ** -10 * 1.01 * scale), float(np.max(np.abs(y - r) / scale))


# Q6_K and Q3_K re-encoded by a thread per 16 weights: one super-block, odd counts
# of them (rows starting on 2-byte boundaries), and a last workgroup partly filled.
@pytest.mark.parametrize("M,K,N", [(1, 256, 17), (3, 768, 17), (65, 2304, 40), (300, 4096, 129)])
@pytest.mark.parametrize("qtype", [11, 14])
def test_repacked_gemm_edges(qtype, M, K, N):
    """The bound of the stored blocks' test: one fp16 rounding of each operand."""
    test_stored_block_gemm_edges(qtype, M, K, N)


@pytest.mark.parametrize("N", [384, 385])
def test_q2_k_gemm_on_either_side_of_its_packing_line(N):
    """The stored blocks' bound, and the no-allocation variant's bits."""
    test_stored_block_gemm_edges(10, 130, 768, N)
    M, K = 130, 768
    t = synth.tensor(10, 72, "q2line", M, K)
    x = synth.normal(73, "q2linex", N * K, 1.0).reshape(N, K)
    ref = gpu_matmul(10, t.data, x, M, K)
    w_d, x_d = hiprt.DeviceBuffer.from_numpy(t.data, pad=256), hiprt.DeviceBuffer.from_numpy(x)
    y_d = hiprt.DeviceBuffer(4 * N * M)
    _native.check(_native.hip_lib().chatnet_matmul_noalloc(10, w_d.ptr, x_d.ptr, y_d.ptr, M, K, N, None))
    hiprt.synchronize()
    assert np.array_equal(y_d.to_numpy(np.float32, N * M).reshape(N, M), ref)
