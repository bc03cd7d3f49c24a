"""Products and Linear backwards whose sizes sit at the edges of the kernels' ranges: reductions
that end on a short step, widths that are no multiple of a 16-byte chunk, outputs of a few tiles
(fp32 straight from memory, 16 x 16 and 32 x 32), of 64 x 64 and of 128 x 128 tiles, and rows few enough
that nothing is split.  All against float64 products of the rounded inputs."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_close, normal

pytestmark = pytest.mark.gpu

from mograd_amd import BF16, F16, F32, AnyBuffer  # noqa: E402
from mograd_amd.runtime import round_to_dtype  # noqa: E402

RT = {F32: 1e-5, F16: 2e-3, BF16: 1.6e-2}
SHAPES = [(1, 1, 1), (5, 3, 4), (64, 10, 256), (33, 17, 65), (130, 65, 100), (64, 256, 784), (333, 257, 129), (200, 136, 264),
          (1000, 72, 88), (1023, 264, 8), (1025, 96, 384), (1999, 1001, 767), (2587, 256, 256), (1056, 1152, 384)]


def check_linear(device, dtype, M, N, K):
    """Forward (bias, ReLU) and the three gradients (ReLU mask, accumulating dX) of one layer."""
    lib, st, rt = device.lib, device.stream, RT[dtype]
    x = np.maximum(round_to_dtype(normal(60, 0, (M, K)), dtype), 0)
    w = round_to_dtype(normal(60, 1, (N, K), std=0.1), dtype)
    b = round_to_dtype(normal(60, 2, (N,), std=0.1), dtype)
    dy = round_to_dtype(normal(60, 3, (M, N), std=0.5), dtype)
    prior = round_to_dtype(normal(60, 4, (M, K)), dtype)
    bx, bw, bb, bdy = (AnyBuffer.from_numpy(device, a, dtype) for a in (x, w, b, dy))
    dx = AnyBuffer.from_numpy(device, prior, dtype)
    y, dw, db = (AnyBuffer.create(dtype, device, n) for n in (M * N, N * K, N))
    P = lambda t: t.data_ptr()  # noqa: E731
    lib.mg_matmul_bias_relu_bt(P(bx), P(bw), P(bb), P(y), 1, M, N, K, K, 1, K, 1, M * K, N * K, dtype, st)
    lib.mg_linear_bwd_fused(P(bdy), P(bx), P(bw), P(dx), P(dw), P(db), M, N, K, 1, 1, dtype, st)
    x, w, b, dy, prior = (a.astype(np.float64) for a in (x, w, b, dy, prior))
    want = np.maximum(x @ w.T + b, 0)
    assert_close(y.to_numpy((M, N)), want, rt, rt * max(np.abs(want).max(), 1e-3), "y")
    want = dy @ w * (x > 0)
    assert_close(dx.to_numpy((M, K)), prior + want, 2 * rt, 2 * rt * max(np.abs(want).max(), 1e-3), "dx")
    want = dy.T @ x
    assert_close(dw.to_numpy((N, K)), want, rt, rt * max(np.abs(want).max(), 1e-3), "dw")
    want = dy.sum(axis=0)
    assert_close(db.to_numpy(), want, rt, rt * max(np.abs(want).max(), 1e-3), "db")


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_forward_and_backward(device, dtype, M, N, K):
    check_linear(device, dtype, M, N, K)


# Both sides of each choice that the dispatch makes by size, at sizes where it could go either way
@pytest.mark.parametrize("dtype,knob,values,shapes", [
    # fp32: tiles straight from memory, of 64 x 64, of 128 x 128, aligned and copied operands
    (F32, "GEMM_F32_TILE", (32, 64, 128), [(300, 264, 200), (257, 129, 333), (70, 33, 1030)]),
    # fp32 backward: one launch from memory (up to so many MFLOP), or a launch for each product
    (F32, "LINEAR_BWD_F32_MFLOP", (0, 100000), [(300, 264, 200), (257, 129, 333), (1500, 10, 260)]),
    # 16-bit operands off the 16-byte chunks: staged as they are, or copied first
    (BF16, "GEMM16_PAD", (0, 1), [(300, 265, 200), (257, 129, 333), (1030, 130, 67)]),
    (F16, "GEMM16_PAD", (0, 1), [(257, 129, 333)]),
    # 16-bit forward on 64 x 64 and on 128 x 128 tiles
    (BF16, "GEMM16_PIPE", (64, 128), [(300, 264, 200), (129, 72, 1024)]),
    # 16-bit backward on 128-row tiles or 64 x 64 ones, and those with dW's rows in 1, 3 or 7 ranges
    (BF16, "LINEAR_BWD_SMALL", (0, 1), [(2048, 264, 200), (1999, 129, 333), (2600, 776, 384)]),
    (BF16, "LINEAR_BWD_SPLITS", (1, 3, 7), [(1030, 264, 200), (999, 129, 65)]),
    (F16, "LINEAR_BWD_SPLITS", (1, 3), [(999, 129, 65)]),
    # 16-bit backward of layers off the 16-byte chunks on 64 x 64 tiles: from copies or from where the arrays are
    (BF16, "LINEAR_BWD_ANY", (0, 1), [(497, 45, 27), (1344, 77, 264), (1481, 299, 1088)]),
    (F16, "LINEAR_BWD_ANY", (0, 1), [(1103, 152, 93)]),
])
def test_both_sides_of_a_choice(device, monkeypatch, dtype, knob, values, shapes):
    for value in values:
        monkeypatch.setenv("MOGRAD_HIP_" + knob, str(value))
        for M, N, K in shapes:
            check_linear(device, dtype, M, N, K)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("offset", [0, 1])  # elements that the operands start off a 16-byte boundary
@pytest.mark.parametrize("M,N,K", [(96, 160, 133), (520, 390, 1026), (1500, 1300, 130)])
def test_every_layout_batched(device, dtype, offset, M, N, K):
    lib, st, rt, B = device.lib, device.stream, RT[dtype], 2
    a = round_to_dtype(normal(61, 0, (B, M, K)), dtype)
    b = round_to_dtype(normal(61, 1, (B, N, K), std=0.1), dtype)
    want = a.astype(np.float64) @ b.astype(np.float64).transpose(0, 2, 1)

    def up(t):
        flat = AnyBuffer.from_numpy(device, np.concatenate([np.zeros(offset, np.float32), t.reshape(-1)]), dtype)
        return AnyBuffer(flat.storage, dtype, t.size, offset)

    for la in "km":
        for lb in "kn":
            ba = up(a if la == "k" else a.transpose(0, 2, 1))
            bb = up(b if lb == "k" else b.transpose(0, 2, 1))
            c = AnyBuffer.create(dtype, device, B * M * N)
            lib.mg_matmul(ba.data_ptr(), bb.data_ptr(), c.data_ptr(), B, M, N, K, *((K, 1) if la == "k" else (1, M)),
                          *((1, K) if lb == "k" else (N, 1)), M * K, N * K, dtype, st)
            assert_close(c.to_numpy((B, M, N)), want, rt, rt * np.abs(want).max(), la + lb)


# 16-bit 64 x 64 tiles of operands off the 16-byte chunks: a reduction and edges that end anywhere in a chunk, every number of
# steps under way, rows from any element on, K ranges
@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("offset", [0, 1, 6])
@pytest.mark.parametrize("M,N,K", [(8, 9, 8), (9, 64, 63), (65, 10, 65), (64, 71, 129), (70, 66, 193), (67, 130, 257), (33, 129, 321),
                                   (129, 15, 391), (77, 65, 1681)])
def test_tiles_of_64_off_the_chunks(device, monkeypatch, dtype, offset, M, N, K):
    monkeypatch.setenv("MOGRAD_HIP_GEMM16_PIPE", "64")
    lib, st, rt, B = device.lib, device.stream, RT[dtype], 2
    a = round_to_dtype(normal(64, 0, (B, M, K)), dtype)
    b = round_to_dtype(normal(64, 1, (B, N, K), std=0.1), dtype)
    bias = round_to_dtype(normal(64, 2, (N,)), dtype)
    want = a.astype(np.float64) @ b.astype(np.float64).transpose(0, 2, 1)

    def up(t):  # (what lies around the operand is no number)
        flat = np.full(t.size + offset + 16, np.nan, np.float32)
        flat[offset:offset + t.size] = t.reshape(-1)
        whole = AnyBuffer.from_numpy(device, flat, dtype)
        return AnyBuffer(whole.storage, dtype, t.size, offset), whole

    for la in "km":
        for lb in "kn":
            (ba, _a), (bb, _b) = up(a if la == "k" else a.transpose(0, 2, 1)), up(b if lb == "k" else b.transpose(0, 2, 1))
            c = AnyBuffer.create(dtype, device, B * M * N)
            lib.mg_matmul(ba.data_ptr(), bb.data_ptr(), c.data_ptr(), B, M, N, K, *((K, 1) if la == "k" else (1, M)),
                          *((1, K) if lb == "k" else (N, 1)), M * K, N * K, dtype, st)
            assert_close(c.to_numpy((B, M, N)), want, rt, rt * np.abs(want).max(), la + lb)
    (ba, _a), (bb, _b), (bbias, _c) = up(a), up(b), up(bias)
    c = AnyBuffer.create(dtype, device, B * M * N)
    lib.mg_matmul_bias_bt(ba.data_ptr(), bb.data_ptr(), bbias.data_ptr(), c.data_ptr(), B, M, N, K, K, 1, K, 1, M * K, N * K,
                          dtype, st)
    assert_close(c.to_numpy((B, M, N)), want + bias, rt, rt * np.abs(want).max(), "bias")
    # and one launch for a layer's three gradients
    monkeypatch.delenv("MOGRAD_HIP_GEMM16_PIPE")
    monkeypatch.setenv("MOGRAD_HIP_LINEAR_BWD_SMALL", "1")
    dy = round_to_dtype(normal(64, 3, (M, N), std=0.5), dtype)
    (bdy, _d), (bx, _x), (bw, _w) = up(dy), up(a[0]), up(b[0])
    for splits in ("1", "2"):
        monkeypatch.setenv("MOGRAD_HIP_LINEAR_BWD_SPLITS", splits)
        dx, dw, db = (AnyBuffer.create(dtype, device, n) for n in (M * K, N * K, N))
        lib.mg_linear_bwd_fused(bdy.data_ptr(), bx.data_ptr(), bw.data_ptr(), dx.data_ptr(), dw.data_ptr(), db.data_ptr(), M, N, K,
                                0, 0, dtype, st)
        x64, w64, dy64 = (t.astype(np.float64) for t in (a[0], b[0], dy))
        for got, ref, what in ((dx.to_numpy((M, K)), dy64 @ w64, "dx"), (dw.to_numpy((N, K)), dy64.T @ x64, "dw"),
                               (db.to_numpy(), dy64.sum(0), "db")):
            assert_close(got, ref, rt, rt * max(np.abs(ref).max(), 1e-3), f"{what}, {splits}")


# 16-bit 64 x 64 tiles: k steps of 64 around the four copies, one tile and many, K ranges, both gradient types
@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 192), (65, 72, 256), (262, 768, 768), (330, 64, 320), (72, 1032, 64),
                                   (2000, 64, 128), (262, 768, 3072)])
def test_tiles_of_64(device, dtype, M, N, K):
    lib, st, rt = device.lib, device.stream, RT[dtype]
    x = round_to_dtype(normal(62, 0, (M, K)), dtype)
    w = round_to_dtype(normal(62, 1, (N, K), std=0.1), dtype)
    dy = round_to_dtype(normal(62, 2, (M, N), std=0.5), dtype)
    r = round_to_dtype(normal(62, 3, (M, N)), dtype)
    bx, bw, bdy, br = (AnyBuffer.from_numpy(device, a, dtype) for a in (x, w, dy, r))
    P = lambda t: t.data_ptr()  # noqa: E731
    y = AnyBuffer.create(dtype, device, M * N)
    lib.mg_matmul_bt_add(P(bx), P(bw), P(br), P(y), 1, M, N, K, K, 1, K, 1, M * K, N * K, dtype, st)
    x, w, dy, r = (a.astype(np.float64) for a in (x, w, dy, r))
    assert_close(y.to_numpy((M, N)), x @ w.T + r, rt, 2 * rt * np.abs(x @ w.T).max(), "y")
    pending = C.c_void_p()
    lib.mg_deferred_create(C.byref(pending))
    for grad in (dtype, F32):
        dx = AnyBuffer.create(dtype, device, M * K)
        dw, db = AnyBuffer.create(grad, device, N * K, fill=3.0), AnyBuffer.create(grad, device, N, fill=3.0)
        lib.mg_linear_bwd_deferred(P(bdy), P(bx), P(bw), P(dx), P(dw), P(db), M, N, K, 0, 0, dtype, grad, pending, st)
        lib.mg_finish_deferred(pending, st)
        g = rt if grad == dtype else 1e-5
        for got, want, tol, name in ((dx.to_numpy((M, K)), dy @ w, rt, "dx"), (dw.to_numpy((N, K)), dy.T @ x, g, "dw"),
                                     (db.to_numpy(), dy.sum(axis=0), g, "db")):
            assert_close(got, want, tol, tol * np.abs(want).max(), f"{name} {grad}")
    lib.mg_deferred_destroy(pending)


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("M,N,K", [(3, 5, 7), (64, 256, 784), (700, 33, 40), (1040, 72, 200)])
def test_weight_gradients_alone(device, dtype, M, N, K):
    lib, st, rt = device.lib, device.stream, RT[dtype]
    x = round_to_dtype(normal(63, 0, (M, K)), dtype)
    dy = round_to_dtype(normal(63, 1, (M, N), std=0.5), dtype)
    bx, bdy = AnyBuffer.from_numpy(device, x, dtype), AnyBuffer.from_numpy(device, dy, dtype)
    dw, db = AnyBuffer.create(dtype, device, N * K), AnyBuffer.create(dtype, device, N)
    lib.mg_linear_bwd_fused(bdy.data_ptr(), bx.data_ptr(), None, None, dw.data_ptr(), db.data_ptr(), M, N, K, 0, 0, dtype, st)
    x, dy = x.astype(np.float64), dy.astype(np.float64)
    assert_close(dw.to_numpy((N, K)), dy.T @ x, rt, rt * np.abs(dy.T @ x).max(), "dw")
    assert_close(db.to_numpy(), dy.sum(axis=0), rt, rt * np.abs(dy.sum(axis=0)).max(), "db")


# fp32, a short reduction into a large output: the plain kernel up to its k-step of 16 and, for operands that
# do not lie on 16-byte chunks, below 32; tiles elsewhere, and wherever the plain kernel's grid ends
@pytest.mark.parametrize("B,M,N,K", [(1, 1024, 1024, 4), (1, 1024, 1028, 16), (1, 1028, 1024, 20), (1, 1024, 1024, 28),
                                     (1, 1024, 1024, 17), (1, 1030, 1021, 31), (1, 4096, 4096, 24), (300, 64, 60, 20),
                                     (65537, 8, 8, 16), (65537, 8, 8, 10), (65537, 8, 7, 20), (1, 4194305, 4, 16)])
def test_short_reductions_into_large_outputs(device, B, M, N, K):
    lib, st = device.lib, device.stream
    a, b = normal(64, 0, (B, M, K)), normal(64, 1, (B, N, K))
    want = np.matmul(a.astype(np.float64), b.astype(np.float64).transpose(0, 2, 1))
    for lb in "kn":
        ba = AnyBuffer.from_numpy(device, a)
        bb = AnyBuffer.from_numpy(device, b if lb == "k" else b.transpose(0, 2, 1))
        c = AnyBuffer.create(F32, device, B * M * N)
        lib.mg_matmul(ba.data_ptr(), bb.data_ptr(), c.data_ptr(), B, M, N, K, K, 1, *((1, K) if lb == "k" else (N, 1)),
                      M * K, N * K, F32, st)
        # K products and K - 1 sums, each rounded once: K 2^-24 of sum |a b| at most
        bound = K * 2.0**-24 * np.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64).transpose(0, 2, 1))
        assert np.all(np.abs(c.to_numpy((B, M, N)) - want) <= bound), lb


# fp32 operands of at most 128 rows that are contiguous along neither axis, with a long K: copied to
# k-contiguous rows, so that the product is bit for bit that of the copy
@pytest.mark.parametrize("B,M,N,K,which", [(1, 10, 4096, 2048, "a"), (1, 1, 300, 512, "a"), (1, 256, 128, 1001, "b"),
                                           (1, 96, 100, 1024, "ab"), (3, 128, 260, 520, "a"), (3, 200, 7, 640, "b"),
                                           (1, 129, 64, 512, "a"), (1, 64, 300, 511, "a")])
def test_thin_operands_without_a_unit_stride(device, B, M, N, K, which):
    lib, st = device.lib, device.stream
    a, b = normal(65, 0, (B, M, 2 * K)), normal(65, 1, (B, N, 2 * K))
    ops = {"a": a, "b": b}
    flat = {k: np.ascontiguousarray(t[..., ::2]) for k, t in ops.items()}

    def product(strided):
        buf = {k: AnyBuffer.from_numpy(device, ops[k] if k in strided else flat[k]) for k in "ab"}
        ld = {k: (2 * K, 2, ops[k].shape[1] * 2 * K) if k in strided else (K, 1, ops[k].shape[1] * K) for k in "ab"}
        c = AnyBuffer.create(F32, device, B * M * N)
        lib.mg_matmul_bt(buf["a"].data_ptr(), buf["b"].data_ptr(), c.data_ptr(), B, M, N, K, *ld["a"][:2], *ld["b"][:2],
                         ld["a"][2], ld["b"][2], F32, st)
        return c.to_numpy((B, M, N))

    got, x, y = product(which), flat["a"].astype(np.float64), flat["b"].astype(np.float64).transpose(0, 2, 1)
    # K products and K - 1 sums, each rounded once: K 2^-24 of sum |a b| at most
    assert np.all(np.abs(got - x @ y) <= K * 2.0**-24 * (np.abs(x) @ np.abs(y)))
    if K >= 512 and all(ops[k].shape[1] <= 128 for k in which):
        np.testing.assert_array_equal(got, product(""))
