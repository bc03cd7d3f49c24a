"""The copied-tile kernels of 16-bit products (output tiles of 128 x 128, 128 x 192 and 256 x 256) at the edges of
their pipeline: reductions shorter than the copies they keep, of one and two steps, ending on a short step; tiles
cut off on either side.  Every tile adds each output element's products over k in the same order on
the same MFMA as the register-staged kernel, so all must agree bit for bit; that kernel is held to
float64 products of the rounded inputs."""
import numpy as np
import pytest

from helpers import assert_close, normal

pytestmark = pytest.mark.gpu

from mograd_amd import BF16, F16, AnyBuffer  # noqa: E402
from mograd_amd.runtime import round_to_dtype  # noqa: E402

RT = {F16: 2e-3, BF16: 1.6e-2}


def tiles_agree(device, monkeypatch, dtype, layout, batch, M, N, K):
    lib, st = device.lib, device.stream
    a = round_to_dtype(normal(91, 0, (batch, M, K)), dtype)
    b = round_to_dtype(normal(91, 1, (batch, N, K), std=0.1), dtype)
    bias = round_to_dtype(normal(91, 2, (N,), std=0.5), dtype)
    res = round_to_dtype(normal(91, 3, (batch, M, N)), dtype)
    ba = AnyBuffer.from_numpy(device, a if layout[0] == "k" else np.ascontiguousarray(a.swapaxes(1, 2)), dtype)
    bb = AnyBuffer.from_numpy(device, b if layout[1] == "k" else np.ascontiguousarray(b.swapaxes(1, 2)), dtype)
    bbias, bres = AnyBuffer.from_numpy(device, bias, dtype), AnyBuffer.from_numpy(device, res, dtype)
    sa = (K, 1) if layout[0] == "k" else (1, M)
    sb = (K, 1) if layout[1] == "k" else (1, N)  # strides of element (n, k)
    args = (batch, M, N, K, *sa, *sb, M * K, N * K, dtype, st)
    results, n = {}, batch * M * N
    for tile in ("0", "128", "2000", "4000"):
        monkeypatch.setenv("MOGRAD_HIP_GEMM16_PIPE", tile)
        # canaries behind the result
        y, z = (AnyBuffer.from_numpy(device, np.full(n + 64, 7.0, np.float32), dtype) for _ in range(2))
        lib.mg_matmul_bias_relu_bt(ba.data_ptr(), bb.data_ptr(), bbias.data_ptr(), y.data_ptr(), *args)
        lib.mg_matmul_bt_add(ba.data_ptr(), bb.data_ptr(), bres.data_ptr(), z.data_ptr(), *args)
        for t in (y, z):
            assert (t.to_numpy()[n:] == 7.0).all(), tile
        results[tile] = (y.to_numpy()[:n], z.to_numpy()[:n])
    for tile in ("128", "2000", "4000"):
        for got, want, name in zip(results[tile], results["0"], ("bias, relu", "residual")):
            np.testing.assert_array_equal(got, want, err_msg=f"{tile}: {name}")
    p = a.astype(np.float64) @ b.astype(np.float64).swapaxes(1, 2)
    rt = RT[dtype]
    for got, want in zip(results["0"], (np.maximum(p + bias, 0), p + res)):
        assert_close(got.reshape(batch, M, N), want, rt, rt * max(np.abs(want).max(), 1e-3))


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("layout", ["kk", "kn", "mk", "mn"])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (136, 200, 64), (264, 392, 72), (128, 192, 128), (256, 256, 136), (392, 328, 192),
                                   (64, 576, 200), (520, 72, 264), (264, 264, 448)])
def test_tiles_agree_at_every_length(device, monkeypatch, dtype, layout, M, N, K):
    # (neither operand contiguous along k: any length)
    tiles_agree(device, monkeypatch, dtype, layout, 1, M, N, K - 3 if layout == "mn" else K)


@pytest.mark.parametrize("layout", ["kk", "kn", "mk", "mn"])
@pytest.mark.parametrize("batch,M,N,K", [(1, 136, 129, 64), (3, 392, 5, 203), (2, 264, 333, 72), (2, 130, 201, 131), (2, 131, 195, 2051),
                                         (3, 256, 264, 192)])
def test_tiles_agree_at_odd_edges_and_in_batches(device, monkeypatch, layout, batch, M, N, K):
    # Rows of the result off the 16-byte chunks: those over the right edge go out element by element.  Operands off
    # them are copied first.  (2051: K in ranges, of which every tile has the same.)
    monkeypatch.setenv("MOGRAD_HIP_GEMM16_PAD", "1")
    tiles_agree(device, monkeypatch, BF16, layout, batch, M, N, K)


@pytest.mark.parametrize("tile", ["128", "192"])
@pytest.mark.parametrize("accumulate", [0, 1])
@pytest.mark.parametrize("M,N,K", [(512, 72, 200), (1000, 264, 192), (2587, 136, 104), (1999, 392, 328), (1000, 264, 193),
                                   (515, 129, 5)])
def test_linear_backward_tiles(device, monkeypatch, tile, accumulate, M, N, K):
    # dX, dW and db in one launch with either tile: odd numbers of rows (dW's last range ends on a short step), dX from
    # one to seven steps, its rows on 16-byte chunks and off them.
    lib, st, dtype = device.lib, device.stream, BF16
    monkeypatch.setenv("MOGRAD_HIP_LINEAR_BWD_SMALL", "0")
    monkeypatch.setenv("MOGRAD_HIP_LINEAR_BWD_TILE", tile)
    x = np.maximum(round_to_dtype(normal(92, 0, (M, K)), dtype), 0)
    w = round_to_dtype(normal(92, 1, (N, K), std=0.1), dtype)
    dy = round_to_dtype(normal(92, 2, (M, N), std=0.5), dtype)
    bx, bw, bdy = (AnyBuffer.from_numpy(device, t, dtype) for t in (x, w, dy))
    prior = round_to_dtype(normal(92, 3, (M, K)), dtype)
    dx, dw, db = AnyBuffer.from_numpy(device, prior, dtype), *(AnyBuffer.create(dtype, device, n) for n in (N * K, N))
    lib.mg_linear_bwd_fused(bdy.data_ptr(), bx.data_ptr(), bw.data_ptr(), dx.data_ptr(), dw.data_ptr(), db.data_ptr(), M, N, K,
                            accumulate, 1, dtype, st)
    x, w, dy = (t.astype(np.float64) for t in (x, w, dy))
    rt = RT[dtype]
    for got, want, name in ((dx.to_numpy((M, K)), dy @ w * (x > 0) + accumulate * prior, "dx"), (dw.to_numpy((N, K)), dy.T @ x, "dw"),
                            (db.to_numpy(), dy.sum(axis=0), "db")):
        assert_close(got, want, rt, rt * np.abs(want).max(), name)
