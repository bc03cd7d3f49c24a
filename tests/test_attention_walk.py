"""The 16-bit attention forward at the edges of its pipelined walk: sequences that end anywhere in a step or a query
block, every number of multiplied columns, and rows whose maximum keeps growing along the walk (the
keys are walked from the last to the first), by little and by much.  Against float64 attention of the rounded
inputs; both kernels."""
import numpy as np
import pytest

from helpers import normal

pytestmark = pytest.mark.gpu

from mograd_amd import BF16, F16, F32, AnyBuffer  # noqa: E402
from mograd_amd.runtime import round_to_dtype  # noqa: E402


def reference(q, k, v, scale, causal):
    s = np.einsum("bmhd,bnhd->bhmn", q, k) * scale
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    top = s.max(-1, keepdims=True)
    p = np.exp(s - top)
    l = p.sum(-1, keepdims=True)
    return np.einsum("bhmn,bnhd->bhmd", p / l, v), (top + np.log(l))[..., 0], np.einsum("bhmn,bnhd->bhmd", p / l, np.abs(v))


@pytest.mark.parametrize("pipe", ["0", "1"])
@pytest.mark.parametrize("dtype,half_ulp", [(BF16, 2.0 ** -8), (F16, 2.0 ** -11)])
@pytest.mark.parametrize("S,D", [(1, 64), (31, 32), (65, 64), (129, 64), (160, 8), (191, 72), (193, 64), (255, 96), (256, 128),
                                 (257, 104), (383, 40), (449, 128), (640, 64)])
def test_forward_walk(device, monkeypatch, pipe, dtype, half_ulp, S, D):
    monkeypatch.setenv("MOGRAD_HIP_ATTN_FWD_PIPE", pipe)
    B, H, scale = 2, 3, D ** -0.5
    grow = np.linspace(6.0, 0.0, S, dtype=np.float32)[None, :, None, None]
    for causal in (0, 1):
        for steep in (0.0, 0.3, 6.0):
            q, k, v = (round_to_dtype(normal(97, i, (B, S, H, D)), dtype) for i in range(3))
            # a component that every query shares and every key has the more of, the earlier it comes
            q = round_to_dtype(q + 1.0, dtype) if steep else q
            k = round_to_dtype(k + steep * grow / D ** 0.5, dtype) if steep else k
            bq, bk, bv = (AnyBuffer.from_numpy(device, t, dtype) for t in (q, k, v))
            o, lse = AnyBuffer.create(dtype, device, B * H * S * D), AnyBuffer.create(F32, device, B * H * S)
            device.lib.mg_flash_attn_fwd(bq.data_ptr(), bk.data_ptr(), bv.data_ptr(), None, o.data_ptr(), lse.data_ptr(),
                                         B, S, H, D, scale, causal, 0, dtype, device.stream)
            want_o, want_lse, mass = reference(*(t.astype(np.float64) for t in (q, k, v)), scale, causal)
            # a probability and the result are each rounded once: half a unit of the sum's mass and of the result; what
            # is computed in fp32 (scores of up to ~100, their exponentials, the sums) adds far less: 1e-4
            err = np.abs(o.to_numpy((B, H, S, D)) - want_o)
            bound = (1.05 * half_ulp + 1e-4) * (mass + np.abs(want_o)) + (2.0 ** -24 if dtype == F16 else 0.0)
            assert (err <= bound).all(), (causal, steep, float((err / bound).max()))
            assert np.abs(lse.to_numpy((B, H, S)) - want_lse).max() <= 1e-4, (causal, steep)


# 256 and 257 tokens: narrow causal heads take either kernel there.
@pytest.mark.parametrize("pipe", ["default", "1"])
@pytest.mark.parametrize("dtype,half_ulp,later", [(BF16, 2.0 ** -8, "inf"), (BF16, 2.0 ** -8, "nan"), (BF16, 2.0 ** -8, "overflow"),
                                                  (F16, 2.0 ** -11, "inf"), (F16, 2.0 ** -11, "nan")])
@pytest.mark.parametrize("S,D", [(256, 64), (257, 64), (300, 96)])
def test_a_later_key_that_is_not_finite_does_not_reach_earlier_rows(device, monkeypatch, pipe, dtype, half_ulp, later, S, D):
    # Every row before key `at` sees finite scores only; its neighbours in a tile of 32 keys are among these rows.
    if pipe != "default":
        monkeypatch.setenv("MOGRAD_HIP_ATTN_FWD_PIPE", pipe)
    B, H, scale, at = 1, 2, D ** -0.5, S - 30
    q, k, v = (round_to_dtype(normal(98, i, (B, S, H, D)), dtype) for i in range(3))
    if later == "overflow":  # finite numbers whose product is not: 2^100 against 2^100 there, against 0 elsewhere
        q[..., 0], k[..., 0] = 2.0 ** 100, 0.0
    k_bad = k.copy()
    k_bad[:, at, :, 0] = {"inf": np.inf, "nan": np.nan, "overflow": 2.0 ** 100}[later]
    bq, bk, bv = (AnyBuffer.from_numpy(device, t, dtype) for t in (q, k_bad, v))
    o, lse = AnyBuffer.create(dtype, device, B * H * S * D), AnyBuffer.create(F32, device, B * H * S)
    device.lib.mg_flash_attn_fwd(bq.data_ptr(), bk.data_ptr(), bv.data_ptr(), None, o.data_ptr(), lse.data_ptr(), B, S, H, D,
                                 scale, 1, 0, dtype, device.stream)
    want_o, want_lse, mass = reference(*(t[:, :at].astype(np.float64) for t in (q, k, v)), scale, True)
    got = o.to_numpy((B, H, S, D))[:, :, :at]
    bound = (1.05 * half_ulp + 1e-4) * (mass + np.abs(want_o)) + (2.0 ** -24 if dtype == F16 else 0.0)
    assert (np.abs(got - want_o) <= bound).all()
    assert np.abs(lse.to_numpy((B, H, S))[:, :, :at] - want_lse).max() <= 1e-4


@pytest.mark.parametrize("S,D", [(257, 64), (300, 96)])
def test_a_row_whose_last_step_has_no_finite_score(device, S, D):
    # Row 64 of a causal problem sees one key of the step that its walk begins with, and its score is -inf: the rest of the
    # row is as without that key.
    B, H, scale = 1, 2, D ** -0.5
    q, k, v = (round_to_dtype(normal(99, i, (B, S, H, D)), BF16) for i in range(3))
    q[:, :, :, 0] = 1.0
    k_bad = k.copy()
    k_bad[:, 64, :, 0] = -np.inf
    bq, bk, bv = (AnyBuffer.from_numpy(device, t, BF16) for t in (q, k_bad, v))
    o, lse = AnyBuffer.create(BF16, device, B * H * S * D), AnyBuffer.create(F32, device, B * H * S)
    device.lib.mg_flash_attn_fwd(bq.data_ptr(), bk.data_ptr(), bv.data_ptr(), None, o.data_ptr(), lse.data_ptr(), B, S, H, D,
                                 scale, 1, 0, BF16, device.stream)
    q64, k64, v64 = (t.astype(np.float64) for t in (q, k, v))
    s = np.einsum("bhd,bnhd->bhn", q64[:, 64], k64[:, :64]) * scale
    p = np.exp(s - s.max(-1, keepdims=True))
    want = np.einsum("bhn,bnhd->bhd", p / p.sum(-1, keepdims=True), v64[:, :64])
    mass = np.einsum("bhn,bnhd->bhd", p / p.sum(-1, keepdims=True), np.abs(v64[:, :64]))
    assert (np.abs(o.to_numpy((B, H, S, D))[:, :, 64] - want) <= (1.05 * 2.0 ** -8 + 1e-4) * (mass + np.abs(want))).all()
    want_lse = s.max(-1) + np.log(p.sum(-1))
    assert np.abs(lse.to_numpy((B, H, S))[:, :, 64] - want_lse).max() <= 1e-4


def test_rows_too_long_for_32bit_offsets(device):
    # Packed Q, K, V with 180000 heads: 69 MB from a token to the next, so that the last rows of a step of 64 lie more than
    # 4 GiB behind its first.  Three heads hold numbers and are compared with the same heads on their own; 24 GB in all.
    lib, st, S, H, D, dtype = device.lib, device.stream, 130, 180000, 64, BF16
    heads, row = (0, H // 2 + 1, H - 1), D * 2
    big = lambda n: AnyBuffer.create(dtype, device, n, fill=0.125)
    place = lambda buf, token, h, n: buf.data_ptr().value + ((token * n) * H + h) * row  # (n: 3 for packed, 1 for O)
    small_in = [AnyBuffer.from_numpy(device, normal(100, h, (S, 4, D)), dtype) for h in range(3)]  # Q, K, V and dO of a head
    qkv, d_qkv, o, d_o = big(S * 3 * H * D), big(S * 3 * H * D), big(S * H * D), big(S * H * D)
    lse = AnyBuffer.create(F32, device, H * S)
    for h, t in zip(heads, small_in):
        for s in range(S):
            src = t.data_ptr().value + s * 4 * row
            for j in range(3):
                lib.mg_copy_device(place(qkv, s, 0, 3) + (j * H + h) * row, src + j * row, row, st)
            lib.mg_copy_device(place(d_o, s, h, 1), src + 3 * row, row, st)
    p = lambda b: b.data_ptr()
    for causal in (0, 1):
        lib.mg_flash_attn_fwd_packed(p(qkv), None, p(o), p(lse), 1, S, H, D, D ** -0.5, causal, 0, dtype, st)
        lib.mg_flash_attn_bwd_packed(p(d_o), p(o), p(qkv), None, p(lse), p(d_qkv), 1, S, H, D, D ** -0.5, causal, 0, dtype, st)
        for h, t in zip(heads, small_in):
            t = t.to_numpy((S, 4, D))
            one = [AnyBuffer.from_numpy(device, np.ascontiguousarray(a), dtype) for a in (t[:, :3], t[:, 3])]
            o1, l1, g1 = (AnyBuffer.create(d, device, n) for d, n in ((dtype, S * D), (F32, S), (dtype, S * 3 * D)))
            lib.mg_flash_attn_fwd_packed(p(one[0]), None, p(o1), p(l1), 1, S, 1, D, D ** -0.5, causal, 0, dtype, st)
            lib.mg_flash_attn_bwd_packed(p(one[1]), p(o1), p(one[0]), None, p(l1), p(g1), 1, S, 1, D, D ** -0.5, causal, 0, dtype, st)
            got_o, got_g = AnyBuffer.create(dtype, device, S * D), AnyBuffer.create(dtype, device, S * 3 * D)
            for s in range(S):
                lib.mg_copy_device(got_o.data_ptr().value + s * row, place(o, s, h, 1), row, st)
                for j in range(3):
                    lib.mg_copy_device(got_g.data_ptr().value + (s * 3 + j) * row, place(d_qkv, s, 0, 3) + (j * H + h) * row, row, st)
            for name, got, want in (("o", got_o, o1), ("gradients", got_g, g1)):
                a, b = got.to_numpy().astype(np.float64), want.to_numpy().astype(np.float64)
                # two kernels that round a probability and a result each: 2^-8 of the largest numbers, over the norm
                assert np.linalg.norm(a - b) <= 2.0 ** -7 * np.linalg.norm(b), (causal, h, name)
    del qkv, d_qkv, o, d_o, lse
    lib.mg_pool_empty_cache()
