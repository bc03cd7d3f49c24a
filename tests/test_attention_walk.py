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
