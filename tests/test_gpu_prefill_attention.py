"""The prompt attention kernel at the edges of its tiles (32 queries per wave,
64 keys per tile, 4- and 8-wave workgroups), against float64 softmax
attention."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _prompt(tokens, kv_heads, scale, device):
    """Dense q and k and the v slice of a fused projection, as prefill has them."""
    gen = torch.Generator(device=device).manual_seed(20261204 + tokens)
    fused = (torch.randn(tokens, kv_heads * 6 * 128, device=device, generator=gen) * scale).half()
    q = fused[:, :kv_heads * 512].reshape(tokens, kv_heads * 4, 128).contiguous()
    k = fused[:, kv_heads * 512:kv_heads * 640].reshape(tokens, kv_heads, 128).contiguous()
    return q, k, fused[:, kv_heads * 640:].view(tokens, kv_heads, 128)


# 4099 tokens x 8 heads (65 x 8 workgroups of 64 queries) and 2111 x 16 take the
# 8-wave kernel
@pytest.mark.parametrize("tokens,kv_heads,scale", [
    (1, 8, 1.0), (31, 1, 1.0), (32, 8, 1.0), (33, 3, 1.0), (63, 8, 1.0), (64, 2, 1.0),
    (65, 8, 1.0), (129, 8, 4.0), (1000, 8, 1.0), (4099, 8, 1.0), (2111, 16, 4.0)])
def test_causal_attention_matches_float64(cuda, tokens, kv_heads, scale):
    from pagegauge_amd import decoder as dec

    print(f"causal attention tokens={tokens} kv_heads={kv_heads} scale={scale}", flush=True)
    q, k, v = _prompt(tokens, kv_heads, scale, cuda)
    assert dec._attention_kernel_takes(q, k, v)
    got = dec._causal_attention(q, k, v).double()
    rows = torch.arange(tokens, device=cuda)
    hidden = rows[None, :] > rows[:, None]
    for h in range(0, q.shape[1], 1 if tokens < 1000 else 5):
        scores = (q[:, h].double() @ k[:, h // 4].double().t()) * 128 ** -0.5
        p = torch.softmax(scores.masked_fill(hidden, float("-inf")), dim=-1)
        vh = v[:, h // 4].double()
        want = p @ vh
        # probabilities (relative to a running maximum, so the largest is at
        # least 1) and the output round to FP16: 2^-11 of the sum of |p v| and
        # of the output; below 2^-14 a probability is off by up to 2^-25
        # instead, per key; scores of 128 float32 products are off by up to
        # 128 * 2^-24 * |q| |k| / sqrt(128) <= 128 * 2^-24 * 2^2 * scale^2 * 4
        score_error = 2.0 ** -13 * scale * scale
        bound = ((2.0 ** -11 + score_error) * (p @ vh.abs() + want.abs())
                 + tokens * 2.0 ** -25 * vh.abs().max())
        assert ((got[:, h] - want).abs() <= bound).all(), (h, ((got[:, h] - want).abs() / bound).max())


@pytest.mark.parametrize("tokens,kv_heads", [(200, 2), (4099, 8)])        # 4 and 8 waves
def test_causal_attention_of_infinite_scores(cuda, tokens, kv_heads):
    """Keys of -inf scores weigh nothing, whole tiles of them from the first
    key on included; a row of nothing else, an infinite maximum and a NaN give
    NaN rows, and every other row stays finite."""
    from pagegauge_amd import decoder as dec

    print(f"causal attention, infinite scores, tokens={tokens} kv_heads={kv_heads}", flush=True)
    q, k, v = _prompt(tokens, kv_heads, 1.0, cuda)
    q[..., 0] = q[..., 0].abs() + 0.5
    k[..., 0] = 0.0
    dead = list(range(0, 70)) + [100, 131]                  # past the first tile of 64
    k[dead, :, 0] = float("-inf")
    q[150], k[170, :, 0], q[:, 3, 0] = float("nan"), float("inf"), 0.25
    got = dec._causal_attention(q, k, v)
    rows = torch.arange(tokens, device=cuda)
    hidden = rows[None, :] > rows[:, None]
    nan = (rows < 70) | (rows == 150) | (rows >= 170)
    for h in range(0, q.shape[1], 3):
        scores = (q[:, h].double() @ k[:, h // 4].double().t()) * 128 ** -0.5
        p = torch.softmax(scores.masked_fill(hidden, float("-inf")), dim=-1)
        want = p @ v[:, h // 4].double()
        assert torch.equal(want.isnan().any(-1), nan) and torch.equal(got[:, h].isnan().all(-1), nan)
        # FP16 probabilities and output, as in the test above (scale 1)
        bound = ((2.0 ** -11 + 2.0 ** -13) * (p @ v[:, h // 4].double().abs() + want.abs())
                 + tokens * 2.0 ** -25 * v.double().abs().max())
        assert ((got[:, h].double() - want).abs() <= bound)[~nan].all(), h


def test_causal_attention_takes_other_layouts_through_torch(cuda):
    from pagegauge_amd import decoder as dec

    q, k, v = _prompt(80, 2, 1.0, cuda)
    want = dec._causal_attention(q, k, v)
    shifted = torch.empty(80 * 256 + 1, device=cuda, dtype=torch.float16)[1:].view(80, 2, 128)
    shifted.copy_(v)                                   # 2-byte aligned rows
    for other in ((q.float(), k.float(), v.float()), (q, k, shifted)):
        assert not dec._attention_kernel_takes(*other)
        got = dec._causal_attention(*other)
        assert (got.float() - want.float()).abs().max() < 1e-2


def test_causal_attention_rejects_bad_arguments(cuda):
    from pagegauge_amd import _capi

    q, k, v = _prompt(16, 2, 1.0, cuda)
    out = torch.empty_like(q)
    stream = torch.cuda.current_stream().cuda_stream

    def call(tokens=16, heads=8, kv_heads=2, k_stride=256, k_at=0, scale=0.1):
        _capi.call("pg_causal_attention", q.data_ptr(), q.stride(0), k.data_ptr() + k_at, k_stride,
                   v.data_ptr(), v.stride(0), out.data_ptr(), out.stride(0), tokens, heads,
                   kv_heads, scale, stream)

    for kwargs, message in (({"tokens": 0}, "at least one token"), ({"heads": 4}, "GQA group"),
                            ({"k_stride": 128}, "strides"), ({"k_stride": 260}, "strides"),
                            ({"k_at": 2}, "aligned"), ({"scale": 0.0}, "sm_scale")):
        with pytest.raises(RuntimeError, match=message):
            call(**kwargs)
