"""The prefill's element-wise kernels against the torch operators they stand
for, at the edges of their rows: RoPE, SwiGLU and the residual add bit for bit,
the norm to one FP16 step (its float32 mean sums in another order)."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _rand(device, *shape, scale=1.0):
    gen = torch.Generator(device=device).manual_seed(sum(shape))
    return (torch.randn(*shape, device=device, generator=gen) * scale).half()


# 2, 4 and 8 vectors of 8 per thread of 256, rows that fill and that do not
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 96), (5, 4096), (2, 4104), (3, 8192),
                                        (2, 8200), (1, 16384)])
@pytest.mark.parametrize("with_delta", [False, True])
def test_norm_rows(cuda, rows, width, with_delta):
    from pagegauge_amd import decoder as dec

    print(f"norm rows={rows} width={width} delta={with_delta}", flush=True)
    x, weight = _rand(cuda, rows, width, scale=3.0), _rand(cuda, width)
    delta = _rand(cuda, rows + 1, width)[1:] if with_delta else None
    want_x = x + delta if with_delta else x.clone()
    got = dec._norm_rows(x, weight, 1e-5, delta)
    assert torch.equal(x, want_x)
    want = dec.rms_norm(want_x, weight, 1e-5)
    # fp16(x * inv) one step apart (2^-10 of it), times the weight, rounded
    # again: 2^-9 relative, and one subnormal step
    assert ((got.float() - want.float()).abs() <= want.float().abs() * 2.0 ** -9 + 2.0 ** -23).all()


@pytest.mark.parametrize("tokens,kv_heads", [(1, 8), (33, 1), (1000, 8)])
def test_rope_rows(cuda, tokens, kv_heads):
    from pagegauge_amd import decoder as dec

    cfg = dec.DecoderConfig(layers=1, hidden=kv_heads * 512, q_heads=4 * kv_heads,
                            kv_heads=kv_heads, intermediate=8, vocab=8)
    qkv = _rand(cuda, tokens, cfg.qkv_width)
    cos, sin = (t.to(cuda) for t in dec.rope_tables(tokens, cfg.rope_theta))
    q, k = dec._rope_rows(cfg, qkv, cos, sin)
    qw, kw = cfg.q_heads * 128, cfg.kv_heads * 128
    assert torch.equal(q, dec.rope(qkv[:, :qw].view(tokens, -1, 128), cos, sin))
    assert torch.equal(k, dec.rope(qkv[:, qw:qw + kw].view(tokens, -1, 128), cos, sin))


# 65537 rows: more than one launch's grid
@pytest.mark.parametrize("rows,width", [(1, 8), (7, 96), (3, 14336), (65537, 8)])
def test_swiglu_rows(cuda, rows, width):
    from pagegauge_amd import decoder as dec

    gate_up = _rand(cuda, rows, 2 * width, scale=4.0)
    gate, up = gate_up.split(width, dim=-1)
    want = F.silu(gate) * up
    got = dec._swiglu_rows(gate_up)
    # expf may differ in its last bit: one step of the FP16 activation
    assert ((got.float() - want.float()).abs() <= want.float().abs() * 2.0 ** -9 + 2.0 ** -23).all()
    assert (got != want).float().mean() < 1e-2


def test_rows_of_extreme_values(cuda):
    """Infinities, NaN and the largest values, as torch operators take them."""
    from pagegauge_amd import decoder as dec

    inf, nan = float("inf"), float("nan")
    extreme = torch.tensor([inf, -inf, nan, 65504.0, -65504.0, 6e-8, -0.0, 1.0], device=cuda).half()
    gate_up = torch.cat((extreme.repeat_interleave(8), extreme.repeat(8))).view(1, 128)
    gate, up = gate_up.split(64, dim=-1)
    assert torch.equal(dec._swiglu_rows(gate_up).nan_to_num(5.0, 7.0, -7.0),
                       (F.silu(gate) * up).nan_to_num(5.0, 7.0, -7.0))
    x = torch.stack([_rand(cuda, 64) for _ in range(8)])
    x[:, 3] = extreme
    want = dec.rms_norm(x, torch.ones(64, device=cuda).half(), 1e-5)
    got = dec._norm_rows(x, torch.ones(64, device=cuda).half(), 1e-5, None)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    got, want = (t.float().nan_to_num(0.0) for t in (got, want))
    assert ((got - want).abs() <= want.abs() * 2.0 ** -9 + 2.0 ** -23).all()


def test_prefill_with_kernels_matches_torch_operators(cuda, monkeypatch):
    from pagegauge_amd import decoder as dec

    cfg = dec.DecoderConfig(layers=2, hidden=512, q_heads=4, kv_heads=1, intermediate=96, vocab=64)
    weights = dec.DecoderWeights(cfg, 7, cuda)
    cos, sin = (t.to(cuda) for t in dec.rope_tables(77, cfg.rope_theta))
    tokens = torch.arange(77, device=cuda) % cfg.vocab
    assert dec._prefill_kernels_take(weights, tokens, cos, sin)

    def both():
        kept = []
        logits = dec.prefill(weights, tokens, cos, sin, lambda i, k, v: kept.extend((k.clone(), v.clone())))
        return [logits, *kept]

    got = both()
    monkeypatch.setattr(dec, "_prefill_kernels_take", lambda *a: False)
    monkeypatch.setattr(dec, "_attention_kernel_takes", lambda *a: False)
    want = both()
    for g, w in zip(got, want):
        # FP16 chains of two layers: a few roundings of 2^-11 apart
        assert (g.double() - w.double()).norm() <= 5e-3 * w.double().norm()
