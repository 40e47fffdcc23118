"""Weights whose shapes are not the configured ones stay off the kernels that
take their sizes from the configuration: torch operators broadcast or refuse
them as they always did, and no kernel reads past them or off the device."""

from __future__ import annotations

import pytest
import torch

CONFIG = dict(layers=2, hidden=1024, q_heads=8, kv_heads=2, intermediate=512, vocab=64)
# (layer weight or model weight, another shape)
SHAPES = [("input_norm", (1,)), ("input_norm", (512,)), ("post_norm", (1,)),
          ("post_norm", (1, 1024)), ("norm", (1,)), ("qkv", (1024, 1024)), ("qkv", (2048, 1024)),
          ("o", (1, 1024)), ("o", (2048, 1024)), ("gate_up", (2048, 1024)), ("down", (1, 512)),
          ("down", (1024, 1024)), ("embed", (64, 512)), ("lm_head", (64, 512))]


def _weights(device="cpu"):
    from pagegauge_amd import decoder as dec

    return dec.DecoderWeights(dec.DecoderConfig(**CONFIG), 5, device)


def _give(weights, name, shape, layer=1):
    w = torch.ones(shape, dtype=torch.float16, device=weights.embed.device)
    if name in weights.layers[layer]:
        weights.layers[layer][name] = w
    else:
        setattr(weights, name, w)


@pytest.mark.parametrize("name,shape", SHAPES)
def test_other_shapes_take_torch_operators(monkeypatch, name, shape):
    from pagegauge_amd import decoder as dec

    monkeypatch.setattr(dec, "_on_current_device", lambda *tensors: True)
    weights = _weights()
    cos, sin = dec.rope_tables(32, 1.0e6)
    tokens = torch.zeros(20, dtype=torch.int64)
    assert dec._prefill_kernels_take(weights, tokens, cos, sin)
    assert dec.PageGaugeDecoder._matrix_projections_take(weights, 8)
    _give(weights, name, shape)
    assert not dec._prefill_kernels_take(weights, tokens, cos, sin)
    assert not dec.PageGaugeDecoder._matrix_projections_take(weights, 8)


H = torch.float16


@pytest.mark.parametrize("weight,delta", [
    (torch.ones(1, dtype=H), None), (torch.ones(512, dtype=H), None), (torch.ones(1024), None),
    (torch.ones(2048, dtype=H)[::2], None), (torch.ones(1024, dtype=H), torch.zeros(3, 2048, dtype=H)),
    (torch.ones(1024, dtype=H), torch.zeros(1, 1024, dtype=H))])
def test_norm_rows_refuses_other_shapes(monkeypatch, weight, delta):
    from pagegauge_amd import _capi, decoder as dec

    launches = []
    monkeypatch.setattr(_capi, "call", lambda *args: launches.append(args))
    monkeypatch.setattr(_capi, "current_stream", lambda: 0)
    x = torch.zeros(3, 1024, dtype=H)
    with pytest.raises(ValueError, match="norm weight|residual"):
        dec._norm_rows(x, weight, 1e-5, delta)
    assert not launches
    dec._norm_rows(x, torch.ones(1024, dtype=H), 1e-5, torch.zeros(3, 1024, dtype=H))
    assert len(launches) == 1


def test_qkv_rope_append_needs_its_norm_weight(monkeypatch):
    """Without one the projection would run on rows that nothing normalised."""
    from pagegauge_amd import _capi, decoder as dec

    launches = []
    monkeypatch.setattr(_capi, "call", lambda *args: launches.append(args))
    pages = torch.zeros(4, 16, 1, 128, dtype=H)
    with pytest.raises(ValueError, match="norm weight"):
        dec.qkv_rope_append(torch.zeros(768, 4096, dtype=H), torch.zeros(1, 4096, dtype=H),
                            norm_weight=None, eps=1e-5, query_heads=4, kv_heads=1,
                            cos=torch.zeros(64, 128, dtype=H), sin=torch.zeros(64, 128, dtype=H),
                            positions=torch.zeros(1, dtype=torch.int32),
                            rotated_query=torch.zeros(1, 4, 128, dtype=H), key_pages=pages,
                            value_pages=pages, key_center=None, value_center=None,
                            pages_per_request=4, sink_pages=0, capacity_tokens=64)
    assert not launches


@pytest.mark.parametrize("entry", ["pg_decoder_gemv", "pg_decoder_gemm"])
def test_projections_refuse_host_operands(monkeypatch, entry):
    """A weight left on the host raises, as it does in torch operators."""
    from pagegauge_amd import _capi, decoder as dec

    launches = []
    monkeypatch.setattr(_capi, "call", lambda *args: launches.append(args))
    monkeypatch.setattr(_capi, "current_stream", lambda: 0)
    with pytest.raises(ValueError, match="one CUDA device"):
        dec._projection(entry, torch.zeros(16, 512, dtype=H), torch.zeros(6, 512, dtype=H),
                        torch.zeros(6, 16, dtype=H), None, 1e-5, False, None)
    assert not launches


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["input_norm", "post_norm", "norm"])
def test_one_element_norm_weights_broadcast(cuda, name):
    """A one-element norm weight of ones is the full weight of ones."""
    from pagegauge_amd import decoder as dec

    weights = _weights(cuda)
    cos, sin = (t.to(cuda) for t in dec.rope_tables(304, 1.0e6))
    prompt = torch.arange(300, device=cuda) % CONFIG["vocab"]
    want = dec.prefill(weights, prompt, cos, sin)
    for layer in range(2):
        _give(weights, name, (1,), layer)
    got = dec.prefill(weights, prompt, cos, sin)
    # FP16 chains of two layers through kernels and through torch operators
    assert (got.double() - want.double()).norm() <= 5e-3 * want.double().norm()
    cache = dec.Fp16Cache(weights.config, 6, 19, cuda)
    steps = dec.PageGaugeDecoder(weights, cache, "fp16", 304, cos, sin, batch_size=6)
    assert not steps.batched
    assert steps.step(prompt[:6], 0).isfinite().all()
