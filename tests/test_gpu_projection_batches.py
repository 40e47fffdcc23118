"""The matrix-core projections (2 to 16 input rows): tile and slice edges
against float64, the fused cache update against projection plus update, and
whole steps against the torch-operator step."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _rand(device, *shape, scale=1.0):
    gen = torch.Generator(device=device).manual_seed(sum(shape))
    return (torch.randn(*shape, device=device, generator=gen) * scale).half()


def _gemm(w, x, out, norm=None, swiglu=False, residual=None):
    from pagegauge_amd import decoder as dec

    return dec._projection("pg_decoder_gemm", w, x, out, norm, 1e-5, swiglu, residual)


# 16-row tiles (8 output rows with SwiGLU) whole and ragged, fewer and more
# tiles than workgroups; widths: resident (4096), streamed with whole blocks
# of 4 steps (8192, 14336), half blocks (512, 1536) and more than one tile of them
@pytest.mark.parametrize("n,k", [(1, 512), (15, 1536), (16, 4096), (17, 4096), (4104, 4096),
                                 (8200, 4096), (4100, 512), (40, 8192), (33, 14336)])
@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 15, 16])
def test_gemm_matches_float64(cuda, n, k, batch):
    print(f"gemm n={n} k={k} batch={batch}", flush=True)
    w, x, res = _rand(cuda, n, k, scale=0.02), _rand(cuda, batch, k), _rand(cuda, batch, n)
    want = x.double() @ w.double().t()
    # one FP16 rounding of a float32 sum of k products (error below k * 2^-24
    # of the sum of magnitudes, in practice its square root)
    slack = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    out = _gemm(w, x, torch.full_like(res, float("nan")))
    assert ((out.double() - want).abs() <= want.abs() * 2.0 ** -11 + slack + 2.0 ** -25).all()
    wide = _gemm(w, x, torch.empty(batch, n, device=cuda, dtype=torch.float32))
    assert torch.equal(wide, out.float())
    hidden = res.clone()
    _gemm(w, x, hidden, residual=hidden)                       # in place
    assert torch.equal(hidden, res + out)


@pytest.mark.parametrize("n,k", [(2, 512), (34, 1536), (2, 4096), (4096, 4096), (4112, 4096)])
@pytest.mark.parametrize("batch", [2, 7, 16])
def test_gemm_norm_and_swiglu(cuda, n, k, batch):
    from pagegauge_amd.decoder import rms_norm

    w, x, g = _rand(cuda, n, k, scale=0.02), _rand(cuda, batch, k, scale=3.0), _rand(cuda, k)
    if k != 4096:                                              # the norm goes first
        with pytest.raises(RuntimeError, match="4096-wide"):
            _gemm(w, x, torch.empty(batch, n, device=cuda, dtype=torch.float16), norm=g)
        x, g = rms_norm(x, g, 1e-5), None
    normed = (x if g is None else rms_norm(x, g, 1e-5)).double()
    # a normalised element may round the other way (rsqrt): 2^-10 of it
    slack = 2.0 ** -10 * (normed.abs() @ w.double().abs().t()) * 4 * k ** -0.5
    want = normed @ w.double().t()
    out = _gemm(w, x, torch.empty(batch, n, device=cuda, dtype=torch.float16), norm=g)
    assert ((out.double() - want).abs() <= want.abs() * 2.0 ** -11 + slack + 2.0 ** -20).all()
    gate, up = out.split(n // 2, dim=-1)
    act = _gemm(w, x, torch.empty(batch, n // 2, device=cuda, dtype=torch.float16), norm=g,
                swiglu=True)
    # the same sums (the tile's row order differs, not the order of k), SiLU to
    # one step of FP16
    ref = (F.silu(gate) * up).float()
    assert ((act.float() - ref).abs() <= ref.abs() * 2.0 ** -9 + 2.0 ** -20).all()


@pytest.mark.parametrize("batch,hidden", [(3, 4096), (5, 4096), (16, 4096), (7, 1024)])
@pytest.mark.parametrize("centered", [True, False])
def test_gemm_rope_append_is_gemm_then_cache_update(cuda, batch, hidden, centered):
    from pagegauge_amd import decoder as dec
    from pagegauge_amd.runtime import load_append_extension

    print(f"gemm append batch={batch} hidden={hidden} centered={centered}", flush=True)
    hkv = hidden // 512
    hq, pages, ring, sink = 4 * hkv, 6, 4 if centered else 6, 1 if centered else 0
    w = _rand(cuda, (hq + 2 * hkv) * 128, hidden, scale=0.02)
    x, g = _rand(cuda, batch, hidden), _rand(cuda, hidden)
    cos, sin = (t.to(cuda) for t in dec.rope_tables(pages * 16, 1.0e6))
    position = torch.full((1,), 37, device=cuda, dtype=torch.int32)
    kc, vc = _rand(cuda, batch, hkv, 128, scale=0.1), _rand(cuda, batch, hkv, 128, scale=0.2)
    got, want = ([torch.zeros(batch, hq, 128, device=cuda, dtype=torch.float16),
                  torch.zeros(batch * ring, 16, hkv, 128, device=cuda, dtype=torch.float16),
                  torch.zeros(batch * ring, 16, hkv, 128, device=cuda, dtype=torch.float16)]
                 for _ in range(2))
    if hidden != 4096:
        x, g = dec.rms_norm(x, g, 1e-5), None
    dec._qkv_rope_append("pg_decoder_gemm_rope_append", w, x, g, 1e-5, hq, hkv, cos, sin, position,
                         *got, kc if centered else None, vc if centered else None, ring, sink,
                         pages * 16)
    qkv = _gemm(w, x, torch.empty(batch, w.shape[0], device=cuda, dtype=torch.float16), norm=g)
    q, k, v = (t.reshape(batch, -1, 128) for t in
               qkv.split([hq * 128, hkv * 128, hkv * 128], dim=-1))
    ext = load_append_extension()
    if centered:
        codes = [torch.zeros(batch * pages, 16, hkv, 128, device=cuda, dtype=torch.int8) for _ in range(2)]
        scales = [torch.zeros(batch * pages, hkv, device=cuda, dtype=torch.float16) for _ in range(2)]
        ext.rope_append_page_gauge_dynamic(q.contiguous(), k.contiguous(), v.contiguous(), cos, sin,
                                           position, kc, vc, *want, *codes, *scales, sink)
    else:
        ext.rope_append_fp16_dynamic(q.contiguous(), k.contiguous(), v.contiguous(), cos, sin,
                                     position, *want)
    for a, b in zip(got, want):
        assert torch.equal(a, b) and a.abs().sum() > 0


@pytest.mark.parametrize("batch,backend", [(6, "page_gauge"), (16, "page_gauge"), (9, "fp16")])
def test_batched_steps_match_torch_operator_steps(cuda, batch, backend):
    """Across a page's end, so that the finalize runs in the decode."""
    from pagegauge_amd import decoder as dec

    cfg = dec.DecoderConfig(layers=2, hidden=1024, q_heads=8, kv_heads=2, intermediate=1536, vocab=512)
    weights = dec.DecoderWeights(cfg, seed=3, device=cuda)
    prompt = torch.randint(0, cfg.vocab, (batch, 304), generator=torch.Generator().manual_seed(4))
    first, _, decoders = dec.build_decoders(weights, prompt, 20, backends=(backend,))
    fast = decoders[backend]
    plain = dec.PageGaugeDecoder(weights, fast.cache.clone(), backend, fast.max_pages * 16,
                                 fast.rope_cos, fast.rope_sin, batch_size=batch, fused=False)
    assert fast.batched and not plain.batched and not fast.fused
    # what the attribute says is what a step does: the QKV projection carries the update
    assert fast.fused_append and not plain.fused_append
    token, kept = first, []
    for i in range(18):
        a, b = fast.step(token, 304 + i), plain.step(token, 304 + i)
        kept.append((a, a.clone()))
        assert float((a - b).abs().max()) <= 0.02 * max(1.0, float(b.abs().max())), i
        assert float(F.cosine_similarity(a, b, dim=-1).min()) > 0.9999
        token = b.argmax(-1)
    assert all(torch.equal(a, b) for a, b in kept)             # every step's logits are its own
    if backend == "page_gauge":
        # the page that closed at position 319 was finalized: scales within the
        # FP16 roundings of two steps' chains
        assert torch.allclose(fast.cache.key_scales.float(), plain.cache.key_scales.float(), rtol=0.02)
