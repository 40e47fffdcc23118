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


@pytest.mark.parametrize("batch,hidden", [(3, 4096), (4, 4096), (5, 4096), (16, 4096), (16, 1024)])
@pytest.mark.parametrize("centered", [True, False])
def test_rope_append_takes_a_position_per_row(cuda, batch, hidden, centered):
    """Each row at its own position (a prefix page, page ends and the last
    token among them) against the projection and a one-row cache update; rows
    at, past and before the cache's range write nothing.  Up to 4 rows through
    ``qkv_rope_append``, more through the 16-row entry."""
    from pagegauge_amd import decoder as dec
    from pagegauge_amd.runtime import load_append_extension

    print(f"append positions batch={batch} hidden={hidden} centered={centered}", flush=True)
    hkv = hidden // 512
    hq, pages, ring, sink = 4 * hkv, 6, 4 if centered else 6, 1 if centered else 0
    w = _rand(cuda, (hq + 2 * hkv) * 128, hidden, scale=0.02)
    x, g = _rand(cuda, batch, hidden), _rand(cuda, hidden)
    if hidden != 4096:
        x, g = dec.rms_norm(x, g, 1e-5), None
    cos, sin = (t.to(cuda) for t in dec.rope_tables(pages * 16, 1.0e6))
    where = [37, 10_000, -1, 95, 0, 96, 15, 16, 63, 64, 2 ** 31 - 1, 80, -2 ** 31, 31, 5, 50][:batch]
    positions = torch.tensor(where, device=cuda, dtype=torch.int32)
    kc, vc = ((_rand(cuda, batch, hkv, 128, scale=s) if centered else None) for s in (0.1, 0.2))
    got, want = ([torch.full((batch, hq, 128), 7.0, device=cuda, dtype=torch.float16),
                  torch.full((batch * ring, 16, hkv, 128), 7.0, device=cuda, dtype=torch.float16),
                  torch.full((batch * ring, 16, hkv, 128), 7.0, device=cuda, dtype=torch.float16)]
                 for _ in range(2))
    if batch <= 4:
        dec.qkv_rope_append(w, x, norm_weight=g, eps=1e-5, query_heads=hq, kv_heads=hkv, cos=cos,
                            sin=sin, positions=positions, rotated_query=got[0], key_pages=got[1],
                            value_pages=got[2], key_center=kc, value_center=vc,
                            pages_per_request=ring, sink_pages=sink, capacity_tokens=pages * 16)
    else:
        dec._qkv_rope_append("pg_decoder_gemm_rope_append", w, x, g, 1e-5, hq, hkv, cos, sin,
                             positions, *got, kc, vc, ring, sink, pages * 16)
    qkv = _gemm(w, x, torch.empty(batch, w.shape[0], device=cuda, dtype=torch.float16), norm=g)
    ext = load_append_extension()
    for b, position in enumerate(where):
        if not 0 <= position < pages * 16:
            continue
        q, k, v = (t.reshape(1, -1, 128) for t in
                   qkv[b].split([hq * 128, hkv * 128, hkv * 128], dim=-1))
        row = (q, k, v, cos, sin, positions[b:b + 1])
        mine = [want[0][b:b + 1], *(t[b * ring:(b + 1) * ring] for t in want[1:])]
        if centered:
            codes = [torch.zeros(pages, 16, hkv, 128, device=cuda, dtype=torch.int8) for _ in range(2)]
            scales = [torch.zeros(pages, hkv, device=cuda, dtype=torch.float16) for _ in range(2)]
            ext.rope_append_page_gauge_dynamic(*row, kc[b:b + 1], vc[b:b + 1], *mine, *codes,
                                               *scales, sink)
        else:
            ext.rope_append_fp16_dynamic(*row, *mine)
    for a, b in zip(got, want):
        assert torch.equal(a, b) and (a != 7.0).any()


def _batched_pair(dec, device, batch, hidden, tail, prompt_tokens, steps):
    """Two batched decoders over the same prompt's caches."""
    heads = hidden // 128
    cfg = dec.DecoderConfig(layers=2, hidden=hidden, q_heads=heads, kv_heads=heads // 4,
                            intermediate=512, vocab=512)
    weights = dec.DecoderWeights(cfg, seed=9, device=device)
    gen = torch.Generator().manual_seed(10)
    prompt = torch.randint(0, cfg.vocab, (batch, prompt_tokens), generator=gen)
    first, _, built = dec.build_decoders(weights, prompt, steps + 1, backends=("page_gauge",))
    base = built["page_gauge"]
    pair = [dec.PageGaugeDecoder(weights, base.cache.clone(), "page_gauge", base.max_pages * 16,
                                 base.rope_cos, base.rope_sin, batch_size=batch,
                                 tail_attention=tail) for _ in range(2)]
    assert all(d.batched and d.fused_append for d in pair)
    return first, weights, pair


@pytest.mark.parametrize("batch,hidden,tail", [
    (6, 1024, "segmented"), (6, 1024, "heterogeneous"), (5, 4096, "segmented"),
    (16, 4096, "heterogeneous")])
def test_batched_graph_replay_is_bitwise_eager(cuda, batch, hidden, tail):
    """Captured steps across the close of a page, each replay checked against
    an eager step run beside it; then the caches."""
    from pagegauge_amd import decoder as dec

    print(f"batched graph batch={batch} hidden={hidden} tail={tail}", flush=True)
    steps = 20
    token, _, (eager, graphed) = _batched_pair(dec, cuda, batch, hidden, tail, 304, steps)
    for i in range(steps):
        want = eager.step(token, 304 + i).clone()
        if graphed.plan_signature_after(304 + i) not in graphed.graph_bank:
            graphed.capture(304 + i)
        got = graphed.step(token, 304 + i)
        torch.cuda.synchronize()
        assert torch.equal(got, want), i
        assert torch.equal(graphed.graph_next, want.argmax(-1)), i
        token = want.argmax(-1)
    assert graphed.graph_replays == steps and len(graphed.graph_bank) >= 2
    for name in ("key_codes", "value_codes", "key_scales", "value_scales", "exact_key", "exact_value"):
        assert torch.equal(getattr(eager.cache, name), getattr(graphed.cache, name)), name
    assert eager.cache.key_scales[:, 19::eager.max_pages].abs().min() > 0   # closed at 319


def test_batched_generate_matches_eager_steps(cuda):
    from pagegauge_amd import decoder as dec

    first, _, (eager, graphed) = _batched_pair(dec, cuda, 6, 1024, "segmented", 304, 20)
    tokens, logits = graphed.generate(first, 304, 18)
    token = first
    for i in range(18):
        want = eager.step(token, 304 + i)
        assert torch.equal(logits[i], want), i
        token = want.argmax(-1)
        assert torch.equal(tokens[i], token), i


@pytest.mark.parametrize("batch,tail", [(5, "segmented"), (16, "heterogeneous")])
def test_batched_steps_at_the_resident_width(cuda, batch, tail):
    """Hidden 4096: the norm in the projection, the input resident, against
    the torch-operator step (bounds as at the streamed width above)."""
    from pagegauge_amd import decoder as dec

    token, weights, (fast, other) = _batched_pair(dec, cuda, batch, 4096, tail, 304, 6)
    plain = dec.PageGaugeDecoder(weights, other.cache, "page_gauge", other.max_pages * 16,
                                 other.rope_cos, other.rope_sin, batch_size=batch, fused=False,
                                 tail_attention=tail)
    for i in range(4):
        a, b = fast.step(token, 304 + i), plain.step(token, 304 + i)
        assert float((a - b).abs().max()) <= 0.02 * max(1.0, float(b.abs().max())), i
        assert float(F.cosine_similarity(a, b, dim=-1).min()) > 0.9999
        token = b.argmax(-1)
