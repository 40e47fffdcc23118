"""The work that a program on this package has it do, as cases to be timed.

Every case goes through the package's public entry points on a Mistral-7B
shaped layer (32 query heads, 8 KV heads, head_dim 128, 16-token pages), the
shape of the package's own configurations and benchmark:

* ``decode``: one attention call of a decode step over paged KV: INT8 history
  with an FP16 exact tail (segmented), the same over one unified table
  (heterogeneous), or plain FP16 pages;
* ``append``: the cache update of one decode step (RoPE, centered append,
  finalize of the pages that close);
* ``populate``: one layer of a prompt's K/V into the compressed cache;
* ``step``: a whole decode step of the decoder (four layers and the head);
* ``prefill``: a prompt through the decoder (two layers and the head).

``listed`` gives the named cases, ``draw`` more of the same ranges.
``prepare`` makes what a program holds before the call, ``run`` is one pass,
``work`` the bytes and operations it cannot do without, ``tolerance`` how far
another correct implementation may be off, and ``exact`` the same outputs in
64 bits from plain torch.
"""

import math
import random

import torch

HQ, HKV, DIM, PAGE = 32, 8, 128, 16
TAIL_PAGES = 16
SM_SCALE = DIM ** -0.5
WORKSPACE_BYTES = 256 << 20
ROPE_THETA = 1.0e6
PREFILL_LAYERS = 2
STEP_LAYERS = 4


def listed():
    return [
        # a chat turn on a short context: the smallest attention call, where
        # launches and latency count
        {"name": "decode_b1_4k", "op": "decode", "kind": "segmented", "batch": 1, "low": 4096,
         "high": 4096, "ragged": 0},
        # one user with a long document: the benchmark's headline shape
        {"name": "decode_b1_49k", "op": "decode", "kind": "segmented", "batch": 1, "low": 49152,
         "high": 49152, "ragged": 0},
        # four long requests through the one-table kernel
        {"name": "decode_het_b4_20k", "op": "decode", "kind": "heterogeneous", "batch": 4,
         "low": 20480, "high": 20480, "ragged": 0},
        # eight ragged requests on an uncompressed cache (the FP16 backend)
        {"name": "decode_fp16_b8", "op": "decode", "kind": "fp16", "batch": 8, "low": 4096,
         "high": 32768, "ragged": 1},
        # a serving batch of short requests
        {"name": "decode_b256_serving", "op": "decode", "kind": "segmented", "batch": 256,
         "low": 512, "high": 4096, "ragged": 2},
        # the cache update of eight requests at a page's last token
        {"name": "append_b8", "op": "append", "batch": 8, "mode": "dynamic", "position": 4095},
        # a 16K prompt's K/V of one layer into the compressed cache
        {"name": "populate_16k", "op": "populate", "pages": 1024, "sink": 0},
        # single-user decoding behind a 16K prompt
        {"name": "step_b1_16k", "op": "step", "batch": 1, "context": 16391},
        # four 20K requests in lockstep
        {"name": "step_b4_20k", "op": "step", "batch": 4, "context": 20480},
        # sixteen 4K requests in lockstep, at a page's last token
        {"name": "step_b16_4k", "op": "step", "batch": 16, "context": 4095},
        # a short and a long prompt
        {"name": "prefill_1k", "op": "prefill", "tokens": 1000},
        {"name": "prefill_16k", "op": "prefill", "tokens": 16384},
    ]


def draw(rng):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    op = rng.choice(["decode", "decode", "decode", "append", "populate", "step", "prefill"])
    if op == "decode":
        batch = spread(1, 256)
        top = min(65536, 560000 // batch)
        high = spread(min(1024, top), top)
        low = spread(288, high)
        return {"op": op, "kind": rng.choice(["segmented", "heterogeneous", "fp16"]),
                "batch": batch, "low": low, "high": high, "ragged": rng.randrange(1 << 20)}
    if op == "append":
        return {"op": op, "batch": spread(1, 256), "mode": rng.choice(["dynamic", "positions"]),
                "position": rng.choice([spread(272, 4080), 16 * spread(17, 255) - 1])}
    if op == "populate":
        return {"op": op, "pages": spread(20, 1024), "sink": rng.choice([0, 0, 1, 2])}
    if op == "step":
        batch = spread(1, 16)
        return {"op": op, "batch": batch, "context": spread(288, min(32768, 80000 // batch))}
    return {"op": op, "tokens": spread(64, 16384)}


# -- sizes -------------------------------------------------------------------

def _lengths(case):
    """Context tokens of each request."""
    rng = random.Random(case["ragged"])
    return [rng.randint(case["low"], case["high"]) for _ in range(case["batch"])]


def _page_counts(case):
    """(old INT8 pages, exact pages) of each request: the newest 16 pages, the
    last perhaps partial, are exact; FP16 caches have exact pages only."""
    pages = [-(-n // PAGE) for n in _lengths(case)]
    if case["kind"] == "fp16":
        return [0] * len(pages), pages
    return [p - TAIL_PAGES for p in pages], [TAIL_PAGES] * len(pages)


def _step_pages(case):
    return -(-(case["context"] + 1) // PAGE)


def _config(layers):
    from pagegauge_amd.decoder import DecoderConfig

    return DecoderConfig(layers=layers)


_HIDDEN, _MLP, _VOCAB = 4096, 14336, 32768
_LAYER_WEIGHTS = (HQ + 2 * HKV) * DIM * _HIDDEN + _HIDDEN * _HIDDEN + 3 * _HIDDEN * _MLP


def work(case):
    op = case["op"]
    kv_row = 2 * HKV * DIM                       # K and V values of one token
    if op == "decode":
        old, exact = (sum(c) for c in _page_counts(case))
        batch = case["batch"]
        return {"bytes": old * (PAGE * kv_row + 4 * HKV) + exact * PAGE * kv_row * 2
                + 4 * (old + exact) + batch * (HQ * DIM * 4 + HQ * 4 + HKV * DIM * 2),
                "flops": 4.0 * sum(_lengths(case)) * HQ * DIM}
    if op == "append":
        batch = case["batch"]
        # q, k, v and the centers in; rotated q, the ring rows out
        moved = batch * (HQ * DIM * 4 + kv_row * 2 * 3) + DIM * 4
        if case["position"] % PAGE == PAGE - 1:  # the closing pages in, their codes out
            closing = batch if case["mode"] == "dynamic" else -(-batch // PAGE)
            moved += closing * (PAGE * kv_row * 3 + 4 * HKV)
        return {"bytes": moved, "flops": 3.0 * batch * (HQ + HKV) * DIM}
    if op == "populate":
        tokens = case["pages"] * PAGE
        exact = (TAIL_PAGES + case["sink"]) * PAGE
        return {"bytes": tokens * kv_row * 3 + case["pages"] * 4 * HKV + exact * kv_row * 2,
                "flops": 4.0 * tokens * kv_row}
    if op == "step":
        pages, batch = _step_pages(case), case["batch"]
        kv = batch * ((pages - TAIL_PAGES) * (PAGE * kv_row + 4 * HKV)
                      + TAIL_PAGES * PAGE * kv_row * 2)
        weights = STEP_LAYERS * _LAYER_WEIGHTS + _VOCAB * _HIDDEN
        return {"bytes": STEP_LAYERS * kv + 2 * weights + batch * _VOCAB * 4,
                "flops": 2.0 * batch * weights
                + 4.0 * STEP_LAYERS * batch * (case["context"] + 1) * HQ * DIM}
    tokens = case["tokens"]
    return {"bytes": 2 * (PREFILL_LAYERS * (_LAYER_WEIGHTS + tokens * kv_row) + _VOCAB * _HIDDEN
                          + tokens * _HIDDEN),
            "flops": PREFILL_LAYERS * (2.0 * tokens * _LAYER_WEIGHTS
                                       + 2.0 * tokens * (tokens + 1) * HQ * DIM)
            + 2.0 * _VOCAB * _HIDDEN}


def tolerance(case):
    # the update paths are bit for bit what they are defined as
    if case["op"] in ("append", "populate"):
        return "exact"
    # FP16 outputs of float32 sums: 2.2e-4 off 64 bits, four times that
    if case["op"] == "decode":
        return {"rel": 1e-3, "max": 1e-2}
    # logits behind a chain of FP16 roundings (two to four layers): 1.6e-3 to
    # 2.8e-3 off 64 bits, four times that; a code on a rounding boundary may
    # fall either way
    return {"rel": 1e-2, "max": 6e-2, "differ": 1e-3}


# -- inputs ------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _channel_gain(gen):
    """Four of a head's 128 channels carry outliers, as cached keys and values do."""
    gain = torch.ones(DIM, device="cuda")
    gain[torch.randperm(DIM, device="cuda", generator=gen)[:4]] = 8.0
    return gain


def _normal(gen, *shape):
    return torch.randn(*shape, device="cuda", generator=gen)


def _fp16_pages(gen, gain, pages):
    out = torch.empty(pages, PAGE, HKV, DIM, device="cuda", dtype=torch.float16)
    for begin in range(0, pages, 4096):
        part = out[begin:begin + 4096]
        part.copy_(_normal(gen, *part.shape) * gain)
    return out


def _int8_pages(gen, gain, pages):
    """Codes and FP16 scales of centered pages (round(x / scale) to +-127)."""
    codes = torch.empty(pages, PAGE, HKV, DIM, device="cuda", dtype=torch.int8)
    scales = torch.empty(pages, HKV, device="cuda", dtype=torch.float16)
    for begin in range(0, pages, 4096):
        part = codes[begin:begin + 4096]
        x = _normal(gen, *part.shape) * gain
        scale = (x.abs().amax(dim=(1, 3)) / 127.0).half()
        scales[begin:begin + 4096] = scale
        part.copy_((x / scale.float()[:, None, :, None]).round().clamp(-127, 127))
    return codes, scales


def _indptr(counts):
    return torch.tensor([0] + list(counts), dtype=torch.int64).cumsum(0).to(torch.int32).cuda()


def _permutation(gen, count):
    return torch.randperm(count, device="cuda", generator=gen).to(torch.int32)


def _rope(positions):
    inverse = 1.0 / (ROPE_THETA ** (torch.arange(0, DIM, 2).float() / DIM))
    angles = torch.arange(positions).float()[:, None] * inverse[None, :]
    angles = torch.cat((angles, angles), dim=-1)
    return angles.cos().half().cuda(), angles.sin().half().cuda()


def _decode_inputs(case, seed):
    gen = _generator(seed)
    batch, lengths = case["batch"], _lengths(case)
    old, exact = _page_counts(case)
    gain_k, gain_v = _channel_gain(gen), _channel_gain(gen)
    s = {"case": case,
         "query": _normal(gen, batch, HQ, DIM).half(),
         "exact_indptr": _indptr(exact), "exact_indices": _permutation(gen, sum(exact)),
         "last_len": torch.tensor([(n - 1) % PAGE + 1 for n in lengths], dtype=torch.int32).cuda(),
         "exact_k": _fp16_pages(gen, gain_k, sum(exact)),
         "exact_v": _fp16_pages(gen, gain_v, sum(exact)),
         "out": torch.empty(batch, HQ, DIM, device="cuda", dtype=torch.float16),
         "lse": torch.empty(batch, HQ, device="cuda", dtype=torch.float32)}
    if case["kind"] != "fp16":
        s["old_indptr"], s["old_indices"] = _indptr(old), _permutation(gen, sum(old))
        s["k_codes"], s["k_scale"] = _int8_pages(gen, gain_k, sum(old))
        s["v_codes"], s["v_scale"] = _int8_pages(gen, gain_v, sum(old))
        s["center"] = (_normal(gen, batch, HKV, DIM) * 0.1).half()
    return s


def _append_inputs(case, seed):
    gen = _generator(seed)
    batch, position = case["batch"], case["position"]
    code_pages = position // PAGE + 1
    if case["mode"] == "dynamic":
        positions = torch.tensor([position], dtype=torch.int32)
    else:  # requests at different tokens of their pages
        positions = position - torch.arange(batch, dtype=torch.int32) % PAGE
    fused = _normal(gen, batch, (HQ + 2 * HKV) * DIM).half()
    cos, sin = _rope(position + 1)
    return {"case": case, "positions": positions.cuda(), "cos": cos, "sin": sin,
            "q": fused[:, :HQ * DIM].view(batch, HQ, DIM),
            "k": fused[:, HQ * DIM:(HQ + HKV) * DIM].view(batch, HKV, DIM),
            "v": fused[:, (HQ + HKV) * DIM:].view(batch, HKV, DIM),
            "k_center": (_normal(gen, batch, HKV, DIM) * 0.1).half(),
            "v_center": (_normal(gen, batch, HKV, DIM) * 0.1).half(),
            "rotated": torch.zeros(batch, HQ, DIM, device="cuda", dtype=torch.float16),
            "ring_k": _normal(gen, batch * TAIL_PAGES, PAGE, HKV, DIM).half(),
            "ring_v": _normal(gen, batch * TAIL_PAGES, PAGE, HKV, DIM).half(),
            "codes": [torch.zeros(batch * code_pages, PAGE, HKV, DIM, device="cuda",
                                  dtype=torch.int8) for _ in range(2)],
            "scales": [torch.zeros(batch * code_pages, HKV, device="cuda", dtype=torch.float16)
                       for _ in range(2)]}


def _prompt_kv(gen, gain_k, gain_v, tokens):
    """Keys as RoPE leaves them (dense) and values as a slice of the fused
    QKV projection (strided), token-major."""
    key = (_normal(gen, tokens, HKV, DIM) * gain_k + _normal(gen, HKV, DIM) * 0.5).half()
    fused = torch.empty(tokens, (HQ + 2 * HKV) * DIM, device="cuda", dtype=torch.float16)
    value = fused[:, (HQ + HKV) * DIM:].view(tokens, HKV, DIM)
    value.copy_(_normal(gen, tokens, HKV, DIM) * gain_v + _normal(gen, HKV, DIM) * 0.5)
    return key, value


def _step_inputs(case, seed):
    from pagegauge_amd.decoder import DecoderWeights, GaugeCache

    gen = _generator(seed)
    config = _config(STEP_LAYERS)
    batch, pages = case["batch"], _step_pages(case)
    weights = DecoderWeights(config, seed)
    cache = GaugeCache(config, batch, pages, TAIL_PAGES)
    gain_k, gain_v = _channel_gain(gen), _channel_gain(gen)
    prompt_pages = case["context"] // PAGE
    for layer in range(STEP_LAYERS):
        for request in range(batch):
            cache.populate(layer, request, *_prompt_kv(gen, gain_k, gain_v, prompt_pages * PAGE))
    cos, sin = _rope(pages * PAGE)
    token = torch.randint(0, config.vocab, (batch,), device="cuda", generator=gen)
    return {"case": case, "weights": weights, "cache": cache, "cos": cos, "sin": sin,
            "token": token}


def _prefill_inputs(case, seed):
    from pagegauge_amd.decoder import DecoderWeights

    config = _config(PREFILL_LAYERS)
    cos, sin = _rope(case["tokens"])
    shape = (PREFILL_LAYERS, case["tokens"], HKV, DIM)
    return {"case": case, "weights": DecoderWeights(config, seed), "cos": cos, "sin": sin,
            "tokens": torch.randint(0, config.vocab, (case["tokens"],), device="cuda",
                                    generator=_generator(seed)),
            "key": torch.zeros(shape, device="cuda", dtype=torch.float16),
            "value": torch.zeros(shape, device="cuda", dtype=torch.float16)}


def _unified_table(s):
    """Each request's INT8 page ids, then its exact page ids."""
    old, exact = _page_counts(s["case"])
    parts = [part for pair in zip(torch.split(s["old_indices"], old),
                                  torch.split(s["exact_indices"], exact)) for part in pair]
    return _indptr([a + b for a, b in zip(old, exact)]), torch.cat(parts)


def prepare(case, seed):
    op = case["op"]
    if op == "append":
        from pagegauge_amd.runtime import load_append_extension

        s = _append_inputs(case, seed)
        s["extension"] = load_append_extension()
        return s
    if op == "populate":
        from pagegauge_amd.decoder import GaugeCache

        gen = _generator(seed)
        key, value = _prompt_kv(gen, _channel_gain(gen), _channel_gain(gen), case["pages"] * PAGE)
        return {"case": case, "key": key, "value": value,
                "cache": GaugeCache(_config(1), 1, case["pages"], TAIL_PAGES, case["sink"])}
    if op == "step":
        from pagegauge_amd.decoder import PageGaugeDecoder

        s = _step_inputs(case, seed)
        s["decoder"] = PageGaugeDecoder(s["weights"], s["cache"], "page_gauge",
                                        case["context"] + 1, s["cos"], s["sin"],
                                        exact_tail=TAIL_PAGES * PAGE, batch_size=case["batch"])
        return s
    if op == "prefill":
        return _prefill_inputs(case, seed)

    from pagegauge_amd import decode

    s = _decode_inputs(case, seed)
    workspace = torch.empty(WORKSPACE_BYTES, device="cuda", dtype=torch.uint8)
    if case["kind"] == "segmented":
        d = decode.PageGaugeSegmentedDecode(workspace)
        s["old_last"] = torch.full((case["batch"],), PAGE, device="cuda", dtype=torch.int32)
        d.plan(s["old_indptr"], s["old_indices"], s["old_last"], s["exact_indptr"],
               s["exact_indices"], s["last_len"])
    elif case["kind"] == "heterogeneous":
        d = decode.HeterogeneousDecodeWrapper(workspace)
        s["indptr"], s["indices"] = _unified_table(s)
        s["old_kv_len"] = torch.tensor(_page_counts(case)[0], dtype=torch.int32).cuda() * PAGE
        d.plan(s["indptr"], s["indices"], s["last_len"], exact_tail_pages_hint=TAIL_PAGES)
    else:
        d = decode.BatchDecodeWithPagedKVCacheWrapper(workspace, "NHD")
        d.plan(s["exact_indptr"], s["exact_indices"], s["last_len"], HQ, HKV, DIM, PAGE,
               kv_data_type=torch.float16)
    s["decode"] = d
    return s


# -- one pass ----------------------------------------------------------------

@torch.inference_mode()
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "decode":
        d = s["decode"]
        if case["kind"] == "segmented":
            d.run(s["query"], (s["k_codes"], s["v_codes"]), s["k_scale"], s["v_scale"],
                  (s["exact_k"], s["exact_v"]), s["center"], out=s["out"], lse=s["lse"])
        elif case["kind"] == "heterogeneous":
            d.run(s["query"], (s["k_codes"], s["v_codes"]), s["k_scale"], s["v_scale"],
                  s["exact_k"], s["exact_v"], s["old_kv_len"], s["center"], out=s["out"],
                  lse=s["lse"])
        else:
            d.run(s["query"], (s["exact_k"], s["exact_v"]), out=s["out"], lse=s["lse"])
        return {"out": s["out"], "lse": s["lse"]}
    if op == "append":
        call = (s["extension"].rope_append_page_gauge_dynamic if case["mode"] == "dynamic"
                else s["extension"].rope_append_page_gauge_positions)
        call(s["q"], s["k"], s["v"], s["cos"], s["sin"], s["positions"], s["k_center"],
             s["v_center"], s["rotated"], s["ring_k"], s["ring_v"], *s["codes"], *s["scales"], 0)
        return {"rotated": s["rotated"], "ring_k": s["ring_k"], "ring_v": s["ring_v"],
                "codes": s["codes"], "scales": s["scales"]}
    if op == "populate":
        c = s["cache"]
        c.populate(0, 0, s["key"], s["value"])
        return {"key_center": c.key_center, "value_center": c.value_center,
                "key_codes": c.key_codes, "value_codes": c.value_codes,
                "key_scales": c.key_scales, "value_scales": c.value_scales,
                "exact_key": c.exact_key, "exact_value": c.exact_value}
    if op == "step":
        c = s["cache"]
        logits = s["decoder"].step(s["token"], case["context"])
        return {"logits": logits, "exact_key": c.exact_key, "exact_value": c.exact_value,
                "key_codes": c.key_codes, "value_codes": c.value_codes,
                "key_scales": c.key_scales, "value_scales": c.value_scales}

    from pagegauge_amd.decoder import prefill

    def keep(layer, key, value):
        s["key"][layer].copy_(key)
        s["value"][layer].copy_(value)

    logits = prefill(s["weights"], s["tokens"], s["cos"], s["sin"], keep)
    return {"logits": logits, "key": s["key"], "value": s["value"]}


# -- the same in 64 bits -----------------------------------------------------

def _attend(query, key, value):
    """(output [HQ, DIM], base-2 lse [HQ]) of query [HQ, DIM] over [T, HKV, DIM]."""
    group = HQ // HKV
    out, lse = [], []
    for h in range(HKV):
        scores = (query[group * h:group * (h + 1)] @ key[:, h].t()) * (SM_SCALE / math.log(2.0))
        top = scores.amax(dim=-1, keepdim=True)
        p = torch.exp2(scores - top)
        total = p.sum(dim=-1, keepdim=True)
        out.append((p / total) @ value[:, h])
        lse.append((top + torch.log2(total)).squeeze(-1))
    return torch.cat(out), torch.cat(lse)


def _rotate(x, cos, sin):
    """RoPE of [..., H, DIM] rows with [..., DIM] tables."""
    turned = torch.cat((-x[..., DIM // 2:], x[..., :DIM // 2]), dim=-1)
    return x * cos.unsqueeze(-2) + turned * sin.unsqueeze(-2)


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _linear(x, weight):
    return x @ weight.double().t()


def _decode_exact(case, seed):
    s = _decode_inputs(case, seed)
    old_counts, exact_counts = _page_counts(case)
    outs, lses, old_at, exact_at = [], [], 0, 0
    for b, length in enumerate(_lengths(case)):
        old, exact = old_counts[b], exact_counts[b]
        kv = []
        for name in ("k", "v"):
            ids = s["exact_indices"][exact_at:exact_at + exact].long()
            x = s["exact_" + name][ids].double()
            if old:
                ids = s["old_indices"][old_at:old_at + old].long()
                codes = s[name + "_codes"][ids].double()
                x = torch.cat((codes * s[name + "_scale"][ids].double()[:, None, :, None], x))
            kv.append(x.reshape(-1, HKV, DIM)[:length])
        out, lse = _attend(s["query"][b].double(), *kv)
        if old:
            out = out + s["center"][b].double().repeat_interleave(HQ // HKV, dim=0)
        outs.append(out)
        lses.append(lse)
        old_at, exact_at = old_at + old, exact_at + exact
    return {"out": torch.stack(outs), "lse": torch.stack(lses)}


def _append_exact(case, seed):
    s = _append_inputs(case, seed)
    batch = case["batch"]
    positions = s["positions"].long().expand(batch)
    cos, sin = s["cos"].double()[positions], s["sin"].double()[positions]
    ring_k, ring_v = s["ring_k"].double(), s["ring_v"].double()
    page = torch.arange(batch, device="cuda") * TAIL_PAGES + positions // PAGE % TAIL_PAGES
    ring_k[page, positions % PAGE] = _rotate(s["k"].double(), cos, sin) - s["k_center"].double()
    ring_v[page, positions % PAGE] = s["v"].double() - s["v_center"].double()
    return {"rotated": _rotate(s["q"].double(), cos, sin), "ring_k": ring_k, "ring_v": ring_v,
            "codes": None, "scales": None}


def _populate_exact(case, seed):
    gen = _generator(seed)
    pages, sink = case["pages"], case["sink"]
    gain_k, gain_v = _channel_gain(gen), _channel_gain(gen)
    names = {"key_codes": None, "value_codes": None}
    for name, x in zip(("key", "value"), _prompt_kv(gen, gain_k, gain_v, pages * PAGE)):
        x = x.double()
        center = x.mean(dim=0)
        centered = (x - center).view(pages, PAGE, HKV, DIM)
        scales = (centered.abs().amax(dim=(1, 3)) / 127.0).clamp_min(2.0 ** -20)
        exact = torch.zeros(sink + TAIL_PAGES, PAGE, HKV, DIM, device="cuda", dtype=torch.float64)
        exact[:sink] = centered[:sink]
        for page in range(pages - TAIL_PAGES, pages):
            exact[sink + page % TAIL_PAGES] = centered[page]
        names.update({name + "_center": center[None, None], name + "_scales": scales[None],
                      "exact_" + name: exact[None]})
    return names


def _step_exact(case, seed):
    s = _step_inputs(case, seed)
    c, config, batch = s["cache"], s["weights"].config, case["batch"]
    position, pages = case["context"], _step_pages(case)
    old = pages - TAIL_PAGES
    group = HQ // HKV
    slots = torch.arange(old, pages, device="cuda") % TAIL_PAGES
    cos, sin = s["cos"].double()[position], s["sin"].double()[position]
    hidden = s["weights"].embed[s["token"]].double()
    rings = {"key": [], "value": []}
    for layer, w in enumerate(s["weights"].layers):
        qkv = _linear(_rms(hidden, w["input_norm"], config.rms_eps), w["qkv"])
        q = _rotate(qkv[:, :HQ * DIM].view(batch, HQ, DIM), cos, sin)
        k = _rotate(qkv[:, HQ * DIM:(HQ + HKV) * DIM].view(batch, HKV, DIM), cos, sin)
        v = qkv[:, (HQ + HKV) * DIM:].view(batch, HKV, DIM)
        seen = {}
        for name, row in (("key", k), ("value", v)):
            ring = getattr(c, "exact_" + name)[layer].double().view(batch, TAIL_PAGES, PAGE, HKV, DIM)
            center = getattr(c, name + "_center")[layer].double()
            ring[:, position // PAGE % TAIL_PAGES, position % PAGE] = row - center
            rings[name].append(ring.reshape(-1, PAGE, HKV, DIM))
            seen[name] = ring
        rows = []
        for b in range(batch):
            kv = []
            for name in ("key", "value"):
                at = slice(b * pages, b * pages + old)
                codes = getattr(c, name + "_codes")[layer, at].double()
                codes *= getattr(c, name + "_scales")[layer, at].double()[:, None, :, None]
                kv.append(torch.cat((codes, seen[name][b, slots])).reshape(-1, HKV, DIM)[:position + 1])
            out, _ = _attend(q[b], *kv)
            rows.append(out + c.value_center[layer, b].double().repeat_interleave(group, dim=0))
        hidden = hidden + _linear(torch.stack(rows).view(batch, -1), w["o"])
        x = _rms(hidden, w["post_norm"], config.rms_eps)
        gate, up = _linear(x, w["gate_up"]).split(config.intermediate, dim=-1)
        hidden = hidden + _linear(torch.nn.functional.silu(gate) * up, w["down"])
    logits = _linear(_rms(hidden, s["weights"].norm, config.rms_eps), s["weights"].lm_head)
    return {"logits": logits, "exact_key": torch.stack(rings["key"]),
            "exact_value": torch.stack(rings["value"]), "key_codes": None, "value_codes": None,
            "key_scales": None, "value_scales": None}


def _prefill_exact(case, seed):
    s = _prefill_inputs(case, seed)
    config, tokens = s["weights"].config, case["tokens"]
    group = HQ // HKV
    cos, sin = s["cos"].double(), s["sin"].double()
    hidden = s["weights"].embed[s["tokens"]].double()
    keys, values = [], []
    for w in s["weights"].layers:
        qkv = _linear(_rms(hidden, w["input_norm"], config.rms_eps), w["qkv"])
        q = _rotate(qkv[:, :HQ * DIM].view(tokens, HQ, DIM), cos, sin)
        k = _rotate(qkv[:, HQ * DIM:(HQ + HKV) * DIM].view(tokens, HKV, DIM), cos, sin)
        v = qkv[:, (HQ + HKV) * DIM:].view(tokens, HKV, DIM)
        keys.append(k)
        values.append(v)
        attended = torch.empty(tokens, HQ, DIM, device="cuda", dtype=torch.float64)
        for h in range(HQ):
            for begin in range(0, tokens, 4096):
                end = min(tokens, begin + 4096)
                scores = (q[begin:end, h] @ k[:end, h // group].t()) * SM_SCALE
                rows = torch.arange(begin, end, device="cuda")
                scores.masked_fill_(torch.arange(end, device="cuda")[None, :] > rows[:, None],
                                    float("-inf"))
                attended[begin:end, h] = torch.softmax(scores, dim=-1) @ v[:end, h // group]
        hidden = hidden + _linear(attended.view(tokens, -1), w["o"])
        x = _rms(hidden, w["post_norm"], config.rms_eps)
        gate, up = _linear(x, w["gate_up"]).split(config.intermediate, dim=-1)
        hidden = hidden + _linear(torch.nn.functional.silu(gate) * up, w["down"])
    logits = _linear(_rms(hidden[-1:], s["weights"].norm, config.rms_eps), s["weights"].lm_head)
    return {"logits": logits, "key": torch.stack(keys), "value": torch.stack(values)}


@torch.inference_mode()
def exact(case, seed):
    return {"decode": _decode_exact, "append": _append_exact, "populate": _populate_exact,
            "step": _step_exact, "prefill": _prefill_exact}[case["op"]](case, seed)
