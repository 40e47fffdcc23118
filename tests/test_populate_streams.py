"""Cache population shares nothing between calls but the cache: calls for
different layers or requests may overlap on the GPU, since none of them waits
for it."""

from __future__ import annotations

import pytest
import torch

FIELDS = ("key_codes", "value_codes", "key_scales", "value_scales", "key_center", "value_center",
          "exact_key", "exact_value")


def test_populates_share_no_scratch(monkeypatch):
    """Neither a scratch handed from one call to the next nor one kept on the
    cache (the kernels are replaced: this looks at the host side alone)."""
    from pagegauge_amd import decoder as dec

    scratch = []

    def centers(key, value, key_center, value_center, workspace=None):
        scratch.append(workspace)

    monkeypatch.setattr(dec, "token_major_centers", centers)
    monkeypatch.setattr(dec, "prefill_page_gauge_layout", lambda *args: None)
    cfg = dec.DecoderConfig(layers=2, hidden=512, q_heads=4, kv_heads=1, intermediate=8, vocab=8)
    cache = dec.GaugeCache(cfg, 2, 6, 2, device="cpu")
    kept = set(vars(cache))
    for layer, pages in ((0, 4), (1, 6), (0, 3)):
        key = torch.zeros(pages * 16, 1, 128, dtype=torch.float16)
        cache.populate(layer, layer, key, key)
    given = [w.data_ptr() for w in scratch if w is not None]
    assert len(scratch) == 3 and len(set(given)) == len(given)
    extra = [v for k, v in vars(cache).items() if k not in FIELDS and isinstance(v, torch.Tensor)]
    assert set(vars(cache)) == kept and not extra


@pytest.mark.gpu
def test_populates_on_two_streams_match_one_stream(cuda):
    from pagegauge_amd import decoder as dec

    cfg = dec.DecoderConfig(layers=2, hidden=4096, intermediate=8, vocab=8)
    gen = torch.Generator(device=cuda).manual_seed(21)
    # growing prefixes, so that a scratch that is kept would be replaced too
    prompts = [[(torch.randn(pages * 16, 8, 128, device=cuda, generator=gen) + request).half()
                for _ in range(2)] for request, pages in enumerate((40, 300, 130, 512))]
    serial, overlapped = (dec.GaugeCache(cfg, 4, 512, 16, device=cuda) for _ in range(2))
    for layer in range(2):
        for request, (key, value) in enumerate(prompts):
            serial.populate(layer, request, key, value)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for request, (key, value) in enumerate(prompts):
        for layer, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                overlapped.populate(layer, request, key, value)
    torch.cuda.synchronize()
    for name in FIELDS:
        assert torch.equal(getattr(serial, name), getattr(overlapped, name)), name
