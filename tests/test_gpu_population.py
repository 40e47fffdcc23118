"""The bulk quantizer's two access widths against each other, bit for bit, and
the prefill's layout form against its map form."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int16) if t.dtype == torch.float16 else t


def _source(kind, tokens, heads, pad, device):
    """Token rows heads * 128 + pad elements apart: pad 0 takes the 16-byte
    kernel, pad 2 the 4-byte one."""
    gen = torch.Generator(device=device).manual_seed(tokens + heads)
    x = torch.randn(tokens, heads, 128, device=device, generator=gen)
    if kind == "tiny":                                  # scale floor 2^-20, subnormals
        x = x * 2.0 ** -20
    elif kind == "large":
        x = (x * 3.0e4).clamp(-65504, 65504)
    elif kind == "outliers":
        x[..., ::32] *= 8
        x[16:32] = 0.0                                  # an all-zero page
    elif kind == "nan":                                 # a finite scale: the products' path
        x[3, :, 5], x[21, :, 9] = float("nan"), float("nan")
    elif kind == "not_finite":
        x[3, :, 5], x[20, :, 7], x[20, :, 9] = float("inf"), float("nan"), float("-inf")
    rows = torch.zeros(tokens, heads * 128 + pad, device=device, dtype=torch.float16)
    out = rows[:, :heads * 128].view(tokens, heads, 128)
    out.copy_(x)
    return out


@pytest.mark.parametrize("kind", ["plain", "outliers", "tiny", "large", "nan", "not_finite"])
@pytest.mark.parametrize("pages,heads", [(3, 8), (5, 1), (33, 3)])
def test_prefill_widths_agree(cuda, kind, pages, heads):
    from pagegauge_amd.update import prefill_page_gauge

    print(f"prefill widths {kind} pages={pages} heads={heads}", flush=True)
    centers = [(torch.randn(heads, 128, device=cuda) * 0.25).half() for _ in range(2)]
    exact_map = torch.full((pages,), -1, device=cuda, dtype=torch.int32)
    exact_map[0], exact_map[-1] = 1, 0
    results = []
    for pad in (0, 2):
        k, v = (_source(kind, pages * 16, heads, pad, cuda) for _ in range(2))
        out = [torch.zeros(pages, 16, heads, 128, device=cuda, dtype=torch.int8) for _ in range(2)]
        out += [torch.zeros(pages, heads, device=cuda, dtype=torch.float16) for _ in range(2)]
        rings = [torch.zeros(2, 16, heads, 128, device=cuda, dtype=torch.float16) for _ in range(2)]
        prefill_page_gauge(k, v, *centers, *out, exact_map, *rings)
        results.append(out + rings)
    for wide, narrow in zip(*results):
        assert torch.equal(_bits(wide), _bits(narrow))


@pytest.mark.parametrize("kind", ["outliers", "tiny", "large", "nan", "not_finite"])
def test_half_even_widths_agree(cuda, kind):
    from pagegauge_amd.update import quantize_page_gauge

    x = _source(kind, 96, 8, 0, cuda).view(6, 16, 8, 128)
    shifted = torch.zeros(8 * 128 + 1, device=cuda, dtype=torch.float16)[1:].view(8, 128)
    shifted.copy_((torch.randn(8, 128, device=cuda) * 0.25).half())   # 2-byte aligned: narrow
    narrow, wide = quantize_page_gauge(x, shifted), quantize_page_gauge(x, shifted.clone())
    assert torch.equal(wide[0], narrow[0]) and torch.equal(_bits(wide[2]), _bits(narrow[2]))


@pytest.mark.parametrize("sink,suffix,initial,tail,pages,request_index", [
    (0, 0, None, 16, 17, 0), (2, 0, None, 16, 40, 1), (1, 3, 12, 4, 12, 0), (0, 5, 20, 4, 33, 2),
    (1, 6, 20, 4, 21, 1)])
def test_layout_form_is_the_map_form(cuda, sink, suffix, initial, tail, pages, request_index):
    from pagegauge_amd import page_table as pt
    from pagegauge_amd.update import prefill_page_gauge, prefill_page_gauge_layout

    layout = pt.ExactPageLayout.checked(sink, suffix, initial, tail)
    k, v = (_source("outliers", pages * 16, 2, 0, cuda) for _ in range(2))
    centers = [(torch.randn(2, 128, device=cuda) * 0.25).half() for _ in range(2)]
    exact_map = torch.full((pages,), -1, dtype=torch.int32)
    partition = pt.page_gauge_logical_partition(pages, tail, sink, 16, suffix, initial)
    for page in partition["exact_logical_pages"]:
        exact_map[page] = pt.exact_physical_page_index(request_index, page, tail, sink, suffix, initial)
    results = []
    for form in ("map", "layout"):
        out = [torch.zeros(pages, 16, 2, 128, device=cuda, dtype=torch.int8) for _ in range(2)]
        out += [torch.zeros(pages, 2, device=cuda, dtype=torch.float16) for _ in range(2)]
        rings = [torch.zeros(3 * layout.storage, 16, 2, 128, device=cuda, dtype=torch.float16)
                 for _ in range(2)]
        if form == "map":
            prefill_page_gauge(k, v, *centers, *out, exact_map.to(cuda), *rings)
        else:
            prefill_page_gauge_layout(k, v, *centers, *out, *rings, request_index, layout)
        results.append(out + rings)
    for a, b in zip(*results):
        assert torch.equal(_bits(a), _bits(b))
    with pytest.raises(RuntimeError, match="past the exact pages"):
        prefill_page_gauge_layout(k, v, *centers, *results[0][:4], *results[0][4:], 3, layout)


# chunks of 64 tokens; 16 rows of the second launch; column groups that do not
# divide the block; 4-byte rows
@pytest.mark.parametrize("tokens,heads,pad", [(1, 1, 0), (64, 8, 0), (1025, 3, 0), (1088, 9, 0),
                                              (65, 17, 0), (130, 3, 2), (2049, 5, 2)])
@pytest.mark.parametrize("kind", ["plain", "tiny", "large"])
def test_centers_are_the_exact_mean(cuda, tokens, heads, pad, kind):
    from oracle import pg_oracle as oracle
    from pagegauge_amd.update import token_major_centers

    print(f"centers {kind} tokens={tokens} heads={heads} pad={pad}", flush=True)
    k, v = _source(kind, tokens, heads, pad, cuda), _source(kind, tokens, heads, pad, cuda).neg()
    if pad:
        v = _source(kind, tokens, heads, pad, cuda)
    for got, x in zip(token_major_centers(k, v), (k, v)):
        want = torch.from_numpy(oracle.exact_center(x.cpu().numpy()[:, None]))
        assert torch.equal(_bits(got.cpu()), _bits(want))


def test_centers_of_not_finite_values_do_not_depend_on_the_width(cuda):
    from pagegauge_amd.update import token_major_centers

    results = [token_major_centers(x, x)[0] for x in
               (_source("not_finite", 300, 2, pad, cuda) for pad in (0, 2))]
    assert torch.equal(_bits(results[0]), _bits(results[1]))
