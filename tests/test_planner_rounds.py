"""Balanced plans that fill their last round of workgroups: where the 64-page
cap or the raggedness of a batch leaves it nearly empty, the planner cuts up
to three half-size items for every two CUs, within a workspace that holds
them, and otherwise keeps the fewest items.  Sizes are around a target of 16
CUs, so that a case stays small."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.helpers import max_abs

CUS = 16
RAGGED = [70, 70, 70, 90, 100, 127, 128, 120, 66]       # 18 items of at most 64 pages
MEDIUM = [40, 40, 40, 40, 30, 30, 20, 20, 20]           # 9 items: over half the CUs


def _plan(pages, kind=torch.float16, **kwargs):
    from pagegauge_amd.decode import plan_work_items

    ptr = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32).tolist()
    return plan_work_items(ptr, [16] * len(pages), kv_data_type=kind, num_cus=CUS, **kwargs)


@pytest.mark.parametrize("kind", [torch.float16, "heterogeneous"])
@pytest.mark.parametrize("pages,least,most", [
    (RAGGED, 19, 24),            # past one round: up to 3/2 of the CUs
    (MEDIUM, 13, 24),            # 9 uncut items are not left at two workgroups each
    ([64] * 16, 16, 16),         # an even round of one item per CU stays
    ([64] * 17, 17, 24),         # one item past it
    ([64] * 24, 24, 24),         # exactly 3/2
    ([64] * 25, 25, 25),         # past 3/2: the uncut items
    ([50] * 8, 8, 8),            # half the CUs: medium
    ([0, 64, 0] + [64] * 16, 17, 24),
])
def test_rounds_are_filled(pages, least, most, kind):
    plan, items, ptr = _plan(pages, kind)
    assert least <= plan.num_items <= most
    rows = items.numpy()
    start = np.concatenate([[0], np.cumsum(pages)])
    for b in range(len(pages)):
        mine = rows[int(ptr[b]):int(ptr[b + 1])]
        assert (mine[:, 4] - mine[:, 3] <= 64).all()
        covered = [p for r in mine for p in range(r[3], r[4])]
        assert covered == list(range(start[b], start[b + 1]))


def test_large_targets_keep_the_items_of_one_request_in_range():
    """A target whose half again would pass 4096 items per request."""
    from pagegauge_amd.decode import plan_work_items

    plan, _, _ = plan_work_items([0, 4 * 3000], [16], kv_data_type=torch.float16, num_cus=3000)
    assert plan.num_items <= 3000


@pytest.mark.gpu
@pytest.mark.parametrize("pages", [RAGGED, MEDIUM])
def test_both_plans_of_a_batch_match_attention(cuda, pages):
    """With room for the fuller plan, with room for the fewest items only, and
    one byte less, which stays refused.  Outputs are compared with softmax
    attention in float64 (2e-3: the decode kernels' bound on this data)."""
    from pagegauge_amd import _capi, decode

    g = torch.Generator(device=cuda).manual_seed(5)
    total, batch = sum(pages), len(pages)
    key = torch.randn(total, 16, 8, 128, device=cuda, generator=g).half()
    value = torch.randn(total, 16, 8, 128, device=cuda, generator=g).half()
    query = torch.randn(batch, 32, 128, device=cuda, generator=g).half()
    order = torch.randperm(total, device=cuda, generator=g).int()
    ptr = torch.tensor(np.concatenate([[0], np.cumsum(pages)]), dtype=torch.int32)
    last = torch.full((batch,), 16, dtype=torch.int32, device=cuda)
    fuller, _, _ = _plan(pages)
    # without the fuller rounds: one item per 64 pages past one round, and
    # 7/16 of the CUs, never fewer than those, in a medium plan
    fewest = sum(-(-n // 64) for n in pages)
    most = max(-(-n // 64) for n in pages)
    lib = _capi.library()
    small = int(lib.pg_decode_workspace_bytes(batch, 32, fewest, most))
    assert small < fuller.workspace_bytes

    outs = []
    for size in (fuller.workspace_bytes, small):
        d = decode.BatchDecodeWithPagedKVCacheWrapper(
            torch.empty(size, device=cuda, dtype=torch.uint8), "NHD")
        d.plan(ptr.to(cuda), order, last, 32, 8, 128, 16, kv_data_type=torch.float16, num_cus=CUS)
        outs.append((d.num_work_items, d.run(query, (key, value)).clone()))
    assert [n for n, _ in outs] == [fuller.num_items, fewest]
    d = decode.BatchDecodeWithPagedKVCacheWrapper(
        torch.empty(small - 1, device=cuda, dtype=torch.uint8), "NHD")
    with pytest.raises(RuntimeError, match=f"need {small} bytes"):
        d.plan(ptr.to(cuda), order, last, 32, 8, 128, 16, kv_data_type=torch.float16, num_cus=CUS)

    for b in range(batch):
        rows = order[int(ptr[b]):int(ptr[b + 1])].long()
        k = key[rows].reshape(-1, 8, 128).double().repeat_interleave(4, dim=1)
        v = value[rows].reshape(-1, 8, 128).double().repeat_interleave(4, dim=1)
        p = torch.softmax((k * query[b].double()).sum(-1) * 128 ** -0.5, dim=0)
        ref = (p[:, :, None] * v).sum(0)
        for _, out in outs:
            assert max_abs(out[b], ref.cpu()) <= 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("kind,old,exact", [
    ("heterogeneous", [70, 70, 90, 100, 127, 60, 50], 4), ("heterogeneous", MEDIUM, 3),
    ("segmented", [120, 120, 60, 40], 16), ("segmented", [50, 64, 30, 20, 44], 8)])
def test_both_plans_of_a_compressed_batch_match_attention(cuda, kind, old, exact):
    """The same over an INT8 history and exact pages, as two segments and as
    one table: the fuller plan and the fewest items (in a workspace of just
    their size) against attention in float64 over the dequantised pages (2e-3
    as above)."""
    import re

    from pagegauge_amd import decode

    g = torch.Generator(device=cuda).manual_seed(6)
    batch, total, tails = len(old), sum(old), exact * len(old)

    def normal(*shape):
        return torch.randn(*shape, device=cuda, generator=g)

    codes = [normal(total, 16, 8, 128).mul(40).round().clamp(-127, 127).to(torch.int8) for _ in range(2)]
    scales = [(normal(total, 8).abs() * 0.01 + 0.02).half() for _ in range(2)]
    pages = [normal(tails, 16, 8, 128).half() for _ in range(2)]
    query, center = normal(batch, 32, 128).half(), (normal(batch, 8, 128) * 0.1).half()
    old_ids = torch.randperm(total, device=cuda, generator=g).int()
    exact_ids = torch.randperm(tails, device=cuda, generator=g).int()
    last = torch.tensor([16 - b % 5 for b in range(batch)], dtype=torch.int32, device=cuda)
    ends = np.concatenate([[0], np.cumsum(old)]).astype(np.int32)
    old_ptr, exact_ptr = torch.tensor(ends), torch.arange(0, tails + 1, exact, dtype=torch.int32)
    full = torch.full((batch,), 16, dtype=torch.int32, device=cuda)
    unified = torch.cat([t for b in range(batch)
                         for t in (old_ids[ends[b]:ends[b + 1]], exact_ids[b * exact:(b + 1) * exact])])
    old_kv_len = torch.tensor(old, dtype=torch.int32, device=cuda) * 16

    def attend(size):
        ws = torch.empty(size, device=cuda, dtype=torch.uint8)
        out = dict(value_center=center, return_lse=True)
        if kind == "segmented":
            d = decode.PageGaugeSegmentedDecode(ws)
            d.plan(old_ptr, old_ids, full, exact_ptr, exact_ids, last, num_cus=CUS)
            result = d.run(query, codes, *scales, pages, **out)
        else:
            d = decode.HeterogeneousDecodeWrapper(ws)
            d.plan(old_ptr + exact_ptr, unified, last, num_cus=CUS, exact_tail_pages_hint=exact)
            result = d.run(query, codes, *scales, *pages, old_kv_len, **out)
        return d.num_work_items, [t.clone() for t in result]

    with pytest.raises(RuntimeError, match="workspace too small") as refused:
        attend(512)
    small = int(re.search(r"need (\d+) bytes", str(refused.value)).group(1))
    (most, fuller), (least, fewest) = attend(1 << 22), attend(small)
    assert least < most <= CUS * 3 // 2
    for b in range(batch):
        rows = old_ids[ends[b]:ends[b + 1]].long()
        tail = exact_ids[b * exact:(b + 1) * exact].long()
        tokens = (exact - 1) * 16 + int(last[b])
        k, v = (torch.cat(((c[rows].double() * s[rows].double()[:, None, :, None]).reshape(-1, 8, 128),
                           p[tail].double().reshape(-1, 8, 128)[:tokens])).repeat_interleave(4, dim=1)
                for c, s, p in zip(codes, scales, pages))
        scores = (k * query[b].double()).sum(-1) * 128 ** -0.5
        p = torch.softmax(scores, dim=0)
        want = (p[:, :, None] * v).sum(0) + center[b].double().repeat_interleave(4, dim=0)
        lse = torch.logsumexp(scores, dim=0) / np.log(2.0)
        for out, got_lse in (fuller, fewest):
            # beyond the output's own FP16 rounding
            excess = (out[b].double() - want).abs() - want.abs() * 2.0 ** -11
            assert float(excess.max()) <= 2e-3 and max_abs(got_lse[b], lse.cpu()) <= 2e-3
