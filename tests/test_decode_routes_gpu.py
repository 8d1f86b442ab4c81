"""Head counts and page sizes at the edges of the decode dispatch, against the CPU oracle.

Up to 16 heads run the few-heads kernel, 17..63 the warp-specialized kernel padded to 64, more than 64 its
groups of 64 in one launch (the last group padded), and any count the general kernel when row offsets do not fit
in 32 bits (of the queries, or of the pool with pages under 32 tokens). Tolerances: bf16 output atol = rtol = 2e-2,
fp32 LSE atol 1e-3 (as everywhere in the decode tests).
"""

from __future__ import annotations

import pytest
import torch

from minisgl_amd.benchmark.inputs import make_decode_case
from minisgl_amd.kernel import lib
from oracle import ref_mla as R

pytestmark = pytest.mark.gpu

DEV = "cuda"
O_TOL = dict(atol=2e-2, rtol=2e-2)
LSE_TOL = dict(atol=1e-3, rtol=0.0)


def _decode(q, kv, pt, lens, ps, num_ctas, spare_slots=0):
    B, H, _ = q.shape
    plan_np, slots = lib.decode_plan(lens, ps, num_ctas)
    ws_o, ws_lse = lib.decode_workspace(slots + spare_slots, H, DEV)
    # one more head than the call's: its rows must stay untouched
    out = torch.full((B, H + 1, 512), 7.0, dtype=torch.bfloat16, device=DEV)
    lse = torch.full((B, H + 1), 7.0, dtype=torch.float32, device=DEV)
    lib.mla_decode(q.to(DEV), kv.to(DEV), pt.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV),
                   torch.from_numpy(plan_np).to(DEV), num_ctas, ws_o, ws_lse, R.DEFAULT_SCALE, out[:, :H], lse[:, :H])
    torch.cuda.synchronize()
    assert torch.all(out[:, H] == 7.0) and torch.all(lse[:, H] == 7.0)
    return out[:, :H].cpu(), lse[:, :H].cpu()


@pytest.mark.parametrize("heads,ps,num_ctas", [
    (1, 64, 300), (16, 1, 7), (16, 128, 400), (5, 8, 2), (17, 64, 64), (33, 1, 64), (47, 32, 300), (63, 4, 5),
    (65, 64, 64), (80, 1, 16), (127, 64, 300), (130, 16, 9),
])
def test_decode_dispatch_edges(heads, ps, num_ctas):
    """Empty requests first, last and in between; pieces shorter than a tile; more ranges than compute units."""
    print(f"[decode edges] heads={heads} ps={ps} ctas={num_ctas}", flush=True)
    lens = [0, 1, 31, 0, 33, 700, 2049, 64, 0]
    case = make_decode_case(len(lens), heads, ps, lens=lens, seed=heads + ps)
    out, lse = _decode(case.q, case.kv_pool, case.page_table, lens, ps, num_ctas)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, lens)
    full = torch.tensor([L > 0 for L in lens])
    torch.testing.assert_close(out[full].float(), o_ref[full], **O_TOL)
    torch.testing.assert_close(lse[full], lse_ref[full], **LSE_TOL)
    assert torch.all(out[~full] == 0) and torch.all(torch.isneginf(lse[~full]))


@pytest.mark.parametrize("heads,ps", [(8, 64), (8, 1), (24, 64), (70, 8)])
def test_decode_growing_logits(heads, ps):
    """Scores that pass the piece's exponent reference by more than 2^64, several times over."""
    case = make_decode_case(2, heads, ps, lens=[900, 2000], seed=29)
    kv = case.kv_pool.float()
    for b, L in enumerate(case.lens):  # grows along each request
        rows = R.token_rows(case.page_table[b], L, ps)
        kv.view(-1, 576)[rows, 512] = torch.linspace(0, 160.0, L)
    case.kv_pool = kv.to(torch.bfloat16)
    case.q[..., 512] = 20.0
    out, lse = _decode(case.q, case.kv_pool, case.page_table, case.lens, ps, 8)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, case.lens)
    torch.testing.assert_close(out.float(), o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)


@pytest.mark.parametrize("heads,L,num_ctas", [(3, 64 * 9, 9), (8, 64 * 33 + 5, 40), (66, 64 * 70, 70), (64, 64 * 200, 200)])
def test_decode_merge_widths_give_the_same_bits(heads, L, num_ctas):
    """One request in many pieces, merged by four waves per head and, with a second request's slots spread
    over a batch of short ones, by one wave: the same partials give the same bits either way."""
    case = make_decode_case(1, heads, 64, lens=[L], seed=heads)
    plan, slots = lib.decode_plan([L], 64, num_ctas)
    assert slots >= num_ctas // 2
    wide = _decode(case.q, case.kv_pool, case.page_table, [L], 64, num_ctas)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, [L])
    torch.testing.assert_close(wide[0].float(), o_ref, **O_TOL)
    torch.testing.assert_close(wide[1], lse_ref, **LSE_TOL)
    # the same partials merged in a batch of `slots` requests (one slot per request on average: one wave)
    ws_o, ws_lse = lib.decode_workspace(slots, heads, DEV)
    out = torch.empty((slots, heads, 512), dtype=torch.bfloat16, device=DEV)
    lse = torch.empty((slots, heads), dtype=torch.float32, device=DEV)
    plan_dev = torch.from_numpy(plan).to(DEV)
    lib.mla_decode(case.q.to(DEV), case.kv_pool.to(DEV), case.page_table.to(DEV),
                   torch.tensor([L], dtype=torch.int32, device=DEV), plan_dev, num_ctas, ws_o, ws_lse, R.DEFAULT_SCALE,
                   out[:1], lse[:1], split_only=True)
    info = plan_dev[num_ctas * 4 :].view(1, 3).expand(slots, 3).contiguous()
    lib.mla_decode_merge(ws_o, ws_lse, info, out, lse)
    torch.cuda.synchronize()
    for b in (0, slots - 1):
        assert torch.equal(out[b].cpu().view(torch.int16), wide[0][0].view(torch.int16))
        assert torch.equal(lse[b].cpu(), wide[1][0])


def test_decode_head_counts_beyond_32_bit_offsets():
    """A page-size-1 pool of more than 4 GiB: every head count takes the general kernel, above 64 heads in
    one launch per group."""
    pages = (1 << 32) // 1152 + 4096
    lens = [300, 77]
    g = torch.Generator().manual_seed(41)
    pool = torch.empty((pages, 1, 576), dtype=torch.bfloat16, device=DEV)
    rows = torch.randn((1000, 1, 576), generator=g).to(torch.bfloat16)
    pool[:500] = rows[:500].to(DEV)
    pool[pages - 500 :] = rows[500:].to(DEV)
    perm = torch.randperm(1000, generator=g)
    small_pt = torch.zeros((2, 300), dtype=torch.int32)
    small_pt[0] = perm[:300].to(torch.int32)
    small_pt[1, :77] = perm[300:377].to(torch.int32)
    pt = torch.where(small_pt < 500, small_pt, small_pt - 1000 + pages)
    for heads in (5, 20, 40, 70):
        q = torch.randn((2, heads, 576), generator=g).to(torch.bfloat16)
        o_ref, lse_ref = R.mla_decode(q, rows, small_pt, lens)
        out, lse = _decode(q, pool, pt, lens, 1, 12)
        torch.testing.assert_close(out.float(), o_ref, **O_TOL)
        torch.testing.assert_close(lse, lse_ref, **LSE_TOL)


@pytest.mark.parametrize("heads", [8, 24, 64, 130])
@pytest.mark.parametrize("ps", [32, 64])
def test_decode_page_table_row_stride_is_not_its_width(heads, ps):
    """A one-row table made by a transpose has strides (1, 1), and rows that overlap have a stride below their
    width: neither bounds the columns. 16 plan ranges: most lie inside one request, its last one among them."""
    print(f"[decode table stride] heads={heads} ps={ps}", flush=True)
    case = make_decode_case(1, heads, ps, lens=[1500], seed=heads + ps)
    pt = case.page_table.view(-1, 1).to(DEV).t()
    assert pt.stride() == (1, 1) and pt.shape[1] > 1
    out, lse = _decode(case.q, case.kv_pool, pt, [1500], ps, 16)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, [1500])
    torch.testing.assert_close(out.float(), o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)
    lens = [1400, 900, 1300]  # row b is the ids from 2b on
    ids = torch.cat([case.page_table[0].to(torch.int32), case.page_table[0, :4].to(torch.int32)])
    pt = ids.to(DEV).as_strided((3, case.page_table.shape[1]), (2, 1))
    q = case.q.expand(3, heads, 576).clone()
    q[1:] = -q[1:]
    out, lse = _decode(q, case.kv_pool, pt, lens, ps, 16)
    o_ref, lse_ref = R.mla_decode(q, case.kv_pool, pt.cpu(), lens)
    torch.testing.assert_close(out.float(), o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)


@pytest.mark.parametrize("heads,num_ctas", [(8, 1), (16, 3), (24, 1), (64, 1)])
def test_decode_tokens_of_infinitely_low_score(heads, num_ctas):
    """Tokens that a query scores -inf (a rope dim of -inf) count for nothing, also where they fill a piece's first
    tile, whose maximum is the exponent reference."""
    lens = [100, 700]
    case = make_decode_case(2, heads, 64, lens=lens, seed=heads)
    kv = case.kv_pool.float()
    for b, L in enumerate(lens):
        kv.view(-1, 576)[R.token_rows(case.page_table[b], L, 64)[:70], 512] = -float("inf")
    case.kv_pool = kv.to(torch.bfloat16)
    case.q[..., 512] = 1.0
    out, lse = _decode(case.q, case.kv_pool, case.page_table, lens, 64, num_ctas)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, lens)
    assert torch.isfinite(o_ref).all()
    torch.testing.assert_close(out.float(), o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)


@pytest.mark.parametrize("heads,ps,stride", [(16, 64, 150_000_000), (20, 64, 120_000_000), (32, 1, 72_000_000),
                                             (70, 64, 72_000_000), (16, 64, 120_000_000), (40, 1, 64_000_000)])
def test_decode_query_rows_beyond_32_bit_offsets(heads, ps, stride):
    """Heads of a query so far apart that a tile of 16 or 32 of its rows spans more than 4 GiB, and (the last two) more
    than 2 GiB, which unsigned offsets hold."""
    print(f"[decode query stride] heads={heads} ps={ps}", flush=True)
    lens = [300]
    case = make_decode_case(1, heads, ps, lens=lens, seed=heads)
    q = torch.empty((heads - 1) * stride + 576, dtype=torch.bfloat16, device=DEV).as_strided(
        (1, heads, 576), (heads * stride, stride, 1))
    q.copy_(case.q)
    out, lse = _decode(q, case.kv_pool, case.page_table, lens, ps, 3)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, lens)
    torch.testing.assert_close(out.float(), o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)


@pytest.mark.parametrize("heads,ps", [(8, 64), (8, 1), (24, 32), (40, 1), (64, 64), (100, 64), (130, 8)])
def test_decode_second_range_of_a_cta(heads, ps):
    """A plan of more non-empty ranges than compute units, padded to 600: a CTA runs one range after another through
    the same LDS ring and tables (the row-offset ring with small pages), and stops at the first padding range."""
    print(f"[decode loop] heads={heads} ps={ps}", flush=True)
    lens = [960 + (37 * i) % 160 for i in range(40)]
    cus = lib.device_cu_count(torch.cuda.current_device())
    plan, _ = lib.decode_plan(lens, ps, 600)
    used = int((plan[: 4 * 600].reshape(600, 4)[:, 0] < len(lens)).sum())
    assert cus < used < 600 and 600 > 2 * cus
    case = make_decode_case(len(lens), heads, ps, lens=lens, seed=heads + ps)
    out, lse = _decode(case.q, case.kv_pool, case.page_table, lens, ps, 600)
    o_ref, lse_ref = R.mla_decode(case.q, case.kv_pool, case.page_table, lens)
    torch.testing.assert_close(out.float(), o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)
