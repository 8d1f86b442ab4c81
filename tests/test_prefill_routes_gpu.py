"""Both CTA shapes of the prefill kernel (128 and 256 query rows) at the edges of their tiles, stages, tables and
of the rule that chooses between them, against the CPU oracle; tolerances as in the other prefill tests
(bf16 output atol = rtol = 2e-2, fp32 LSE atol 1e-3)."""

from __future__ import annotations

import copy

import pytest
import torch

from minisgl_amd.benchmark.inputs import make_decode_case, make_prefill_case
from minisgl_amd.kernel import lib
from oracle import ref_mla as R

pytestmark = pytest.mark.gpu

DEV = "cuda"
O_TOL = dict(atol=2e-2, rtol=2e-2)
LSE_TOL = dict(atol=1e-3, rtol=0.0)


def _run(case):
    T, H, _ = case.q.shape
    out = torch.full((T, H, 128), float("nan"), dtype=torch.bfloat16, device=DEV)
    lse = torch.full((T, H), float("nan"), dtype=torch.float32, device=DEV)
    dev = [t.to(DEV) for t in (case.q, case.k_pool, case.v_pool, case.page_table, case.cu_seqlens_q, case.seq_lens_k)]
    lib.mla_prefill(*dev, R.DEFAULT_SCALE, out, lse)
    torch.cuda.synchronize()
    return out.float().cpu(), lse.cpu()


def _check(case):
    out, lse = _run(case)
    o_ref, lse_ref = R.mla_prefill(case.q, case.k_pool, case.v_pool, case.page_table, case.cu_seqlens_q, case.seq_lens_k)
    torch.testing.assert_close(out, o_ref, **O_TOL)
    torch.testing.assert_close(lse, lse_ref, **LSE_TOL)


def _cta_rows(case):
    """Query rows of a CTA by the launcher's rule."""
    (total, heads, _), batch = case.q.shape, len(case.extends)
    cus = lib.device_cu_count(torch.cuda.current_device())
    rows = -(-total // batch)
    ctas = -(-rows // 256) * batch * heads
    if total % (256 * batch) == 0 and case.page_table.stride(0) * case.page_size >= 2048:
        return 128 if 2 * ctas <= cus else 256
    return 128 if rows <= 640 or ctas <= cus else 256


@pytest.mark.parametrize("heads,ps,extends,prefixes", [
    (3, 64, [1], [0]), (2, 64, [128], [0]), (2, 64, [129], [31]), (5, 128, [127, 1, 130], [1, 1000, 33]),
    (1, 64, [20], [100]),  # a last stage of 24 keys, and waves without rows
    (1, 64, [70], [16500]),  # a second window of stage sources
    (70, 64, [700, 641], [65, 0]),  # 256-row CTAs: over 640 rows a request and more than 256 of them
    (90, 64, [641], [32 * 9 + 5]),  # the first size past the rule's line
    (2, 128, [130], [33000]),  # a third window
])
def test_prefill_cta_shapes(heads, ps, extends, prefixes):
    print(f"[prefill shapes] heads={heads} ps={ps} {extends} {prefixes}", flush=True)
    case = make_prefill_case(heads, ps, extends=extends, prefixes=prefixes, seed=sum(extends))
    assert _cta_rows(case) == (256 if heads >= 70 else 128)
    _check(case)


@pytest.mark.parametrize("cta_rows,heads,extends,prefixes", [
    (128, 90, [640], [293]),  # the last size up to the line in rows
    # whole 256-row blocks: more than half of the compute units busy, half of them, and too few keys
    (256, 70, [256, 256], [1792, 1000]), (128, 64, [256, 256], [1792, 1000]), (128, 70, [256, 256], [1700, 0]),
])
def test_prefill_cta_rule(cta_rows, heads, extends, prefixes):
    print(f"[prefill rule] heads={heads} {extends} {prefixes}", flush=True)
    case = make_prefill_case(heads, 64, extends=extends, prefixes=prefixes, seed=sum(prefixes))
    assert _cta_rows(case) == cta_rows
    _check(case)


def test_prefill_source_windows_of_256_rows():
    """256-row CTAs over more keys than one window of stage sources (1024 stages, 32,768 keys) holds: bit for bit the
    128-row CTAs that a launch of one head takes, and some heads against the oracle."""
    H, E, P = 100, 700, 33500
    case = make_prefill_case(H, 64, extends=[E], prefixes=[P], device=DEV, seed=21)
    assert _cta_rows(case) == 256
    out, lse = _run(case)
    for h in (0, 63, 99):
        head = copy.copy(case)
        head.q, head.k_pool, head.v_pool = (t[..., h:h + 1, :] for t in (case.q, case.k_pool, case.v_pool))
        assert _cta_rows(head) == 128
        o1, l1 = _run(head)
        assert torch.equal(o1, out[:, h:h + 1]) and torch.equal(l1, lse[:, h:h + 1])
        o_ref, lse_ref = R.mla_prefill(head.q.cpu(), head.k_pool.cpu(), head.v_pool.cpu(), case.page_table.cpu(),
                                       case.cu_seqlens_q.cpu(), case.seq_lens_k.cpu())
        torch.testing.assert_close(o1, o_ref, **O_TOL)
        torch.testing.assert_close(l1, lse_ref, **LSE_TOL)


def test_prefill_many_requests_of_mixed_lengths():
    """64 requests (ordered by their keys) and 65 (in batch order), some of one length, one without rows."""
    for n in (64, 65):
        ext = [1 + (7 * i) % 40 for i in range(n)]
        pre = [(i % 5) * 37 for i in range(n)]
        ext[3] = 0
        _check(make_prefill_case(2, 64, extends=ext, prefixes=pre, seed=n))


@pytest.mark.parametrize("heads,extends", [(4, [40, 200]), (260, [300]), (90, [641])])
def test_prefill_after_lds_held_nan(heads, extends):
    """The kernel's first value pass has no stage before it and must not count what the LDS held: a decode over NaN
    rows leaves NaN in every compute unit's LDS, then a prefill over finite inputs runs (90 heads: in 256-row CTAs,
    whose V ring has another last slot)."""
    nan = make_decode_case(8, 64, 64, lens=[4096] * 8, seed=1, device=DEV)
    nan.kv_pool.fill_(float("nan"))
    plan_np, slots = lib.decode_plan(nan.lens, 64, 256)
    ws_o, ws_lse = lib.decode_workspace(slots, 64, DEV)
    out = torch.empty((8, 64, 512), dtype=torch.bfloat16, device=DEV)
    lib.mla_decode(nan.q, nan.kv_pool, nan.page_table, nan.seq_lens, torch.from_numpy(plan_np).to(DEV), 256, ws_o, ws_lse,
                   R.DEFAULT_SCALE, out)
    case = make_prefill_case(heads, 64, extends=extends, prefixes=[0] * len(extends), seed=9)
    assert _cta_rows(case) == (256 if heads == 90 else 128)
    _check(case)
