"""Row widths that are no multiple of 16 bytes, through the public ops: rows
whose last lane shares columns with the one before it (the CSR reductions) and
outputs written in 8- or 4-byte units across row seams (the inverse-plan
gathers and the logsumexp backward), against torch in float64."""

from __future__ import annotations

import ctypes
import math
import os

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible")
    os.environ["RELM_MP_FALLBACK"] = "error"
    from relmo_amd import mp

    assert mp.available()


def _layout(name: str, edges: int, g: torch.Generator):
    """(flat_src, message rows)."""

    if name == "plain":
        return torch.arange(edges, device=DEV), edges
    if name == "slots":  # as many rows as edges, grouped by argument position
        half = edges // 2
        a = torch.arange(half, device=DEV)
        return torch.cat([2 * a, 2 * a + 1, torch.arange(2 * half, edges, device=DEV)]), edges
    rows = edges + edges // 3 + 2  # rows that no edge reads, the last ones among them
    return torch.randperm(rows - 1, device=DEV, generator=g)[:edges], rows


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("emb", [3, 5, 7, 17, 30, 33, 63, 255, 257, 4095, 4097])
@pytest.mark.parametrize("edges,keys", [(1, 1), (3, 2), (501, 77)])
def test_row_widths(dtype, emb: int, edges: int, keys: int) -> None:
    from relmo_amd import mp

    g = torch.Generator(device=DEV).manual_seed(emb * 1000 + edges)
    eps = torch.finfo(dtype).eps
    dst = torch.randint(0, keys, (edges,), device=DEV, generator=g)
    grad = torch.randn(keys, emb, device=DEV, dtype=dtype, generator=g)
    for layout in ("plain", "slots", "gaps"):
        flat, rows = _layout(layout, edges, g)
        rel = torch.randn(rows, emb, device=DEV, dtype=dtype, generator=g).requires_grad_(True)
        msgs = rel.detach().double()[flat]
        at = dst.unsqueeze(1).expand_as(msgs)
        # sum: n additions of terms up to |x| round by at most n * eps * sum |x|
        total = torch.zeros(keys, emb, device=DEV, dtype=torch.float64).index_add_(0, dst, msgs)
        size = torch.zeros_like(total).index_add_(0, dst, msgs.abs())
        out = mp.fanin_reduce(rel, flat, dst, keys, mp.MODE_SUM)
        n = int(torch.bincount(dst).max())
        assert bool(((out.double() - total).abs() <= n * eps * size).all()), layout
        (got,) = torch.autograd.grad(out, rel, grad)
        want = torch.zeros(rows, emb, device=DEV, dtype=dtype).index_copy_(0, flat, grad[dst])
        assert torch.equal(got, want), layout
        # logsumexp: exp and log on the hardware units, some ulps of |x| ~ 5 each
        out = mp.fanin_reduce(rel, flat, dst, keys, mp.MODE_LOGSUMEXP)
        top = torch.full_like(total, -math.inf).scatter_reduce(0, at, msgs, "amax")
        lse = torch.zeros_like(total).index_add_(0, dst, (msgs - top[dst]).exp()).log() + top
        some = torch.bincount(dst, minlength=keys) > 0
        assert bool((out[~some] == -math.inf).all()), layout
        torch.testing.assert_close(out.double()[some], lse[some], rtol=64 * eps, atol=64 * eps)
        (got,) = torch.autograd.grad(out, rel, grad)
        weight = torch.zeros(rows, emb, device=DEV, dtype=torch.float64).index_copy_(
            0, flat, grad.double()[dst] * (msgs - lse[dst]).exp())
        torch.testing.assert_close(got.double(), weight, rtol=64 * eps, atol=64 * eps)
        # fanout: copies, rows without an edge stay zero
        x = grad
        out = mp.fanout_scatter(x, dst, flat, rows)
        assert torch.equal(out, want), layout
        # LGAN step: a sum with a residual row in the epilogue
        step = mp._lgan_relation_graph_step(x, dst, dst, dst, dst, dst, dst, entity_dim_size=keys, mode="mean")
        pair = x.double() + x.double() * some.unsqueeze(1)
        torch.testing.assert_close(step[0].double(), pair, rtol=4 * eps * n, atol=4 * eps * n)


def test_rows_scale_in_place_at_odd_width() -> None:
    """relm_mp_rows_scale with out equal to base: every column is read before it is written."""

    from relmo_amd import capi

    g = torch.Generator(device=DEV).manual_seed(1)
    for emb in (5, 33, 301):
        x = torch.randn(200, emb, device=DEV, generator=g)
        base = torch.randn(200, emb, device=DEV, generator=g)
        want = base + x
        out = base.clone()
        capi.check(capi.lib().relm_mp_rows_scale(0, capi._ptr(x), None, capi.DIV_NONE, None, None, capi._ptr(out),
                                                 200, emb, capi._ptr(out), capi._stream(x)))
        assert torch.equal(out, want)


@pytest.mark.parametrize("dtype,widths", [(torch.float32, (8, 33, 258, 515, 16387)), (torch.float64, (33, 131, 259))])
def test_logsumexp_backward_in_place(dtype, widths) -> None:
    """grad_rel over rel_flat, rows of several column slices among them: the bits of a call with a buffer of its
    own, by the CSR plan of a flat_src that repeats (without hubs) and by the inverse plan of one that does not."""

    from relmo_amd import capi

    g = torch.Generator(device=DEV).manual_seed(3)
    rows, keys = 900, 40
    for emb in widths:
        rel = torch.randn(rows, emb, device=DEV, dtype=dtype, generator=g)
        grad, out = (torch.randn(keys, emb, device=DEV, dtype=dtype, generator=g) for _ in range(2))
        for repeats in (True, False):
            flat = torch.randint(0, rows, (4000,), device=DEV, generator=g) if repeats else torch.randperm(rows, device=DEV, generator=g)
            dst = torch.randint(0, keys, (flat.numel(),), device=DEV, generator=g)
            bp = capi.csr_plan(flat, rows, dst, keys) if repeats else capi.inv_plan(flat, rows, dst, keys)
            want = capi.plan_logsumexp_backward(bp, grad, out, rel, None if repeats else dst)
            over = rel.clone()
            n = capi.lib().relm_mp_plan_compute_scratch_bytes(ctypes.byref(bp.plan), emb, capi._dtype(rel), 1)
            ws = torch.empty(max(n, 1), dtype=torch.uint8, device=DEV)
            capi.check(capi.lib().relm_mp_plan_logsumexp_backward(
                capi._dtype(rel), ctypes.byref(bp.plan), None if repeats else capi._ptr(dst), capi._ptr(grad), capi._ptr(out),
                capi._ptr(over), emb, capi._ptr(over), capi._ptr(ws), ws.numel(), capi._stream(rel)))
            assert torch.equal(over, want), (emb, repeats)


def _bounded(got, want, bound, what) -> None:
    bad = ~((got.double() - want).abs() <= bound)  # a NaN is not below any bound
    assert not bool(bad.any()), (what, int(bad.sum()), float((got.double() - want).abs().max()))


@pytest.mark.parametrize("dtype,emb", [
    *((torch.float32, d) for d in (3, 7, 15, 17, 31, 33, 38, 41, 47, 49, 63, 64, 65, 66, 94, 127, 128, 129, 130, 254, 257, 258, 386, 515)),
    *((torch.float64, d) for d in (3, 5, 19, 21, 32, 33, 63, 65, 127, 129, 191, 193, 259)),
])
@pytest.mark.parametrize("offset", [0, 1])  # tables that start on 16 bytes, and one element behind
def test_csr_reductions_at_every_lane_width(dtype, emb: int, offset: int) -> None:
    """Every reduction over CSR plans at the widths where its lanes change, short segments, hubs of one chunk and of
    several among the keys: against float64, n additions bounded by n * eps * sum |term| on either side."""

    from relmo_amd import capi

    print(f"{dtype} emb={emb} offset={offset}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(emb)
    eps = torch.finfo(dtype).eps
    rows, keys = 700, 90

    def randn(n):
        flat = torch.randn(n * emb + 1, device=DEV, dtype=dtype, generator=g)
        return flat[offset:offset + n * emb].view(n, emb)

    dst = torch.cat([torch.full((5000,), 3, device=DEV), torch.full((2048,), 5, device=DEV), torch.full((65,), 89, device=DEV),
                     torch.randint(6, 88, (2500,), device=DEV, generator=g)])
    dst = dst[torch.randperm(dst.numel(), device=DEV, generator=g)]
    src = torch.randint(0, rows, (dst.numel(),), device=DEV, generator=g)
    x, base, other = randn(rows), randn(keys), randn(keys)
    count = torch.bincount(dst, minlength=keys).double().unsqueeze(1)
    steps = 2 * (count + 64) * eps  # roundings on the path of a term, both sides; 64 for exp, log and the divisions

    def add(terms, index=dst, n=keys):
        return torch.zeros(n, emb, device=DEV, dtype=torch.float64).index_add_(0, index, terms)

    bp = capi.csr_plan(dst, keys, src, rows)
    msgs = x.double()[src]
    total, size = add(msgs), add(msgs.abs())
    _bounded(capi.plan_segment_reduce(bp, x, 0), total, steps * size, "sum")
    mean = capi.plan_segment_sum_scaled(bp, x, capi.DIV_SEGMENT, base=base)
    _bounded(mean, base.double() + total / count.clamp(min=1), steps * (size / count.clamp(min=1) + base.abs()), "mean")
    by_row = capi.csr_plan(src, rows, dst, keys)
    share = msgs / torch.bincount(src, minlength=rows).double().clamp(min=1)[src].unsqueeze(1)
    _bounded(capi.plan_segment_sum_msgdiv(bp, x, by_row, base=base), base.double() + add(share),
             steps * (add(share.abs()) + base.abs()), "divided sum")
    top = torch.full_like(total, -math.inf).scatter_reduce(0, dst.unsqueeze(1).expand_as(msgs), msgs, "amax")
    some = count.squeeze(1) > 0
    lse = (add((msgs - top[dst]).exp()).log() + top)[some]
    got = capi.plan_segment_reduce(bp, x, 1)
    assert bool((got[~some] == -math.inf).all())
    _bounded(got[some], lse, steps[some] * (1 + lse.abs()), "logsumexp")
    # its backward, keyed by the rows a hub of which is gathered: the rows and keys trade places
    weight = other.double()[dst] * (msgs - base.double()[dst]).exp()
    n = 2 * (torch.bincount(src, minlength=rows).double().unsqueeze(1) + 64) * eps
    _bounded(capi.plan_logsumexp_backward(by_row, other, base, x), add(weight, src, rows), n * add(weight.abs(), src, rows), "backward")
    xr, outr, gr = randn(keys), randn(rows), randn(rows)
    weight = gr.double()[src] * (xr.double()[dst] - outr.double()[src]).exp()
    _bounded(capi.plan_logsumexp_backward(bp, gr, outr, xr), add(weight), steps * add(weight.abs()), "backward with hubs")
    # argument slots: two of a line of 2 * emb + 3 columns
    line = randn(rows // 2 * 3).reshape(-1)[: rows // 2 * (2 * emb + 3)].view(rows // 2, 2 * emb + 3)
    slots = line[:, 3:].reshape(rows, emb).double()[src]
    _bounded(capi.plan_segment_sum_grouped(bp, line, 3, 2, emb), add(slots), steps * add(slots.abs()), "slots")


@pytest.mark.parametrize("emb", [2, 5, 30, 33, 62, 301])
def test_rows_scale_over_its_input(emb: int) -> None:
    """relm_mp_rows_scale with out equal to in."""

    from relmo_amd import capi

    g = torch.Generator(device=DEV).manual_seed(emb)
    x, base = (torch.randn(300, emb, device=DEV, generator=g) for _ in range(2))
    div = torch.randint(1, 5, (300,), device=DEV, generator=g)
    want = capi.rows_scale(x, 300, emb, x, div_kind=capi.DIV_VALUES, div_values=div, base=base)
    assert torch.equal(want, base + x / div.float().unsqueeze(1))
    over = x.clone()
    capi.check(capi.lib().relm_mp_rows_scale(0, capi._ptr(over), None, capi.DIV_VALUES, None, capi._ptr(div), capi._ptr(base),
                                             300, emb, capi._ptr(over), capi._stream(x)))
    assert torch.equal(over, want)
