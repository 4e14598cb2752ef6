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
