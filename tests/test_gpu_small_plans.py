"""Plans of small inputs, built by one workgroup in one launch: every array of
the CSR plan and the inverse map against the oracle's stable order, around the
sizes where the kernels change (waves, rounds, the two capacities, one and two
sort passes) and just past them, where the general kernels build the same."""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
ITEM = int(re.search(r"#define RELM_MP_ITEM_SIZE (\d+)",
                     (Path(__file__).parent.parent / "include" / "relm_mp.h").read_text()).group(1))


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible")


def _t(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(a).to(DEV)


def _np(t: torch.Tensor) -> np.ndarray:
    return t.cpu().numpy()


def _arr(bp, name: str, n: int) -> np.ndarray:
    return _np(bp._i32(getattr(bp.plan, name), n)) if n else np.zeros(0, np.int32)


@pytest.mark.parametrize("num_keys,num_edges", [
    (1, 1), (1, 16384), (2, 63), (7, 64), (128, 65), (129, 1023), (4096, 1024), (200, 3200), (4096, 4096),
    (4097, 4096), (300, 4097), (16384, 5), (16384, 16384), (16383, 16321), (1000, 12289), (16385, 100),
    (100, 16385),
])
@pytest.mark.parametrize("form", ["none", "identity", "permuted", "skewed"])
def test_small_plans_against_the_oracle(num_keys: int, num_edges: int, form: str) -> None:
    from relmo_amd import capi

    print(f"small plan keys={num_keys} edges={num_edges} {form}", flush=True)
    rng = np.random.default_rng(num_keys * 31 + num_edges)
    if form == "skewed":  # hubs of one and of several chunks
        keys = np.minimum(rng.pareto(0.5, num_edges).astype(np.int64), num_keys - 1)
    else:
        keys = rng.integers(0, num_keys, num_edges)
    rows = num_edges + 3
    if form == "none":
        gathers = None
    elif form == "identity":
        gathers = np.arange(num_edges)
    else:  # the second snapshot tile holds its own edge ids
        gathers = rng.integers(0, rows, num_edges)
        gathers[4096:8192] = np.arange(num_edges)[4096:8192]
    kt, gt = _t(keys), None if gathers is None else _t(gathers)
    msgs = np.arange(num_edges) if gathers is None else gathers

    bp = capi.csr_plan(kt, num_keys, gt, num_edges if gathers is None else rows)
    offsets, perm = oracle.csr_build(keys, num_keys)
    assert np.array_equal(_np(bp.offsets), offsets)
    assert np.array_equal(_np(bp.gather_sorted), msgs[perm])
    deg = np.diff(offsets)
    hub = deg > bp.plan.hub_threshold
    chunks = np.where(hub, -(-deg // bp.plan.chunk_size), 0)
    counts = (deg.max(), hub.sum(), chunks.sum(), (chunks > 1).sum())
    assert (bp.plan.max_degree, bp.plan.num_hubs, bp.plan.num_chunks, bp.plan.num_multi_hubs) == counts
    assert bp.plan.gather_identity == int(np.array_equal(msgs, np.arange(num_edges)))
    hubs = np.flatnonzero(hub)
    assert np.array_equal(_arr(bp, "hub_key", hubs.size), hubs)
    assert np.array_equal(_arr(bp, "hub_chunk_base", hubs.size), (np.cumsum(chunks) - chunks)[hubs])
    assert np.array_equal(_arr(bp, "chunk_hub", int(chunks.sum())), np.repeat(np.arange(hubs.size), chunks[hubs]))
    assert np.array_equal(_arr(bp, "multi_hubs", int((chunks > 1).sum())), np.flatnonzero(chunks[hubs] > 1))
    short = np.where(hub, 0, deg)
    W = np.concatenate([[0], np.cumsum(1 + short)])
    assert bp.plan.num_items == W[-1] // ITEM + 1
    items = np.append(np.searchsorted(W[:-1], np.arange(bp.plan.num_items) * ITEM, side="left"), num_keys)
    assert np.array_equal(_np(bp.item_first), items)
    short_off = W - np.arange(num_keys + 1)
    assert np.array_equal(_np(bp.short_off), short_off)
    assert np.array_equal(_np(bp.item_short), short_off[items])
    assert bp.plan.num_short == int(short.sum())
    assert np.array_equal(_np(bp.short_gather), msgs[perm][~np.repeat(hub, deg)])

    inv = capi.inv_plan(kt, num_keys, gt, rows, snapshot=True)
    want, collisions = oracle.inverse_build(keys, num_keys)
    assert np.array_equal(_np(inv.inv), want)
    assert inv.plan.collisions == collisions

    # the snapshots: the same indices match, one changed index (the last) does not
    for plan in (bp, inv):
        assert capi.plan_match(kt, gt, [plan]) == [True]
        other = keys.copy()
        other[-1] += 1
        assert capi.plan_match(_t(other), gt, [plan]) == [False]

    # bad indices: the smallest bad edge of each array is the one reported
    if num_edges >= 3:
        bad = keys.copy()
        bad[num_edges // 3], bad[-1] = num_keys + 5, -2
        for build in (capi.csr_plan, capi.inv_plan):
            with pytest.raises((RuntimeError, ValueError), match=rf"key index out of bounds: {num_keys + 5} not in"):
                build(_t(bad), num_keys, gt, rows)
        if gathers is not None:
            bad_g = gathers.copy()
            bad_g[num_edges // 2], bad_g[-1] = -1, rows
            for build in (capi.csr_plan, capi.inv_plan):
                with pytest.raises((RuntimeError, ValueError), match="gather index out of bounds: -1 not in"):
                    build(kt, num_keys, _t(bad_g), rows)


def test_small_identity_inverse() -> None:
    from relmo_amd import capi

    for n, keys in ((1, 1), (4096, 4097), (10_000, 16_384)):
        bp = capi.inv_plan(_t(np.arange(n)), keys, None, 0)
        assert not bp.plan.inv and bp.plan.collisions == 0


@pytest.mark.parametrize("wait", [True, False])
@pytest.mark.parametrize("n", [100, 4096, 16384])
def test_inverse_map_is_stored_when_the_build_returns(n: int, wait: bool) -> None:
    """Once the build (or the validation of one that did not wait) has returned, another stream may read the
    map: a copy that waits for nothing else, into memory that still holds the previous map before the build."""

    from relmo_amd import capi

    side = torch.cuda.Stream()
    rng = np.random.default_rng(n)
    for _ in range(20):
        keys = rng.permutation(n)
        kt = _t(keys)
        torch.cuda.synchronize()
        bp = capi.inv_plan(kt, n, None, 0, wait=wait, snapshot=True)
        if not wait:
            capi.validate(bp)
        with torch.cuda.stream(side):
            got = bp.inv.clone()
            snap = bp._i32(bp.plan.snap_keys, n).clone()
        side.synchronize()
        assert np.array_equal(_np(got), np.argsort(keys))
        plain = _arr(bp, "snap_key_plain", -(-n // 4096))
        assert np.array_equal(np.where(np.repeat(plain, 4096)[:n] != 0, np.arange(n), _np(snap)), keys)



@pytest.mark.parametrize("num_keys,num_edges", [(50, 4096), (16384, 16384)])
def test_csr_build_reads_no_index_array_after_it_returns(num_keys: int, num_edges: int) -> None:
    """A build that returns once the indices are validated leaves them to the caller: overwritten on another
    stream that waits for nothing, they change neither the sorted rows nor the snapshot."""

    from relmo_amd import capi

    side = torch.cuda.Stream()
    rng = np.random.default_rng(num_keys)
    for _ in range(20):
        keys, gathers = rng.integers(0, num_keys, num_edges), rng.permutation(num_edges)
        kt, gt = _t(keys), _t(gathers)
        torch.cuda.synchronize()
        bp = capi.csr_plan(kt, num_keys, gt, num_edges, wait_counts=False)
        with torch.cuda.stream(side):
            gt.fill_(-1)
            kt.fill_(-1)
        torch.cuda.synchronize()
        capi.read_counts(bp, kt)
        offsets, perm = oracle.csr_build(keys, num_keys)
        assert np.array_equal(_np(bp.offsets), offsets)
        assert np.array_equal(_np(bp.gather_sorted), gathers[perm])
        short = np.repeat(np.diff(offsets) <= bp.plan.hub_threshold, np.diff(offsets))
        assert np.array_equal(_np(bp.short_gather), gathers[perm][short])
        assert capi.plan_match(_t(keys), _t(gathers), [bp]) == [True]


@pytest.mark.parametrize("num_edges", [16385, 20480, 100_001])
def test_one_key_past_the_small_plans(num_edges: int) -> None:
    """One key and more edges than a small plan takes: a sort by digits of no bits, whose ranks count on through
    the rounds of a wave (they started again at each round: rows never written, and read by the reduction)."""

    from relmo_amd import capi

    print(f"one key, {num_edges} edges", flush=True)
    rng = np.random.default_rng(num_edges)
    kt = torch.zeros(num_edges, dtype=torch.int64, device=DEV)
    for gathers in (None, np.arange(num_edges), rng.permutation(num_edges)):
        bp = capi.csr_plan(kt, 1, None if gathers is None else _t(gathers), num_edges)
        want = np.arange(num_edges) if gathers is None else gathers
        assert np.array_equal(_np(bp.gather_sorted), want)
        assert np.array_equal(_np(bp.offsets), [0, num_edges])
        assert (bp.plan.max_degree, bp.plan.num_hubs) == (num_edges, 1)
    x = torch.randn(num_edges, 32, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    got = capi.plan_segment_reduce(bp, x, 0)
    n = num_edges * torch.finfo(torch.float32).eps
    assert bool(((got.double() - x.double().sum(0)).abs() <= n * x.double().abs().sum(0)).all())


@pytest.mark.parametrize("num_keys,num_edges", [(7616, 16384), (7617, 16384), (16384, 7616), (15360, 4097), (11999, 12001)])
@pytest.mark.parametrize("form", ["permuted", "skewed"])
def test_small_plans_at_the_limit_of_edges_and_keys(num_keys: int, num_edges: int, form: str) -> None:
    """Up to and past the sum of edges and keys that one workgroup's CSR build takes, even numbers of keys per
    thread among them."""

    test_small_plans_against_the_oracle(num_keys, num_edges, form)
