"""Retained pages and compaction sources built on the device: against the torch expressions they stand for,
over more sequences than one launch takes, row strides, index types and out-of-range entries (GPU)."""
import numpy as np
import pytest
import torch

from unifiedkv_amd import compaction
from unifiedkv_amd.pool import PagedKVPool

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,sink,obs", [(0, 0, 0), (0, 32, 16), (1, 0, 64), (255, 16, 16), (300, 64, 128)])
def test_retained_pages(cuda, k, sink, obs):
    L = 16 * 400 + sink + obs
    g = torch.Generator(device=cuda).manual_seed(k)
    wide = torch.randint(0, 400, (5, k + 3), generator=g, device=cuda, dtype=torch.int32)
    for sel in (wide[:, :k].contiguous(), wide[:, 1:k + 1]):  # rows of a wider tensor too
        got = compaction.retained_pages(L, sel, sink_len=sink, obs_len=obs)
        want = compaction.retained_pages(L, sel.cpu(), sink_len=sink, obs_len=obs)
        assert got.dtype == want.dtype and torch.equal(got.cpu(), want)
        assert torch.equal(compaction.retained_pages(L, sel.long(), sink_len=sink, obs_len=obs).cpu().int(), want)
    if k:
        for value in (-1, 400, 2 ** 31 - 1):
            bad = wide[:, :k].clone()
            bad[3, k - 1] = value
            with pytest.raises(ValueError, match=r"outside \[0, 400\)"):
                compaction.retained_pages(L, bad, sink_len=sink, obs_len=obs)


def test_retained_pages_with_nothing_selected_can_be_captured(cuda):
    sel = torch.empty((3, 0), dtype=torch.int32, device=cuda)
    want = compaction.retained_pages(16 * 8, sel, sink_len=32, obs_len=16)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = compaction.retained_pages(16 * 8, sel, sink_len=32, obs_len=16)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert got.tolist() == want.tolist() == [[0, 1, 7]] * 3


def test_retained_pages_of_more_rows_than_a_grid_takes(cuda):
    sel = torch.arange(65600, dtype=torch.int32, device=cuda).remainder_(5).unsqueeze(1)
    got = compaction.retained_pages(16 * 8, sel, sink_len=32, obs_len=16)
    assert torch.equal(got[:, 1:3].cpu(), torch.stack([torch.ones(65600, dtype=torch.int32), sel[:, 0].cpu() + 2], 1))


def _pool(cuda, layers, n):
    pool = PagedKVPool(16, layers, 2, 64, torch.float16, num_blocks=n, device=cuda)
    g = torch.Generator(device=cuda).manual_seed(0)
    pool.k_cache.normal_(generator=g)
    pool.v_cache.normal_(generator=g)
    return pool


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("free_sources", [False, True])
def test_compact_gathers_every_sequence(cuda, dtype, free_sources):
    rng = np.random.default_rng(3)
    layers, seqs = 3, 70  # two launches of sources
    pool = _pool(cuda, layers, 70 * 6 + 70 * 4)
    order = rng.permutation(pool.allocate_blocks(70 * 6))
    lists = [[int(x) for x in order[6 * s:6 * s + 6]] for s in range(seqs)]
    keeps = []
    for s in range(seqs):
        n = int(rng.integers(0, 5))
        keep = torch.from_numpy(rng.integers(0, 6, (layers, n))).to(cuda, dtype)
        keeps.append(keep[:1].expand(layers, -1) if s % 7 == 0 else keep)
    k0, v0 = pool.k_cache.clone(), pool.v_cache.clone()
    res = compaction.compact(pool, lists, keeps, [16] * seqs, free_sources=free_sources)
    # (with freed sources a later sequence's pages may be an earlier one's old ones, read before)
    seen = set()
    for s in reversed(range(seqs)):
        ids = res.page_lists[s]
        assert len(ids) == keeps[s].shape[1]
        for l in range(layers):
            for j, d in enumerate(ids):
                if (l, d) in seen:
                    continue
                seen.add((l, d))
                p = lists[s][int(keeps[s][l, j])]
                assert torch.equal(pool.k_cache[l, d], k0[l, p]) and torch.equal(pool.v_cache[l, d], v0[l, p])


def test_compact_refuses_bad_indices_and_pages_before_taking_any(cuda):
    pool = _pool(cuda, 2, 20)
    ids = pool.allocate_blocks(8)
    free = pool.free_blocks
    good = torch.zeros((2, 2), dtype=torch.int32, device=cuda)
    for value in (-1, 4, 2 ** 32):
        bad = torch.zeros((2, 2), dtype=torch.int64, device=cuda)
        bad[1, 1] = value
        for b in (bad, bad.int()) if value < 2 ** 31 else (bad,):
            with pytest.raises(ValueError, match="sequence 1"):
                compaction.compact(pool, [ids[:4], ids[4:]], [good, b], [32, 32])
    for page in (-1, 20, 2 ** 40):
        with pytest.raises(ValueError, match="outside the pool"):
            compaction.compact(pool, [ids[:4], ids[4:7] + [page]], [good, good], [32, 32])
    assert pool.free_blocks == free
