"""Workspace size queries: a buffer sized for the largest shape of a range serves the smaller ones.

CPU: without a device the library assumes 256 CUs, as the MI355X has.
"""
import itertools

import pytest

from unifiedkv_amd import _ext

DECODE = dict(batch=[1, 2, 7, 16, 61, 128, 247, 248, 249, 250, 300, 1000], heads=[1, 8, 28, 32, 64, 96, 128],
              dim=[64, 128, 256], pages=[1, 2, 4, 8, 16, 33, 64, 128, 512, 2048])


@pytest.mark.parametrize("axis", list(DECODE))
def test_decode_size_never_falls_as_the_shape_grows(axis):
    size = _ext.load().ukv_page16_workspace_bytes
    others = [k for k in DECODE if k != axis]
    for rest in itertools.product(*(DECODE[k] for k in others)):
        at = dict(zip(others, rest))
        sizes = [int(size(*({**at, axis: x}[k] for k in DECODE))) for x in DECODE[axis]]
        assert sizes == sorted(sizes), (axis, at, sizes)


def test_decode_size_over_every_batch():
    size = _ext.load().ukv_page16_workspace_bytes
    for heads, dim, pages in [(64, 128, 4), (128, 256, 1), (28, 128, 40), (96, 128, 3)]:
        sizes = [int(size(b, heads, dim, pages)) for b in range(1, 700)]
        assert sizes == sorted(sizes), (heads, dim, pages)


@pytest.mark.parametrize("kv_heads,n_rep", [(8, 4), (2, 3)])
@pytest.mark.parametrize("obs,dim,workgroups", [(16, 64, 512), (32, 64, 512), (64, 64, 512), (128, 64, 256), (64, 128, 256)])
def test_scores_of_many_items_fill_what_a_cu_holds(obs, dim, workgroups, kv_heads, n_rep):
    """The plan of 64 items of 8000 tokens (S key ranges and G unit groups an item), read off the size of its
    scratch: S rows of statistics' partials, one of statistics, G running maxima a key (one sum a block where
    G is 1). A CU holds two workgroups at 64 dims with up to two row tiles a wave, one otherwise."""
    items, heads, seq_len = 64, kv_heads * n_rep, 8000
    size = int(_ext.load().ukv_snapkv_workspace_bytes(items, 1, seq_len, 16, obs, heads, kv_heads, dim, n_rep, 16))
    row = items * heads * obs * 8
    blocks = (seq_len - 16 - obs + 15) // 16
    plans = [s * g for g in range(1, kv_heads * n_rep + 1) for s in range(1, 126)
             if 0 <= size - ((s + 1) * row + items * blocks * (4 if g == 1 else 64 * g) + 4 * items) < 4 * 256]
    assert plans and min(plans) * items == workgroups, plans
