"""How many shares a decode call cuts its pages into, seen from the partials it leaves in its workspace.

The host knows a batch's lengths only as the table's width, so the cut is bounded there and decided on
the device: a sequence much longer than the others, in a table wide enough for it, is not cut finer than
the merge of its partials pays for, and an even batch keeps its cut. Outputs against the fp64 closed form.
"""
import numpy as np
import pytest

from test_gpu_decode import assert_close, custom_case, expected_dense, to_f32
from test_zz_no_alloc import _call
from unifiedkv_amd import _ext, workloads

pytestmark = pytest.mark.gpu


def _slots_written(case, cuda):
    """(partial slots the call wrote, its output): slots are [H_q][D] fp32 rows at the workspace's start."""
    import torch

    lib, tc = _ext.load(), workloads.to_torch(case, cuda)
    B, Hq, D = (int(x) for x in tc["q"].shape)
    size = int(lib.ukv_page16_workspace_bytes(B, Hq, D, int(tc["block_table"].shape[1])))
    ws = torch.full((size,), 0xFF, dtype=torch.uint8, device=cuda)  # NaN in every slot
    out = torch.empty_like(tc["q"])
    assert _call(lib, tc, out, ws) == _ext.UKV_OK
    slots = size // (Hq * (4 * D + 8))
    rows = ws[:slots * Hq * D * 4].view(torch.int32).view(slots, -1)
    return int((rows != -1).any(dim=1).sum()), to_f32(out)


# (q heads, KV heads, lengths, table, most slots, fewest): a share of n pages for a longest sequence of n * n * 16
# pages, at most one more slot per sequence.
CUTS = [
    (32, 8, [4096, 17, 17, 17], 256, 76, 32), (4, 1, [4096, 17, 17, 17], 256, 76, 32),
    (32, 8, [1040] + [17] * 15, 65, 80, 40), (32, 8, [4096] + [17] * 69, 256, 176, 96),
    (32, 8, [100, 200, 250, 300], 256, 60, 48), (32, 8, [2048] * 4, 128, 132, 128),
    (16, 16, [4090] * 4, 256, 132, 128),  # two workgroups a share: one round of them
]


@pytest.mark.parametrize("Hq,Hkv,lens,max_blocks,most,fewest", CUTS)
def test_shares_follow_the_lengths_and_not_the_table(cuda, Hq, Hkv, lens, max_blocks, most, fewest):
    case = custom_case(len(lens) + Hkv, len(lens), Hq, Hkv, 128, lens, max_blocks=max_blocks)
    slots, out = _slots_written(case, cuda)
    assert_close(out, expected_dense(case), f"lens {lens[:4]}.. table {max_blocks}")
    assert fewest <= slots <= most, slots


@pytest.mark.parametrize("lens", [[16 * 56], [16 * 57], [7 * 16, 40 * 16 + 1], [0, 0, 16 * 36], [0, 0, 0], [1] * 64 + [500],
                                  [0] * 66 + [16 * 80, 3]])
@pytest.mark.parametrize("Hkv", [1, 8, 16])
def test_cuts_around_the_rule_s_steps(cuda, Hkv, lens):
    """Longest sequences at the steps of pages per share, empty batches, and batches past one wave's lanes."""
    case = custom_case(len(lens), len(lens), 2 * Hkv, Hkv, 64, lens, max_blocks=90)
    slots, out = _slots_written(case, cuda)
    assert_close(out, expected_dense(case), f"lens {lens[-3:]} Hkv={Hkv}")


@pytest.mark.parametrize("B,Hkv,n_rep,D,max_blocks,direct", [
    (64, 8, 4, 128, 64, False), (64, 8, 4, 128, 33, False), (64, 8, 4, 128, 32, True),  # 512 pairs on 256 CUs
    (32, 8, 4, 128, 64, True), (16, 8, 4, 128, 65, False), (15, 8, 4, 128, 33, False),
    (64, 16, 1, 128, 16, False), (64, 16, 1, 128, 8, True), (32, 16, 1, 128, 24, False), (128, 8, 2, 128, 32, False),
    (64, 16, 1, 64, 32, False), (64, 8, 1, 64, 48, False), (256, 8, 1, 64, 32, True),
])
def test_short_tables_leave_what_does_not_fit_at_once_to_the_split(cuda, B, Hkv, n_rep, D, max_blocks, direct):
    """The one-kernel form of short tables writes no partials. One long sequence among short ones."""
    case = custom_case(B + D, B, Hkv * n_rep, Hkv, D, [17] * (B - 1) + [16 * max_blocks], max_blocks=max_blocks)
    slots, out = _slots_written(case, cuda)
    assert_close(out, expected_dense(case), f"B={B} Hkv={Hkv} n_rep={n_rep} D={D} table {max_blocks}")
    assert (slots == 0) == direct, slots
