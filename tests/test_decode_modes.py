"""Page16 decode where a KV head's pages are shared by several waves, and short tables in one kernel.

Few KV heads (1-4) leave waves of a workgroup over, which take every other page of a segment; tables
of at most 32 pages (64 when the (sequence, head) pairs fill half of the device) are attended by one
workgroup per (sequence, KV head) that writes the output itself. Lengths around the waves' page turns
(8 waves x 16 tokens), empty sequences, masked pages and more than 64 sequences, against the fp64
closed form (|err| <= 2e-3 + 1e-2 |ref|) and, for the fused append, against append-then-decode.
"""
import numpy as np
import pytest

from test_decode_step import _fused_vs_unfused
from test_gpu_decode import assert_close, custom_case, decode_gpu, expected_dense, to_f32
from unifiedkv_amd import workloads

pytestmark = pytest.mark.gpu

EDGES = [1, 16, 17, 127, 128, 129, 143, 255, 256, 257, 400, 512]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("Hkv,n_rep,D", [(1, 4, 128), (2, 7, 128), (3, 5, 64), (4, 16, 128), (8, 4, 64), (16, 1, 128)])
@pytest.mark.parametrize("max_blocks", [32, 33, 90])
def test_lengths_around_the_waves_turns(cuda, Hkv, n_rep, D, dtype, max_blocks):
    case = custom_case(Hkv * 10 + n_rep, len(EDGES), Hkv * n_rep, Hkv, D, EDGES, dtype=dtype, max_blocks=max_blocks)
    out = to_f32(decode_gpu(workloads.to_torch(case)))
    assert_close(out, expected_dense(case), f"Hkv={Hkv} n_rep={n_rep} D={D} {dtype} table {max_blocks}")


@pytest.mark.parametrize("Hkv,B,max_blocks", [(1, 70, 20), (2, 130, 64), (4, 66, 100), (8, 65, 1)])
def test_wide_batches_with_empty_sequences_and_masked_pages(cuda, Hkv, B, max_blocks):
    rng = np.random.default_rng(B)
    lens = rng.integers(1, 16 * max_blocks + 1, size=B)
    case = custom_case(B, B, 4 * Hkv, Hkv, 128, lens, max_blocks=max_blocks)
    case["block_table"][rng.random(case["block_table"].shape) < 0.03] = -1
    case["seqlens"][rng.random(B) < 0.2] = 0
    exp = expected_dense(case)
    out = to_f32(decode_gpu(workloads.to_torch(case)))
    assert_close(out, exp, f"Hkv={Hkv} B={B} table {max_blocks}")


def test_long_sequences_over_one_kv_head(cuda):
    """Segments of more than 64 pages per wave: the page-id window is reloaded."""
    case = custom_case(3, 2, 4, 1, 64, [140000, 33], dtype="fp16")
    out = to_f32(decode_gpu(workloads.to_torch(case)))
    assert_close(out, expected_dense(case), "140000 tokens, one KV head")


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("Hq,Hkv,D,max_blocks", [(4, 1, 128, 32), (4, 1, 64, 40), (28, 4, 128, 32), (28, 4, 128, 63),
                                                 (64, 16, 64, 32)])
def test_fused_append(cuda, Hq, Hkv, D, max_blocks, dtype):
    _fused_vs_unfused(cuda, 11, len(EDGES), Hq, Hkv, D, EDGES, dtype, max_blocks=max_blocks)


def test_fused_append_edge_lengths_and_ids(cuda):
    lens = [0, 20, 24 * 16 + 5, 40, 1]
    _fused_vs_unfused(cuda, 6, len(lens), 32, 8, 128, lens, max_blocks=24, bad_tail=3)
