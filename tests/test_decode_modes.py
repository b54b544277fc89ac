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
    """A long and a short sequence over one KV head, a few pages to each wave of a share."""
    case = custom_case(3, 2, 4, 1, 64, [140000, 33], dtype="fp16")
    out = to_f32(decode_gpu(workloads.to_torch(case)))
    assert_close(out, expected_dense(case), "140000 tokens, one KV head")


@pytest.mark.parametrize("Hkv,subs", [(1, 8), (2, 4), (3, 2), (4, 2), (5, 1)])
def test_page_id_window_is_reloaded(cuda, Hkv, subs):
    """More than 64 pages per wave, whose page ids come in windows of 64 (64 * subs pages of a share): one
    sequence of 2.6 million tokens at one KV head, its table naming a small pool's pages many times over. Pages of
    the first windows hold other values than the later ones, so that a window read from the wrong place
    shows. The closed form is the softmax over the pool's tokens, each weighed by how often its page is named."""
    import torch

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    share, D, n_rep, pool = 80 * subs, 64, 2, 64  # pages of a share, one share per CU
    P = share * cus
    assert share / subs > 64
    case = custom_case(Hkv, 1, n_rep * Hkv, Hkv, D, [16 * pool], dtype="fp16", N=pool)
    rng = np.random.default_rng(Hkv)
    first = np.arange(P) % share < 64 * subs
    table = np.where(first, rng.integers(0, pool // 2, P), rng.integers(pool // 2, pool, P)).astype(np.int32)
    case["v_cache"][pool // 2:] = workloads._round_bits(
        rng.standard_normal(case["v_cache"][pool // 2:].shape, dtype=np.float32) + 8.0, "fp16")
    case["block_table"], case["seqlens"] = table[None], np.array([16 * P], np.int32)
    out = to_f32(decode_gpu(workloads.to_torch(case)))
    q, k, v = (case[x].view(np.float16).astype(np.float64) for x in ("q", "k_cache", "v_cache"))
    times = np.repeat(np.bincount(table, minlength=pool), 16)
    want = np.zeros(q.shape)
    for h in range(n_rep * Hkv):
        kh, vh = k[:, :, h // n_rep].reshape(-1, D), v[:, :, h // n_rep].reshape(-1, D)
        s = kh @ q[0, h] * case["scale"]
        w = times * np.exp(s - s.max())
        want[0, h] = w @ vh / w.sum()
    assert_close(out, want, f"{P} pages, Hkv={Hkv}")


def test_decode_batch_reaches_the_one_kernel_form(cuda):
    """DecodeBatch's tables are 64 pages wide at least: from 128 (sequence, KV head) pairs on, steps of short
    sequences run in one kernel (the workspace stays as it was). A step's fused attention against the
    append followed by a plain decode of the same pool."""
    import torch

    from unifiedkv_amd import page16_native, page_ops
    from unifiedkv_amd.decode_step import DecodeBatch
    from unifiedkv_amd.pool import PagedKVPool

    Hkv, n_rep, D = 8, 4, 128
    lens = [1, 15, 16, 17, 127, 128, 300, 511, 512, 513, 700, 900, 1000, 1006, 31, 64]
    B = len(lens)
    pages = [-(-n // 16) for n in lens]
    pool = PagedKVPool(16, 1, Hkv, D, torch.bfloat16, num_blocks=sum(pages) + B, device=cuda)
    gen = torch.Generator(device=cuda).manual_seed(5)
    rand = lambda *shape: torch.randn(shape, generator=gen, device=cuda).to(torch.bfloat16)  # noqa: E731
    pool.k_cache.copy_(rand(*pool.k_cache.shape))
    pool.v_cache.copy_(rand(*pool.v_cache.shape))
    batch = DecodeBatch(pool, [pool.allocate_blocks(n) for n in pages], lens, fused_append=True)
    assert batch.block_table.shape[1] == 64 and B * Hkv == 128
    ws = page16_native._workspace(B, n_rep * Hkv, D, 64, cuda, page16_native._current_stream(cuda))
    for _ in range(3):  # (the first takes new pages)
        batch.begin_step()
        q, k, v = rand(B, n_rep * Hkv, D), rand(B, Hkv, D), rand(B, Hkv, D)
        kc, vc = pool.k_cache[0].clone(), pool.v_cache[0].clone()
        ws.fill_(0xFF)
        out = batch.attention(0, q, k, v, softmax_scale=D ** -0.5, n_rep=n_rep)
        assert int((ws != 0xFF).sum()) == 0
        page_ops.kv_append(kc, vc, batch.block_table, batch.cache_seqlens, k, v, return_new_lens=False)
        want = page16_native.page16_decode_attention(q, kc, vc, batch.block_table, batch.attn_lens,
                                                     softmax_scale=D ** -0.5, n_rep=n_rep)
        assert torch.equal(pool.k_cache[0], kc) and torch.equal(pool.v_cache[0], vc)
        assert torch.equal(out, want)
        batch.end_step()


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("Hq,Hkv,D,max_blocks", [(4, 1, 128, 32), (4, 1, 64, 40), (28, 4, 128, 32), (28, 4, 128, 63),
                                                 (64, 16, 64, 32)])
def test_fused_append(cuda, Hq, Hkv, D, max_blocks, dtype):
    _fused_vs_unfused(cuda, 11, len(EDGES), Hq, Hkv, D, EDGES, dtype, max_blocks=max_blocks)


def test_fused_append_edge_lengths_and_ids(cuda):
    lens = [0, 20, 24 * 16 + 5, 40, 1]
    _fused_vs_unfused(cuda, 6, len(lens), 32, 8, 128, lens, max_blocks=24, bad_tail=3)
