"""SnapKV block scores of few items: units split over workgroups, uneven units, the finish over groups (GPU).

Against the fp32 closed form with test_random_snapkv_scores' bound (fp16-rounded weights, relative 2^-11
each): block counts around the finish kernel's 30 blocks a workgroup, one and two blocks (no pool), q heads
that leave a group's last unit short (7 heads x 128 queries), and many items (one group).
"""
import numpy as np
import pytest
import torch

from oracle import snapkv_oracle as so
from test_random_shapes import _bits, _down, _f, _up
from unifiedkv_amd import _ext, snapkv

pytestmark = pytest.mark.gpu


def _close(got, want, what):
    err = np.abs(got - want)
    bound = 1e-4 * np.abs(want).max() + 1e-3 * np.abs(want)
    assert got.shape == want.shape and np.all(err <= bound), f"{what}: max err {err.max():.3e}"


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("h_kv,n_rep,D,obs,mid", [
    (2, 7, 128, 128, 16 * 30), (1, 7, 64, 128, 16 * 31 - 5), (4, 7, 128, 64, 16 * 61 + 1), (3, 5, 128, 96, 16 * 29),
    (8, 4, 128, 128, 16 * 90 - 15), (2, 3, 64, 16, 17), (1, 4, 128, 32, 16), (2, 16, 128, 48, 200), (1, 1, 64, 128, 4000),
])
def test_few_items(cuda, h_kv, n_rep, D, obs, mid, dt):
    rng = np.random.default_rng(mid + n_rep)
    sink, L = 5, 5 + mid + obs
    K, Q = _bits(rng, (h_kv, L, D), dt), _bits(rng, (h_kv * n_rep, obs, D), dt)
    got = snapkv.score_layer_blocks(_up(K, dt), _up(Q, dt), sink_len=sink, obs_len=obs, n_rep=n_rep).cpu().numpy()
    want = so.score_layer_blocks(_f(K, dt), _f(Q, dt), sink_len=sink, obs_len=obs, n_rep=n_rep)
    _close(got, want, f"h_kv={h_kv} n_rep={n_rep} D={D} obs={obs} mid={mid} {dt}")


def test_many_items_equal_the_same_items_alone(cuda):
    """96 items run one group each, one item several: the same weights, sums and maxima."""
    g = torch.Generator(device="cuda").manual_seed(1)
    layers, seqs, H, R, D, obs, L = 24, 4, 2, 4, 128, 32, 700
    n = seqs * 44
    pool = torch.randn((layers, n, 16, H, D), generator=g, device="cuda").bfloat16()
    q = torch.randn((seqs, layers, H * R, obs, D), generator=g, device="cuda").bfloat16()
    table = torch.randperm(n, generator=g, device="cuda").to(torch.int32).view(seqs, 44)
    kw = dict(seq_len=L, sink_len=16, obs_len=obs, n_rep=R)
    many = snapkv.score_blocks(q, pool, table, **kw)
    for b, l in ((0, 0), (2, 11), (3, 23)):
        one = snapkv.score_blocks(q[b:b + 1, l:l + 1].contiguous(), pool[l:l + 1], table[b:b + 1], **kw)
        torch.testing.assert_close(one[0], many[b * layers + l], rtol=2e-4, atol=1e-6)


def _score_call(lib, q, k, out, L, obs, n_rep, size):
    """ukv_snapkv_scores of dense K [layers][H][L][D] with a workspace of `size` bytes; returns the status."""
    layers, H, _, D = k.shape
    ws = torch.empty(max(size, 1), dtype=torch.uint8, device=k.device)
    return lib.ukv_snapkv_scores(
        q.data_ptr(), _ext.i64_array(q.stride()[:3]), k.data_ptr(),
        _ext.i64_array((k.stride(0), 0, k.stride(2), k.stride(1))), None, 0, 0, layers, 1, L, 16, obs, H * n_rep, H, D,
        n_rep, 16, D ** -0.5, _ext.UKV_DTYPE_F16, out.data_ptr(), out.stride(0), ws.data_ptr(), size,
        torch.cuda.current_stream().cuda_stream)


def test_a_workspace_sized_for_the_longest_sequence_serves_the_shorter_ones(cuda):
    """Where a shorter sequence's own plan takes more scratch it runs with fewer ranges or groups; below the
    least any plan takes it is refused."""
    lib, layers, H, R, D, obs = _ext.load(), 12, 2, 2, 64, 32
    size = lambda L: int(lib.ukv_snapkv_workspace_bytes(layers, 1, L, 16, obs, H * R, H, D, R, 16))
    assert size(4100) < size(4050)
    g = torch.Generator(device="cuda").manual_seed(2)
    q = torch.randn((layers, H * R, obs, D), generator=g, device="cuda").half()
    for L in (4050, 4100, 3000, 200):
        k = torch.randn((layers, H, L, D), generator=g, device="cuda").half()
        n = int(lib.ukv_snapkv_block_count(L, 16, obs, 16))
        want, got = (torch.empty((layers, n), device="cuda") for _ in range(2))
        assert _score_call(lib, q, k, want, L, obs, R, size(L)) == _ext.UKV_OK
        assert _score_call(lib, q, k, got, L, obs, R, size(4100)) == _ext.UKV_OK, L
        torch.testing.assert_close(got, want, rtol=2e-4, atol=1e-6)
    assert _score_call(lib, q, k, got, 200, obs, R, 1024) == _ext.UKV_ERR_WORKSPACE
