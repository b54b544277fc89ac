"""Tiled prefill beyond head_dim 128 with n_rep a divisor of 16, and key parts (GPU).

Head shapes whose q heads straddle the 16-column blocks, 64-dim heads, and launches small enough
that a query block's keys are cut into parts and merged, against the fp64 closed form. Outputs are
rounded to the pool's type once from fp32 sums of fp32-grade weights (two 16-bit parts, relative
error at most 2^-16 in bf16 and 2^-21 in fp16), so a row is off by its own rounding (2^-9 / 2^-12 of
each value) plus 2^-15 of the largest |V|: what FINE_TOL states. Shapes with fp16 weights (relative
error 2^-12 each) get 2^-11 of the largest |V|.
"""
import numpy as np
import pytest
import torch

from oracle import oracle
from test_prefill import check, expected, make_case, run_gpu, to_dev
from unifiedkv_amd import _ext, workloads

ROUND = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}  # one unit in the last place, relative


def _close(got, exp, v_max, dtype, weights, what):
    bound = ROUND[dtype] * np.abs(exp) + weights * v_max
    err = np.abs(got - exp)
    assert np.isfinite(got).all() and (err <= bound).all(), f"{what}: worst excess {np.max(err - bound):.3e}"


def _v_max(case):
    f = lambda a: oracle.bits_to_f32(a, workloads.DTYPE_CODES[case["dtype"]])
    return max(float(np.abs(f(case["v_cache"])).max()), float(np.abs(f(case["v_new"])).max()))


def _parts_bytes(case):
    Hq, Hkv, D = case["q"].shape[1], case["k_cache"].shape[2], case["q"].shape[2]
    return int(_ext.load().ukv_paged_prefill_workspace_bytes(
        len(case["kv_lens"]), len(case["q"]), max(case["chunk"]), Hq, Hkv, D, case["n_rep"],
        case["block_table"].shape[1]))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("n_rep,Hkv,D,prefix,chunk", [
    (7, 2, 128, [0], [1]), (7, 4, 128, [45, 0, 200], [37, 16, 110]), (3, 2, 128, [31, 64], [85, 1]),
    (5, 1, 128, [15], [52]), (6, 2, 128, [0], [43]), (9, 1, 128, [100], [29]), (20, 1, 128, [7], [13]),
    (64, 1, 128, [33], [5]),
    (4, 8, 64, [0, 0, 0], [16, 129, 97]), (1, 2, 64, [63], [385]), (7, 2, 64, [64, 5], [55, 64]), (16, 1, 64, [127], [25]),
])
def test_fine_instances_match_the_closed_form(cuda, n_rep, Hkv, D, prefix, chunk, dtype):
    case = make_case(n_rep * 100 + D + sum(chunk), prefix, chunk, Hq=n_rep * Hkv, Hkv=Hkv, D=D, dtype=dtype)
    out, _ = run_gpu(case, cuda)
    _close(out.float().cpu().numpy(), expected(case), _v_max(case), dtype, 2.0 ** -15,
           f"n_rep={n_rep} Hkv={Hkv} D={D} prefix={prefix} chunk={chunk} {dtype}")


# Launches of few query blocks over many keys. (The second sequence of a batch is short: fewer parts.)
PARTS = [(4, 2, 128, [1531], [37]), (4, 1, 128, [3000, 90], [70, 3]), (16, 1, 128, [2047], [1]),
         (7, 2, 128, [1600], [41]), (5, 1, 128, [4001, 0], [33, 20]), (4, 2, 64, [3100], [64]), (7, 1, 64, [5000, 1], [9, 60])]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("n_rep,Hkv,D,prefix,chunk", PARTS)
def test_key_parts_match_the_closed_form(cuda, n_rep, Hkv, D, prefix, chunk, dtype):
    case = make_case(n_rep * 10 + D + sum(prefix), prefix, chunk, Hq=n_rep * Hkv, Hkv=Hkv, D=D, dtype=dtype)
    assert _parts_bytes(case) > 0  # the shape is cut into parts
    out, _ = run_gpu(case, cuda)
    fine = D != 128 or 16 % n_rep
    _close(out.float().cpu().numpy(), expected(case), _v_max(case), dtype, 2.0 ** -15 if fine else 2.0 ** -11,
           f"parts n_rep={n_rep} Hkv={Hkv} D={D} prefix={prefix} chunk={chunk} {dtype}")


@pytest.mark.gpu
@pytest.mark.parametrize("n_rep,Hkv,D,prefix,chunk", [PARTS[0], PARTS[3], PARTS[5]])
def test_a_launch_without_room_for_its_parts_runs_in_one(cuda, n_rep, Hkv, D, prefix, chunk, monkeypatch):
    case = make_case(n_rep * 10 + D + sum(prefix), prefix, chunk, Hq=n_rep * Hkv, Hkv=Hkv, D=D, dtype="bf16")
    assert _parts_bytes(case) > 0
    empty, refused = torch.empty, []

    def no_scratch(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            refused.append(args)
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", no_scratch)
    out, _ = run_gpu(case, cuda)
    monkeypatch.undo()
    assert refused
    fine = D != 128 or 16 % n_rep
    _close(out.float().cpu().numpy(), expected(case), _v_max(case), "bf16", 2.0 ** -15 if fine else 2.0 ** -11,
           f"one part n_rep={n_rep} Hkv={Hkv} D={D}")


@pytest.mark.gpu
def test_parts_with_an_invalid_page_and_a_last_group_short_of_heads(cuda):
    """A masked page empties one part of the keys; 10 q heads in groups of 4 leave the last group two."""
    import torch

    from unifiedkv_amd import prefill

    case = make_case(5, [1500], [30], Hq=10, Hkv=3, D=128, dtype="bf16")
    bad = case["block_table"].copy()
    bad[0, 20:44] = [-1, 1 << 20] * 12  # keys 320 .. 703: masked
    t = to_dev(case, cuda)
    prefill.write_chunk_kv(t["k_cache"], t["v_cache"], t["k_new"], t["v_new"], t["block_table"], t["cu"], t["kv_lens"], 30)
    t["block_table"] = torch.from_numpy(bad).to(cuda)
    out = prefill.paged_prefill_attention(t["q"], t["k_cache"], t["v_cache"], t["block_table"], t["cu"], t["kv_lens"],
                                          softmax_scale=case["scale"], n_rep=4, max_chunk=30).float().cpu().numpy()
    keep = [p for p in range(bad.shape[1]) if not 20 <= p < 44]  # the same keys without the masked pages
    small = dict(case, block_table=case["block_table"][:, keep], kv_lens=case["kv_lens"] - 24 * 16, n_rep=4)
    _close(out, expected(small), _v_max(case), "bf16", 2.0 ** -11, "masked pages")


@pytest.mark.gpu
@pytest.mark.parametrize("n_rep,Hkv,D,dtype,big", [(4, 2, 128, "bf16", 3.0e38), (7, 2, 128, "bf16", np.inf),
                                                   (7, 2, 128, "bf16", 3.0e38), (7, 1, 64, "fp16", np.inf)])
@pytest.mark.parametrize("prefix,chunk", [([200], [30]), ([4000], [12])])
def test_wide_and_infinite_v(cuda, n_rep, Hkv, D, dtype, big, prefix, chunk):
    """Values the 16-bit P.V cannot carry take the fp32 fallback, in whole blocks and in parts; an
    infinite V gives an infinite output in its dimension and leaves the others alone."""
    case = make_case(9, prefix, chunk, Hq=n_rep * Hkv, Hkv=Hkv, D=D, dtype=dtype)
    case["v_cache"][case["block_table"][0][6], 5, 0, 7] = workloads._round_bits(np.array([big], np.float32), dtype)[0]
    with np.errstate(invalid="ignore"):
        exp = expected(case)
    out, _ = run_gpu(case, cuda)
    got = out.float().cpu().numpy()
    fin = np.isfinite(exp)
    np.testing.assert_array_equal(np.isfinite(got), fin)
    np.testing.assert_array_equal(got[~fin], exp[~fin].astype(np.float32))
    check(np.where(fin, got, 0.0), np.where(fin, exp, 0.0), f"n_rep={n_rep} D={D} |v|={big}")


@pytest.mark.gpu
def test_parts_replay_from_a_captured_graph(cuda):
    import torch

    from unifiedkv_amd import prefill

    case = make_case(3, [1700], [40], Hq=14, Hkv=2, D=128, dtype="fp16")
    t = to_dev(case, cuda)
    args = (t["q"], t["k_cache"], t["v_cache"], t["block_table"], t["cu"], t["kv_lens"])
    kw = dict(softmax_scale=case["scale"], n_rep=7, max_chunk=40)
    want = prefill.paged_prefill_attention(*args, **kw)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        prefill.paged_prefill_attention(*args, **kw)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = prefill.paged_prefill_attention(*args, **kw)
    for _ in range(3):
        got.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        prefill.paged_prefill_attention(*args, **kw)


def test_no_scratch_for_shapes_without_a_tiled_instance():
    lib = _ext.load()
    assert lib.ukv_paged_prefill_workspace_bytes(0, 1, 1, 8, 2, 128, 4, 100) == 0
    assert lib.ukv_paged_prefill_workspace_bytes(1, 64, 64, 8, 2, 96, 4, 1000) == 0


@pytest.mark.gpu
def test_parts_are_taken_only_by_launches_short_of_blocks(cuda):
    """Without a device no shape is cut, so the rule is asked here: 16 blocks a slot (256 CUs, one slot each) and
    more stay whole whatever their keys, launches of few blocks are cut."""
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    size = _ext.load().ukv_paged_prefill_workspace_bytes

    def cut(batch, queries, pages):  # 32/8 heads of 128 dims: blocks of 96 queries
        return size(batch, batch * queries, queries, 32, 8, 128, 4, pages) > 0

    assert not cut(64, 2048, 1000)
    assert not cut(8, 768, 2048)  # 64 pairs of 8 blocks: 512, an XCD's 16 * 32
    assert cut(1, 512, 2048) and cut(1, 96, 100)
    assert not cut(1, 512, 46)  # 23 key tiles: no two parts of 12


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("Hq,Hkv,sink,obs,chunks", [
    (28, 4, 16, 64, [[700, 650], [400, 517]]), (7, 1, 4, 32, [[1900], [40]]), (6, 2, 0, 48, [[300, 90]]),
    (10, 2, 64, 128, [[2500, 300], [128, 140]]),
])
def test_fine_statistics_match_the_oracle(cuda, dtype, Hq, Hkv, sink, obs, chunks):
    """The statistics of head shapes whose n_rep does not divide 16: the weights' two parts are summed and
    taken off alike, so a row's normaliser is off by the fp32 sums' rounding (well under 2^-15; log2 units)."""
    from oracle import snapkv_oracle as so
    from test_obs_stats import _f, _prefill

    r = _prefill(cuda, dtype, chunks, Hq=Hq, Hkv=Hkv, layers=1, sink=sink, obs=obs, seed=13)
    data = r["st"].data.cpu().numpy()
    kept = 0
    for b in range(len(chunks[0])):
        want = so.obs_row_stats(_f(r["dense"][0][b], dtype), _f(r["q_obs"][b, 0], dtype), sink_len=sink, obs_len=obs,
                                n_rep=r["n_rep"], scale=r["scale"])
        got, flags = data[b, 0, :, :, 0], data[b, 0, :, :, 1]
        ok = flags == 0
        kept += int(ok.sum())
        if ok.any():
            assert np.abs(got - want)[ok].max() <= 2.0 ** -14, (b, np.abs(got - want)[ok].max())
    assert kept > 0


def _wide(case, width):
    """The same case in a table of `width` pages a row (zero padded)."""
    table = np.zeros((len(case["block_table"]), width), np.int32)
    table[:, :case["block_table"].shape[1]] = case["block_table"]
    return dict(case, block_table=table)


def _parts_call(case, dev, poison):
    """ukv_paged_prefill_parts over the written pool; returns (output, workspace filled with 0xFF before)."""
    from unifiedkv_amd import prefill

    t, lib = to_dev(case, dev), _ext.load()
    mc, n_rep = max(case["chunk"]), case["n_rep"]
    prefill.write_chunk_kv(t["k_cache"], t["v_cache"], t["k_new"], t["v_new"], t["block_table"], t["cu"], t["kv_lens"], mc)
    (total, Hq, D), Hkv = t["q"].shape, t["k_cache"].shape[2]
    size = _parts_bytes(case)
    ws = torch.full((max(size, 1),), 0xFF, dtype=torch.uint8, device=dev)
    out = torch.full_like(t["q"], poison)
    code = lib.ukv_paged_prefill_parts(
        t["q"].data_ptr(), t["k_cache"].data_ptr(), t["v_cache"].data_ptr(), t["block_table"].data_ptr(), t["cu"].data_ptr(),
        t["kv_lens"].data_ptr(), out.data_ptr(), len(case["chunk"]), total, mc, Hq, Hkv, D, n_rep,
        t["block_table"].shape[1], t["k_cache"].shape[0], _ext.i64_array(t["q"].stride()[:2]),
        _ext.i64_array(t["k_cache"].stride()[:3]), _ext.i64_array(t["v_cache"].stride()[:3]), case["scale"],
        {"bf16": _ext.UKV_DTYPE_BF16, "fp16": _ext.UKV_DTYPE_F16}[case["dtype"]], 0, 0, None, 0, ws.data_ptr(), size,
        torch.cuda.current_stream().cuda_stream)
    assert code == _ext.UKV_OK and size > 0
    return out, ws


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("n_rep,Hkv,D,prefix,chunk", [
    (4, 8, 128, [0, 0], [512, 300]), (4, 2, 128, [90, 0], [37, 64]), (7, 4, 128, [0, 17], [100, 129]),
    (4, 2, 64, [0, 0, 5], [64, 1, 33]), (1, 3, 128, [700], [129]),
])
def test_a_table_wider_than_its_sequences_takes_no_partials(cuda, n_rep, Hkv, D, prefix, chunk, dtype):
    """The plan knows the table's width alone and cuts such a launch; sequences that fill one part are written by
    their blocks, as in an exact table, and leave the scratch as it was."""
    case = _wide(make_case(n_rep + Hkv + D + sum(chunk), prefix, chunk, Hq=n_rep * Hkv, Hkv=Hkv, D=D, dtype=dtype), 2048)
    out, ws = _parts_call(case, cuda, 7.0)
    fine = D != 128 or 16 % n_rep
    _close(out.float().cpu().numpy(), expected(case), _v_max(case), dtype, 2.0 ** -15 if fine else 2.0 ** -11,
           f"wide table n_rep={n_rep} Hkv={Hkv} D={D} {prefix} {chunk}")
    assert int((ws != 0xFF).sum()) == 0  # bytes written


@pytest.mark.gpu
@pytest.mark.parametrize("n_rep,Hkv,D", [(4, 2, 128), (7, 1, 128), (4, 1, 64)])
def test_sequences_in_one_part_beside_sequences_in_many(cuda, n_rep, Hkv, D):
    """One long sequence is merged from its parts, short ones beside it are written whole, and a sequence
    shorter than its chunk (its first queries before key 0) or empty gives NaN rows, as without parts."""
    case = _wide(make_case(21 + D, [3000, 0, 0, 40], [70, 300, 6, 9], Hq=n_rep * Hkv, Hkv=Hkv, D=D, dtype="bf16"), 256)
    want = expected(case)
    lens = np.asarray(case["kv_lens"]).copy()
    out, _ = _parts_call(case, cuda, 7.0)
    fine = D != 128 or 16 % n_rep
    tol = 2.0 ** -15 if fine else 2.0 ** -11
    _close(out.float().cpu().numpy(), want, _v_max(case), "bf16", tol, "one long, three short")
    lens[2], lens[3] = 0, 4  # no keys at all; nine queries of which five lie before the first key
    out, _ = _parts_call(dict(case, kv_lens=lens), cuda, 7.0)
    got = out.float().cpu().numpy()
    _close(got[:370], want[:370], _v_max(case), "bf16", tol, "the others")
    assert np.isnan(got[370:381]).all() and np.isfinite(got[381:]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("long_at", [0, 63, 64, 69, None])
def test_many_sequences_of_which_one_or_none_is_in_parts(cuda, long_at):
    """Seventy sequences in a wide table: each workgroup looks through all lengths, 64 at a time, for one in parts."""
    prefix = [3 * (i % 5) for i in range(70)]
    if long_at is not None:
        prefix[long_at] = 3000
    chunk = [1 + i % 4 for i in range(70)]
    case = _wide(make_case(70, prefix, chunk, Hq=4, Hkv=1, D=128, dtype="bf16"), 256)
    out, ws = _parts_call(case, cuda, 7.0)
    _close(out.float().cpu().numpy(), expected(case), _v_max(case), "bf16", 2.0 ** -11, f"long at {long_at}")
    assert bool((ws != 0xFF).any()) == (long_at is not None)


@pytest.mark.gpu
def test_lengths_the_host_knows_leave_a_wide_table_uncut(cuda):
    """The call in a table of 2048 pages is the one in a table of the sequences' own pages, bit for bit."""
    from unifiedkv_amd import prefill

    case = make_case(5, [0, 40], [300, 257], Hq=16, Hkv=4, D=128, dtype="bf16")
    wide = _wide(case, 2048)
    assert _parts_bytes(wide) > 0 and _parts_bytes(case) == 0
    t, w = to_dev(case, cuda), to_dev(wide, cuda)
    prefill.write_chunk_kv(t["k_cache"], t["v_cache"], t["k_new"], t["v_new"], t["block_table"], t["cu"], t["kv_lens"],
                           300)
    kw = dict(softmax_scale=case["scale"], n_rep=4, max_chunk=300)
    args = (t["q"], t["k_cache"], t["v_cache"])
    want = prefill.paged_prefill_attention(*args, t["block_table"], t["cu"], t["kv_lens"], **kw)
    lens = [int(x) for x in case["kv_lens"]]
    for got in (prefill.paged_prefill_attention(*args, w["block_table"], t["cu"], lens, **kw),
                prefill.paged_prefill_attention(*args, w["block_table"], t["cu"], t["kv_lens"].cpu(), **kw),
                prefill.paged_prefill_attention(*args, w["block_table"], t["cu"], t["kv_lens"],
                                                host_lens=([300, 257], lens), **kw)):
        assert torch.equal(got, want)
    got = prefill.paged_prefill_attention(*args, w["block_table"], t["cu"], t["kv_lens"], host_lens=([300, 257], None),
                                          **kw)  # (not known after all)
    torch.testing.assert_close(got.float(), want.float(), atol=2e-2, rtol=2e-2)
