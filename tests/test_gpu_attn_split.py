"""Key-split attention (pkv_ragged_attn_fwd_ws): launches of a few sequences
with per-head keys -- one layer's heads, as MegaCache.attend issues them
(reference call site pyramidkv/_mega_cache.py:540-559) -- split each
sequence's keys into chunks that spread over every compute unit, and a
second launch merges each query tile's chunks in chunk order.

Checked against float64 softmax attention at the north star's tolerance
(max-abs 2e-2, mean-abs 2e-3): mixed key lengths (empty, one key, tile
edges, and long sequences that split), partial query tiles, every reference
mode of the fast pass and the slow pass inside a chunk, and strided
layouts through the torch op.  The split output also agrees with the unsplit kernels',
repeats bit for bit, and a workspace below the required size runs the
unsplit kernels."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O

if torch.cuda.is_available():
    from gpu_util import DEV, to_dev, to_np
    from pyramidkv import _abi as A
    from pyramidkv import _ops

pytestmark = pytest.mark.gpu

D = 128


def _case(rng, Lq, Lk, H, scale=0.5):
    B = len(Lq)
    cu_q = np.concatenate([[0], np.cumsum(Lq)]).astype(np.int32)
    lk = np.asarray(Lk).reshape(B * H)
    cu_k = np.concatenate([[0], np.cumsum(lk)]).astype(np.int32)
    q = (rng.standard_normal((cu_q[-1], H, D)) * scale).astype(np.float32)
    k = (rng.standard_normal((cu_k[-1], D)) * scale).astype(np.float32)
    v = (rng.standard_normal((cu_k[-1], D)) * scale).astype(np.float32)
    return O.f32_to_bf16(q), O.f32_to_bf16(k), O.f32_to_bf16(v), cu_q, cu_k


def _run(q, k, v, cu_q, cu_k, B, H, workspace):
    qd, kd, vd = to_dev(q), to_dev(k), to_dev(v)
    out = torch.full_like(qd, float("nan"))
    A.ragged_attn_fwd(qd, kd, vd, out, to_dev(cu_q), to_dev(cu_k), B, H, True, int(np.diff(cu_q).max()),
                      D ** -0.5, workspace=workspace)
    torch.cuda.synchronize()
    return to_np(out)


def _check(got_u16, q, k, v, cu_q, cu_k, H):
    got = O.bf16_to_f32(got_u16).astype(np.float64)
    want = O.ragged_attention_ref(O.bf16_to_f32(q), O.bf16_to_f32(k), O.bf16_to_f32(v), cu_q, cu_k, H, True)
    err = np.abs(got - want)
    assert np.isfinite(got).all()
    assert err.max() < 2e-2 and err.mean() < 2e-3, (err.max(), err.mean())
    return got


def _ws():
    return _ops.attention_workspace(DEV)


def test_workspace_size_reported():
    n = A.ragged_attn_workspace_size()
    assert n > 0 and n == int(_ops.ops().ragged_attention_workspace_size())
    assert _ws().numel() >= n


@pytest.mark.parametrize("case", [
    # one layer's heads at a rollout's shape, scaled down: long per-head keys over few query tiles
    dict(Lq=[1000], Lk=[[8000, 5000, 3100, 7777]], H=4),
    # tile edges and empty / one-key heads beside long ones; a partial query tile of 8 rows
    dict(Lq=[392, 1], Lk=[[0, 1, 31, 33, 9000, 64], [6000, 32, 4097, 0, 1, 12000]], H=6),
    # a batch without queries between two with
    dict(Lq=[500, 0, 300], Lk=[[7000, 100], [5000, 5000], [2, 9999]], H=2),
])
def test_split_launch_vs_float64_and_unsplit(case):
    rng = np.random.default_rng(41)
    H = case["H"]
    q, k, v, cu_q, cu_k = _case(rng, case["Lq"], case["Lk"], H)
    print(f"split attention Lq={case['Lq']} Lk={case['Lk']}", flush=True)
    B = len(case["Lq"])
    got = _run(q, k, v, cu_q, cu_k, B, H, _ws())
    split = _check(got, q, k, v, cu_q, cu_k, H)
    plain = O.bf16_to_f32(_run(q, k, v, cu_q, cu_k, B, H, None)).astype(np.float64)
    assert np.abs(split - plain).max() < 2e-2
    again = _run(q, k, v, cu_q, cu_k, B, H, _ws())
    assert np.array_equal(got, again), "split launch is not deterministic"


def test_split_reference_modes_and_slow_pass_in_chunks():
    """Query rows scaled by 1, 2 and 4 and per-head constant key blocks at the
    start of different chunks, so that a row's chunks take different
    references (P = 2^S, P = 2^(S - m), and the moving-maximum pass after a
    spike ~98 or ~130 log2 units above a chunk's first tile) before they are
    merged."""
    rng = np.random.default_rng(43)
    H = 4
    Lq, Lk = [1000], [[9000, 8000, 6000, 7500]]
    q, k, v, cu_q, cu_k = _case(rng, Lq, Lk, H)
    alpha = np.array([1.0, 2.0, 4.0], np.float32)[np.arange(q.shape[0]) % 3]
    q[:] = O.f32_to_bf16(np.broadcast_to(alpha[:, None, None], q.shape).astype(np.float32))
    lk = np.diff(cu_k)
    for h in range(H):
        for j, (pos, val) in enumerate([(0, 0.8), (2500, -1.0), (4000, 3.0), (lk[h] - 1, 1.5), (5500, 8.0)]):
            if pos < lk[h] and (h + j) % 2 == 0:
                n = min(32, int(lk[h] - pos)) if val not in (1.5, 8.0) else 1
                k[cu_k[h] + pos:cu_k[h] + pos + n] = O.f32_to_bf16(np.full((n, D), val, np.float32))
    got = _run(q, k, v, cu_q, cu_k, 1, H, _ws())
    _check(got, q, k, v, cu_q, cu_k, H)


def test_split_needs_the_whole_workspace():
    """A workspace below pkv_ragged_attn_workspace_size runs the unsplit
    kernels: the output equals the launch without a workspace bit for bit."""
    rng = np.random.default_rng(47)
    q, k, v, cu_q, cu_k = _case(rng, [800], [[7000, 3000]], 2)
    small = torch.empty(A.ragged_attn_workspace_size() - 1, dtype=torch.uint8, device=DEV)
    got = _run(q, k, v, cu_q, cu_k, 1, 2, small)
    plain = _run(q, k, v, cu_q, cu_k, 1, 2, None)
    assert np.array_equal(got, plain)
    _check(got, q, k, v, cu_q, cu_k, 2)


def test_split_through_the_torch_op_on_strided_views():
    """ragged_attention with the device workspace on Q / K / V / O that are
    the first 128 columns of 256-wide rows."""
    rng = np.random.default_rng(53)
    H = 3
    q, k, v, cu_q, cu_k = _case(rng, [700], [[6500, 2000, 9100]], H)
    wide = lambda a: np.concatenate([a, np.zeros(a.shape, np.uint16)], axis=-1)
    qw, kw, vw = to_dev(wide(q)), to_dev(wide(k)), to_dev(wide(v))
    out = _ops.ragged_attention(qw[..., :D], kw[..., :D], vw[..., :D], to_dev(cu_q), to_dev(cu_k), 700,
                                workspace=_ws())
    torch.cuda.synchronize()
    _check(to_np(out), q, k, v, cu_q, cu_k, H)


@pytest.mark.parametrize("Lq,Lk,H,kv_per_head", [
    # two rounds of items: 108 tiles, above 3/8 of the compute units
    ([1300, 1300], [[3000 + 251 * h for h in range(9)]] * 2, 9, True),
    # three rounds: 290 tiles, more than there are compute units
    ([290] * 29, [[4200 + (s * 37 + h * 211) % 1500 for h in range(5)] for s in range(29)], 5, True),
    # more than 64 sequences, several per lane of the plan, some without rows or keys
    ([10, 0, 33] * 13, [[(s * 613 + h * 97) % 2600 for h in range(3)] for s in range(39)], 3, True),
    # the edges of a chunk: one key more and fewer than the shortest two, and a
    # single row over a long sequence
    ([1], [[1023, 1024, 1025, 1151, 20000]], 5, True),
    # key sequences shared by the heads
    ([257, 5], [[5000], [1300]], 4, False),
])
def test_split_by_the_op_vs_float64(Lq, Lk, H, kv_per_head):
    """The op without a workspace, which splits by its own rule: against
    float64, and twice with the same bits, other ones than the unsplit kernels'
    (a chunk rounds its probabilities against its own reference)."""
    rng = np.random.default_rng(61)
    B = len(Lq)
    cu_q = np.concatenate([[0], np.cumsum(Lq)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(np.asarray(Lk).reshape(-1))]).astype(np.int32)
    shape = (int(cu_k[-1]), D) if kv_per_head else (int(cu_k[-1]), H, D)
    q, k, v = (O.f32_to_bf16((rng.standard_normal(s) * 0.5).astype(np.float32))
               for s in ((int(cu_q[-1]), H, D), shape, shape))
    print(f"attention split by the op: {B} x {H} sequences, up to {np.max(Lq)} x {np.max(Lk)}", flush=True)
    run = lambda: to_np(_ops.ragged_attention(to_dev(q), to_dev(k), to_dev(v), to_dev(cu_q), to_dev(cu_k),
                                              int(np.max(Lq)), kv_per_head=kv_per_head))
    assert _workspace_for(B, H, int(np.max(Lq)), shape[0] // (B * H if kv_per_head else B)) > 0
    got = run()
    assert np.array_equal(got, run())
    qd, plain = to_dev(q), torch.empty_like(to_dev(q))
    A.ragged_attn_fwd(qd, to_dev(k), to_dev(v), plain, to_dev(cu_q), to_dev(cu_k), B, H, kv_per_head,
                      int(np.max(Lq)), D ** -0.5)
    assert not np.array_equal(got, to_np(plain)), "the launch did not split"
    got = O.bf16_to_f32(got).astype(np.float64)
    want = O.ragged_attention_ref(O.bf16_to_f32(q), O.bf16_to_f32(k), O.bf16_to_f32(v), cu_q, cu_k, H, kv_per_head)
    err = np.abs(got - want)
    assert err.max() < 2e-2 and err.mean() < 2e-3, (err.max(), err.mean())


def test_split_chunks_of_keys_whose_scores_are_minus_infinity():
    """Keys whose score is -inf weigh nothing, also where they are the first
    tile of a chunk, or all of it, and other chunks have finite scores."""
    rng = np.random.default_rng(53)
    q, k, v, cu_q, cu_k = _case(rng, [300], [[9000, 7000]], 2)
    q[..., 0] = O.f32_to_bf16(np.ones(q.shape[:-1], np.float32))
    k[cu_k[0] + 500:cu_k[0] + 6000, 0] = 0xFF80  # -inf
    k[cu_k[1] + 700:cu_k[1] + 7000, 0] = 0xFF80
    got = _run(q, k, v, cu_q, cu_k, 1, 2, _ws())
    _check(got, q, k, v, cu_q, cu_k, 2)


def test_split_rows_whose_scores_are_all_minus_infinity():
    """A row without a finite score is NaN, as 0 / 0 and in the unsplit
    kernels, whether its sequence is one chunk of the launch or many; the
    other sequences are not touched by it."""
    rng = np.random.default_rng(59)
    q, k, v, cu_q, cu_k = _case(rng, [300], [[9000, 400, 5000]], 3)
    q[..., 0] = O.f32_to_bf16(np.ones(q.shape[:-1], np.float32))
    k[:cu_k[2], 0] = 0xFF80  # -inf
    for ws in (None, _ws()):
        got = O.bf16_to_f32(_run(q, k, v, cu_q, cu_k, 1, 3, ws))
        assert np.isnan(got[:, :2]).all() and np.isfinite(got[:, 2]).all()


def _workspace_for(batches, heads, rows, keys=0, head_dim=D):
    return int(A.lib().pkv_ragged_attn_workspace_for(
        A.AttnArgs(num_batches=batches, num_heads_q=heads, max_seqlen_q=rows, head_dim=head_dim), keys))


def test_workspace_is_sized_by_the_launch():
    """One, two or three items per compute unit, by the query tiles of 256
    rows; the full size serves the largest."""
    full, cus = A.ragged_attn_workspace_size(), torch.cuda.get_device_properties(0).multi_processor_count
    sizes = [_workspace_for(1, 1, 256 * t) for t in (1, cus * 3 // 8, cus * 3 // 8 + 1, cus * 9 // 10, cus + 1)]
    assert sizes[0] == sizes[1] < sizes[2] == sizes[3] < sizes[4] == full
    assert full // 3 <= sizes[0] < full // 3 + 65536
    assert _workspace_for(1, 1, 256 * cus) == _workspace_for(1, 1, 512 * cus) == _workspace_for(1, 257, 1) == 0
    assert _workspace_for(1, 1, 256, head_dim=64) == 0
    # no sequence long enough for two chunks and what a second launch costs
    bound = lambda keys: int(A.lib().pkv_ragged_attn_workspace_bound(
        A.AttnArgs(num_batches=1, num_heads_q=3, max_seqlen_q=256, head_dim=D), keys))
    assert bound(1024) == 0 and bound(1025) == bound(0) == sizes[0] == _workspace_for(1, 3, 256, 1024)


def test_no_room_for_the_workspace_runs_unsplit():
    """A device whose memory would not hold the workspace attends all the same
    (the limit is the allocator's own)."""
    rng = np.random.default_rng(67)
    q, k, v, cu_q, cu_k = _case(rng, [300], [[9000, 7000]], 2)
    args = [to_dev(x) for x in (q, k, v, cu_q, cu_k)]
    plain = _run(q, k, v, cu_q, cu_k, 1, 2, None)
    split = _ops.ragged_attention(*args, 300)
    assert not np.array_equal(to_np(split), plain)  # other chunks, other roundings
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + (8 << 20)
    torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(_workspace_for(1, 2, 300), dtype=torch.uint8, device=DEV)
        out = _ops.ragged_attention(*args, 300)
        assert np.array_equal(to_np(out), plain)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(_ops.ragged_attention(*args, 300), split)


def test_split_by_the_longest_sequence_whatever_buffer_holds_the_keys():
    """With max_seqlen_k the rule reads that alone: one long sequence beside
    short ones splits, and the bits are the same where K is part of a larger
    buffer."""
    rng = np.random.default_rng(71)
    H = 10
    q, k, v, cu_q, cu_k = _case(rng, [300], [[2500] + [10 + h for h in range(H - 1)]], H)
    plain = _run(q, k, v, cu_q, cu_k, 1, H, None)
    room = lambda a: np.concatenate([a, np.zeros((40000, D), np.uint16)])
    runs = [to_np(_ops.ragged_attention(to_dev(q), to_dev(kk), to_dev(vv), to_dev(cu_q), to_dev(cu_k), 300,
                                        max_seqlen_k=2500)) for kk, vv in ((k, v), (room(k), room(v)))]
    assert np.array_equal(*runs)
    assert not np.array_equal(runs[0], plain)  # split: other roundings
    _check(runs[0], q, k, v, cu_q, cu_k, H)
