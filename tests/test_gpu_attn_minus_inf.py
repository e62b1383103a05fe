"""Keys whose score is -inf weigh nothing wherever they stand: at the start of
a sequence, where they leave a row without a maximum for its first tiles, in
every attention kernel; a row without any finite score is NaN (0 / 0).  Against
float64 softmax attention."""
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


def _run(q, k, v, cu_q, cu_k, H, workspace=None):
    qd = to_dev(q)
    out = torch.full_like(qd, float("nan"))
    A.ragged_attn_fwd(qd, to_dev(k), to_dev(v), out, to_dev(cu_q), to_dev(cu_k), len(cu_q) - 1, H, True,
                      int(np.diff(cu_q).max()), q.shape[-1] ** -0.5, workspace=workspace)
    torch.cuda.synchronize()
    return O.bf16_to_f32(to_np(out))


@pytest.mark.parametrize("kernel,batches,heads,rows,keys,D", [
    ("head_dim 64", 2, 3, 70, 300, 64),
    ("256 rows", 2, 3, 300, 200, 128),
    ("key split, one chunk beside several", 1, 5, 300, 400, 128),
    ("384 rows and tails of 9", 43, 12, 393, 640, 128),
])
@pytest.mark.parametrize("dead", [1, 31, 32, 33, 96, 150])
def test_sequences_that_begin_with_keys_of_score_minus_infinity(kernel, batches, heads, rows, keys, D, dead):
    rng = np.random.default_rng(dead)
    n = batches * heads
    lens = np.array([keys + 13 * (s % 5) for s in range(n)])
    split = kernel.startswith("key split")
    if split:
        lens[0] = 9000
    cu_q = (np.arange(batches + 1) * rows).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    q, k, v = (O.f32_to_bf16((rng.standard_normal(s, np.float32) * 0.5)) for s in
               ((int(cu_q[-1]), heads, D), (int(cu_k[-1]), D), (int(cu_k[-1]), D)))
    q[..., 0] = O.f32_to_bf16(np.ones(q.shape[:-1], np.float32))
    for s in range(n):  # every third sequence is untouched, sequence 1 has no finite score
        if s % 3 != 2:
            k[cu_k[s]:cu_k[s] + (lens[s] if s == 1 else dead), 0] = 0xFF80  # -inf
    print(f"{kernel}: {batches} x {heads} sequences of {rows} rows, {dead} keys of score -inf", flush=True)
    got = _run(q, k, v, cu_q, cu_k, heads, _ops.attention_workspace(DEV) if split else None)
    for s in list(range(min(n, 9))) + list(range(n - 3, n)):
        b, h = divmod(s, heads)
        g = got[cu_q[b]:cu_q[b + 1], h]
        if s == 1:
            assert bool(np.isnan(g).all()), s
            continue
        f = lambda x: O.bf16_to_f32(x).astype(np.float64)
        lo = cu_k[s] + (dead if s % 3 != 2 else 0)
        sc = f(q[cu_q[b]:cu_q[b + 1], h]) @ f(k[lo:cu_k[s + 1]]).T * D ** -0.5
        p = np.exp(sc - sc.max(1, keepdims=True))
        err = np.abs(g - (p / p.sum(1, keepdims=True)) @ f(v[lo:cu_k[s + 1]]))
        worst, mean = float(err.max()), float(err.mean())
        assert worst < 2e-2 and mean < 2e-3, (s, worst, mean)
