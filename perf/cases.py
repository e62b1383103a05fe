"""The workloads by which this framework's speed is judged, each through its
public entry points.

Sizes are those of the Wan2.1-T2V-1.3B shaped rollout that the cache serves
(30 layers of 12 heads of 128, 30 x 52 tokens per latent frame, chunks of 3
frames, a 512-token text context) and of the small grids of the tests, with
odd sizes between them.  A case names its ``kind``; the kinds, and what each
stands for in a user's program:

* ``step``      one layer's denoising pass: MegaCache.update (noisy) of the
                block's K and V, then MegaCache.attend of its queries (plan,
                pack with RoPE, ragged attention), the call pattern of 4 of a
                chunk's 5 forwards;
* ``commit``    one layer's cache through a whole block: the first noisy pass
                and the clean pass that commits it (FIFO shift, middle
                writes, Veil merge), rolling on block after block;
* ``cache``     the cache side of a forward over all layers: update, then
                MegaCache.attend_kv (plan + pack with RoPE) per layer;
* ``attn``      ragged attention of many (layer, head) sequences with a key
                length per head;
* ``cross``     attention of a block's queries over the shared text context
                (flash_attn_varlen_func's layout);
* ``evict``     the Veil merge of evicted frames, many or one per call;
* ``qk``        what turns the QKV product into attention operands: the q and
                k RMSNorms on its column slices and the query RoPE;
* ``residual``  the gated residual update of the fp32 stream with the
                modulated LayerNorm that reads it next;
* ``dit``       a whole forward of the causal DiT through its caches.

``exact`` restates each kind in 64 bits with plain torch, without this
package: the cache policy by the frames that a head holds at a time.
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "pyramid-forcing_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

DEV = "cuda:0"
D = 128                                   # head_dim
MAX_SINK, MAX_MIDDLE, MAX_RECENT = 3, 24, 4  # frames per head of the shipped policy's pools
SINKS = {-1: 1, 1: 3, 2: 3}               # sink frames of Wave, Anchor and Veil heads
PERIOD, BUCKET, INTERVAL, RING = 6, 4, 6, 4  # Wave buckets, Anchor ring
MERGE_CAP, BLOCK, GROUPS = 4, 4, 420      # Veil: anchors kept, frames per block, groups an anchor can hold


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    full = dict(heads=12, grid_h=30, grid_w=52, frames=3)
    return [
        # the smallest cache call: latency and launches (the smoke test's shape)
        dict(name="step_tiny", kind="step", heads=3, grid_h=8, grid_w=8, frames=3, chunks=3, labels=0),
        # an odd grid (no whole 2x2 patches), 2-frame blocks
        dict(name="step_odd", kind="step", heads=7, grid_h=21, grid_w=33, frames=2, chunks=11, labels=1),
        # one layer of the production rollout in its steady state
        dict(name="step_layer", kind="step", chunks=13, labels=2, **full),
        # that layer's cache from block to block
        dict(name="commit_layer", kind="commit", chunks=13, labels=3, **full),
        # the cache side of a whole forward, 30 layers
        dict(name="cache_30", kind="cache", layers=30, chunks=13, labels=4, **full),
        # every (layer, head) sequence of a forward in one launch
        dict(name="attn_30", kind="attn", batches=30, heads=12, rows=4680, keys_lo=6240, keys_hi=32760),
        # cross-attention of one block to the text context
        dict(name="cross_text", kind="cross", heads=12, rows=4680, keys=512),
        # 40 frames leaving the window in one call, and one frame per call
        dict(name="evict_40", kind="evict", heads=12, grid_h=30, grid_w=52, frames=40),
        dict(name="evict_1", kind="evict", heads=12, grid_h=30, grid_w=52, frames=1),
        # the row operations of one transformer block
        dict(name="qk_rows", kind="qk", heads=12, rows=4680),
        dict(name="residual_rows", kind="residual", cols=1536, rows=4680),
        # two blocks of the DiT, embeddings and head
        dict(name="dit_forward", kind="dit", blocks=2, ffn=8960, text_len=512, text_dim=4096, chunks=7, labels=5,
             **full),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _grid(rng: random.Random) -> dict:
    while True:
        h, w = rng.randint(6, 30), rng.randint(8, 52)
        if h * w >= 48:
            return dict(grid_h=h, grid_w=w)


def draw(rng: random.Random):
    kind = rng.choice(["step", "step", "commit", "cache", "attn", "cross", "evict", "qk", "residual", "dit"])
    c = dict(kind=kind)
    if kind in ("step", "commit", "cache", "dit"):
        c.update(_grid(rng), heads=rng.randint(1, 12), frames=rng.randint(1, 3), chunks=rng.randint(1, 24),
                 labels=rng.randint(6, 1 << 20))
    if kind == "cache":
        c.update(layers=_log(rng, 1, 30))
    if kind == "dit":
        c.update(blocks=rng.randint(1, 3), ffn=64 * rng.randint(8, 140), text_len=_log(rng, 16, 512),
                 text_dim=64 * rng.randint(1, 64))
    if kind == "attn":
        hi = _log(rng, 700, 32760)
        c.update(batches=_log(rng, 1, 30), heads=rng.randint(1, 12), rows=_log(rng, 96, 4680),
                 keys_lo=rng.randint(64, hi), keys_hi=hi)
    if kind == "cross":
        c.update(heads=rng.randint(1, 16), rows=_log(rng, 48, 4680), keys=_log(rng, 16, 512))
    if kind == "evict":
        c.update(_grid(rng), heads=rng.randint(1, 16), frames=_log(rng, 1, 64))
    if kind == "qk":
        c.update(heads=rng.randint(1, 16), rows=_log(rng, 48, 4680))
    if kind == "residual":
        c.update(cols=32 * rng.randint(8, 128), rows=_log(rng, 48, 4680))
    return c


# ---------------------------------------------------------------------------
# inputs (from the seed alone)
# ---------------------------------------------------------------------------
def _gen(*key) -> torch.Generator:
    n = 0
    for k in key:
        n = (n * 1000003 + int(k) + 17) % ((1 << 61) - 1)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    return g


def _rand(g: torch.Generator, *shape, std: float = 1.0) -> torch.Tensor:
    return (torch.randn(shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _labels(case, layers: int):
    rng = random.Random(case["labels"])
    return [[rng.choice([-1, 1, 2]) for _ in range(case["heads"])] for _ in range(layers)]


def _fs(case) -> int:
    return case["grid_h"] * case["grid_w"]


def _chunk(case, seed: int, layer: int, chunk: int):
    """K (RMS-normalised scale) and V of a chunk, [frames * tokens, heads, D]."""
    n = case["frames"] * _fs(case)
    g = _gen(seed, 1, layer, chunk)
    return _rand(g, n, case["heads"], D), _rand(g, n, case["heads"], D, std=0.5)


def _queries(case, seed: int) -> torch.Tensor:
    return _rand(_gen(seed, 2), 1, case["frames"] * _fs(case), case["heads"], D)


def _key_lengths(case, seed: int):
    rng = random.Random(seed)
    lo, hi = case["keys_lo"], case["keys_hi"]
    return [rng.randint(lo, hi) for _ in range(case["batches"] * case["heads"])]


def _attn_inputs(case, seed: int):
    g = _gen(seed, 3)
    lens = _key_lengths(case, seed)
    q = _rand(g, case["batches"] * case["rows"], case["heads"], D)
    return q, _rand(g, sum(lens), D), _rand(g, sum(lens), D, std=0.5), lens


def _cross_inputs(case, seed: int):
    g = _gen(seed, 4)
    return (_rand(g, case["rows"], case["heads"], D), _rand(g, case["keys"], case["heads"], D),
            _rand(g, case["keys"], case["heads"], D, std=0.5))


def _evict_inputs(case, seed: int):
    g = _gen(seed, 5)
    shape = (case["frames"], case["heads"], _fs(case), D)
    return _rand(g, *shape), _rand(g, *shape), torch.rand(case["frames"], generator=g, device=DEV) * 0.9 + 0.1


def _qk_inputs(case, seed: int):
    g = _gen(seed, 6)
    C = D * case["heads"]
    qkv = _rand(g, case["rows"], 3 * C)
    w = [1.0 + 0.1 * torch.randn(C, generator=g, device=DEV) for _ in range(2)]
    tok = torch.arange(case["rows"], device=DEV)
    pos = torch.stack([60 + tok // 1560, tok % 1560 // 52, tok % 52], dim=1)
    return qkv, w[0], w[1], pos.repeat_interleave(case["heads"], dim=0).contiguous()


def _residual_inputs(case, seed: int):
    g = _gen(seed, 7)
    n, C = case["rows"], case["cols"]
    x = torch.randn(n, C, generator=g, device=DEV)
    y = _rand(g, n, C)
    return x, y, *(0.3 * torch.randn(C, generator=g, device=DEV) for _ in range(3))


def _dit_shape(case) -> dict:
    return dict(num_blocks=case["blocks"], dim=D * case["heads"], heads=case["heads"], ffn=case["ffn"],
                text_dim=case["text_dim"], text_len=case["text_len"], grid_h=case["grid_h"], grid_w=case["grid_w"])


def _dit_inputs(case, seed: int):
    g = _gen(seed, 8)
    text = _rand(g, case["text_len"], case["text_dim"])
    return text, _rand(g, 16, case["frames"], 2 * case["grid_h"], 2 * case["grid_w"])


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _caches(case, seed: int, layers: int):
    """The caches of a rollout `chunks` chunks in, under the shipped policy."""
    from pyramidkv import factory
    from pyramidkv._mega_cache import build_mega_caches
    from pyramidkv.rope import wan_freqs
    comps = factory.shipped_compositions(layers, case["heads"], labels=_labels(case, layers))
    caches = build_mega_caches(layers, case["heads"], D, _fs(case), MAX_SINK, MAX_MIDDLE, MAX_RECENT, comps,
                               device=DEV, freqs=wan_freqs(D), spatial_width=case["grid_w"],
                               spatial_height=case["grid_h"], **factory.PYRAMID_FORCING_REMAP)
    for c in range(case["chunks"]):
        for l, cache in enumerate(caches):
            k, v = _chunk(case, seed, l, c)
            cache.update(k[None], v[None], c * case["frames"] * _fs(case), cache_update_mode="clean")
    return caches


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("step", "commit", "cache"):
        layers = case.get("layers", 1)
        s["caches"] = _caches(case, seed, layers)
        s["kv"] = [tuple(t[None] for t in _chunk(case, seed, l, case["chunks"])) for l in range(layers)]
        s["start"] = case["chunks"] * case["frames"] * _fs(case)
        s["q"] = _queries(case, seed)
        if kind == "cache":  # the tokens that a layer's plan packs: known to the program from its policy
            s["caches"][-1].update(*s["kv"][-1], s["start"], cache_update_mode="noisy")
            s["total"] = int(s["caches"][-1].attend_kv(s["start"], case["frames"])[-1].item())
    elif kind == "attn":
        q, k, v, lens = _attn_inputs(case, seed)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        i32 = dict(dtype=torch.int32, device=DEV)
        s.update(q=q, k=k, v=v, cu_k=torch.tensor(cu, **i32),
                 cu_q=torch.arange(0, (case["batches"] + 1) * case["rows"], case["rows"], **i32))
    elif kind == "cross":
        q, k, v = _cross_inputs(case, seed)
        i32 = dict(dtype=torch.int32, device=DEV)
        s.update(q=q, k=k, v=v, cu_q=torch.tensor([0, case["rows"]], **i32),
                 cu_k=torch.tensor([0, case["keys"]], **i32))
    elif kind == "evict":
        from pyramidkv import _mega_state_ops, _mega_state_ref, _ops
        H, F, FS = case["heads"], case["frames"], _fs(case)
        k, v, w = _evict_inputs(case, seed)
        z = lambda *shape, dt=torch.float32: torch.zeros(shape, dtype=dt, device=DEV)
        bf, i32, i64 = torch.bfloat16, torch.int32, torch.int64
        rec = _mega_state_ops.pack_states([_mega_state_ref.make_merge(2, 6) for _ in range(H)])
        s.update(k=k, v=v, w=w, states=torch.frombuffer(bytearray(rec.tobytes()), dtype=torch.uint8).to(DEV),
                 times=torch.arange(1, 1 << 22, dtype=i64, device=DEV), at=0,
                 desc=[torch.full((H * F,), -1, dtype=i32, device=DEV) for _ in range(8)],
                 acc=[z(H, 2, GROUPS, D), z(H, 2, GROUPS, D), z(H, 2, GROUPS, 3, dt=i64), z(H, 2, FS, dt=i32),
                      z(H, 2, GROUPS), z(H, 2, dt=i32), z(H, 2), z(H, 6, GROUPS, D, dt=bf), z(H, 6, GROUPS, D, dt=bf),
                      z(H, 6, GROUPS, 3, dt=i64), z(H, 6, dt=i32)],
                 ws=z(_ops.ops().mega_evict_merge_workspace_size(H), dt=torch.uint8))
    elif kind == "qk":
        from pyramidkv.rope import flat_freq_parts, wan_freqs
        s["qkv"], s["wq"], s["wk"], s["pos"] = _qk_inputs(case, seed)
        s["freqs"] = flat_freq_parts(wan_freqs(D), DEV)
    elif kind == "residual":
        s["x"], s["y"], s["gate"], s["mul"], s["add"] = _residual_inputs(case, seed)
    elif kind == "dit":
        from pyramidkv.causal_dit import CausalDiT, WanShape
        text, s["latent"] = _dit_inputs(case, seed)
        s["caches"] = _caches(case, seed, case["blocks"])
        s["model"] = CausalDiT(WanShape(**_dit_shape(case)), DEV, seed=int(seed))
        s["model"].set_context(text)
        s["start"] = case["chunks"] * case["frames"] * _fs(case)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "step":
        cache = s["caches"][0]
        cache.update(*s["kv"][0], s["start"], cache_update_mode="noisy")
        out = cache.attend(s["q"], s["start"])
        mgr = cache.ctx.mgr
        return dict(out=out, recent_k=mgr.recent_k_pool(), recent_v=mgr.recent_v_pool(),
                    recent_pos=mgr.recent_pos_pool())
    if kind == "commit":
        cache = s["caches"][0]
        cache.update(*s["kv"][0], s["start"], cache_update_mode="noisy")
        cache.update(*s["kv"][0], s["start"], cache_update_mode="clean")
        s["start"] += case["frames"] * _fs(case)
        mgr = cache.ctx.mgr
        return dict(recent_k=mgr.recent_k_pool(), recent_v=mgr.recent_v_pool(), recent_pos=mgr.recent_pos_pool(),
                    middle_k=mgr.middle_k_pool(), middle_v=mgr.middle_v_pool(), middle_pos=mgr.middle_pos_pool(),
                    merge_k=mgr.merge_k_pool(), merge_v=mgr.merge_v_pool(), merge_pos=mgr.merge_pos_pool(),
                    states=cache.states_bytes_for_layer, valid=mgr.valid_count())
    if kind == "cache":
        for cache, kv in zip(s["caches"], s["kv"]):
            cache.update(*kv, s["start"], cache_update_mode="noisy")
            cu = cache.attend_kv(s["start"], case["frames"])
        mgr, n = s["caches"][-1].ctx.mgr, s["total"]
        return dict(k=mgr.k_flat_out().view(-1, D)[:n], v=mgr.v_flat_out().view(-1, D)[:n],
                    pos=mgr.pos_flat_out()[:n], cu=cu, recent_k=mgr.recent_k_pool(), recent_v=mgr.recent_v_pool())
    if kind == "attn":
        from pyramidkv import _ops
        return _ops.ragged_attention(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], case["rows"], kv_per_head=True)
    if kind == "cross":
        from pyramidkv._mega_attention import flash_attn_varlen_func
        return flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], case["rows"], case["keys"])
    if kind == "evict":
        from pyramidkv import _ops
        F = case["frames"]
        t = s["times"][s["at"]:s["at"] + F]
        s["at"] += F
        _ops.ops().mega_evict_merge(s["states"], t, s["k"], s["v"], case["grid_w"], s["w"], *s["desc"], *s["acc"],
                                    s["ws"])
        a = s["acc"]
        return dict(merge_k=a[7], merge_v=a[8], merge_pos=a[9], merge_count=a[10], sum_k=a[0], sum_v=a[1],
                    states=s["states"], desc=s["desc"][0])
    if kind == "qk":
        from pyramidkv import _ops
        ops, C = _ops.ops(), D * case["heads"]
        q = ops.dit_rms_norm(s["qkv"][:, :C], s["wq"], 1e-6)
        k = ops.dit_rms_norm(s["qkv"][:, C:2 * C], s["wk"], 1e-6)
        return dict(q=ops.rope_apply(q.view(-1, D), s["pos"], *s["freqs"]), k=k)
    if kind == "residual":
        from pyramidkv import _ops
        out = _ops.ops().dit_residual_layer_norm_(s["x"], s["y"], s["gate"], s["mul"], s["add"], True, 1e-6)
        return dict(x=s["x"], out=out)
    mgr = s["caches"][0].ctx.mgr
    out = s["model"].forward(s["latent"], 500.0, s["start"], s["caches"], "noisy")
    return dict(velocity=out, recent_k=mgr.recent_k_pool(), recent_v=mgr.recent_v_pool())


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _held(case, label: int, t_now: int, clean: bool):
    """The segments of one head for a query frame t_now, in plan order: lists
    of (what, t): ("sink", t), ("recent", t), ("middle", t) frames and
    ("merge", (block, median t)) anchors, after the block at `chunks` came in
    by a noisy (or clean) pass."""
    done = case["chunks"] * case["frames"]     # frames committed
    seen = done + case["frames"]               # frames in the sink and the recent FIFO
    if clean:
        done = seen
    cap = SINKS[label]
    segs = [("sink", t) for t in range(min(cap, seen))]
    segs += [("recent", t) for t in range(max(cap, seen - MAX_RECENT), seen)]
    if label in (-1, 1):
        ts = [t for t in range(done) if t % PERIOD == (t_now % PERIOD if label == -1 else 0)]
        ring = [None] * (BUCKET if label == -1 else RING)
        for i, t in enumerate(ts):
            ring[i % len(ring)] = t
        segs += [("middle", t) for t in ring if t is not None and t >= cap]
    else:
        kept, entries = _veil_blocks(done // BLOCK)
        segs += [("merge", (kept[slot], BLOCK * b + (BLOCK - 1) // 2)) for slot, b in entries if b > 0]
    return segs


def _veil_blocks(n: int):
    """After n whole blocks: slot -> block whose mean it holds, and the FIFO's
    (slot, block) entries.  An entry that moves down keeps the slot that it
    was finalized into, as the reference's record does."""
    kept, fifo = {}, []
    for b in range(n):
        if len(fifo) == MERGE_CAP:
            fifo = fifo[1:]
        slot = len(fifo)
        fifo.append((slot, b))
        kept[slot] = b
    return kept, fifo


def _groups(case) -> int:
    return ((case["grid_h"] + 1) // 2) * ((case["grid_w"] + 1) // 2)


def _packed(case, labels):
    """Tokens that one layer packs, and the tokens that it holds once each."""
    FS, t0 = _fs(case), case["chunks"] * case["frames"]
    packed = held = pairs = 0
    for label in labels:
        own = set()
        for f in range(case["frames"]):
            segs = _held(case, label, t0 + f, False)
            n = sum(_groups(case) if w == "merge" else FS for w, _ in segs)
            packed += n
            pairs += n * FS
            own |= {(w, t if w != "merge" else t[0]) for w, t in segs}
        held += sum(_groups(case) if w == "merge" else FS for w, _ in own)
    return packed, held, pairs


def work(case):
    kind = case["kind"]
    row = 2 * D * 2  # a token's K and V rows of one head
    if kind in ("step", "commit", "cache"):
        H, FS, n_new = case["heads"], _fs(case), case["frames"] * _fs(case) * case["heads"]
        update = n_new * (row + row + 24)
        if kind == "commit":
            # both passes' K and V in, the FIFO out; the committed FIFO's copy; middle frames and merge sums out
            labels = _labels(case, 1)[0]
            b = 2 * update + 2 * H * MAX_RECENT * FS * (row + 24)
            for label in labels:
                if label == 2:
                    b += 2 * 2 * _groups(case) * D * 4
                else:
                    b += case["frames"] * FS * (row + 24) / (1 if label == -1 else INTERVAL)
            return dict(bytes=float(b), flops=0.0)
        if kind == "step":
            _, held, pairs = _packed(case, _labels(case, 1)[0])
            return dict(bytes=float(update + held * row + 2 * n_new * D * 2), flops=4.0 * pairs * D)
        b = 0
        for labels in _labels(case, case["layers"]):
            packed, held, _ = _packed(case, labels)
            b += update + held * (row + 24) + packed * (row + 24)
        return dict(bytes=float(b), flops=0.0)
    if kind == "attn":
        seqs, mean = case["batches"] * case["heads"], (case["keys_lo"] + case["keys_hi"]) / 2
        return dict(bytes=seqs * (case["rows"] * row + mean * row), flops=4.0 * seqs * case["rows"] * mean * D)
    if kind == "cross":
        H = case["heads"]
        return dict(bytes=float(H * (case["rows"] + case["keys"]) * row), flops=4.0 * H * case["rows"] * case["keys"] * D)
    if kind == "evict":
        H, F, G = case["heads"], case["frames"], _groups(case)
        # frames in, the running sums in and out, finished means out
        return dict(bytes=float(H * (F * _fs(case) * row + 2 * 2 * G * D * 4 + F / BLOCK * G * (row + 24))),
                    flops=float(2 * 2 * H * F * _fs(case) * D))
    if kind == "qk":
        n = case["rows"] * case["heads"]
        return dict(bytes=float(n * (4 * 2 * D + 24)), flops=float(n * D * 12))
    if kind == "residual":
        n = case["rows"] * case["cols"]
        return dict(bytes=float(n * (4 + 4 + 2 + 2)), flops=float(n * 10))
    C, N, T = D * case["heads"], case["frames"] * _fs(case), case["text_len"]
    pairs = sum(_packed(case, l)[2] for l in _labels(case, case["blocks"]))
    weights = case["blocks"] * (6 * C * C + 2 * C * case["ffn"]) + 6 * C * C + 2 * 64 * C
    flops = 2.0 * N * case["blocks"] * (6 * C * C + 2 * C * case["ffn"]) + 4.0 * D * pairs
    flops += case["blocks"] * 4.0 * N * T * C + 4.0 * N * 64 * C
    held = sum(_packed(case, l)[1] for l in _labels(case, case["blocks"]))
    return dict(bytes=float(2 * weights + held * row + case["blocks"] * (N * C * 4 + T * C * 4) + 4 * 64 * N), flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind in ("commit", "evict", "cache"):
        # copies, and bf16 roundings of fp32 sums, means and rotations: in another order of the sums about one
        # value in 30,000 rounds to its neighbour, 2^-8 away at most
        return {"rel": 1e-4, "max": 0.01}
    if kind in ("step", "attn", "cross"):
        return {"rel": 1e-2, "max": 0.1}   # bf16 probabilities and outputs: 2.3e-3 to 2.9e-3 from 64 bits
    if kind == "qk":
        return {"rel": 2e-3, "max": 0.02}  # the norm's bf16 rounding before the rotation, or none
    if kind == "residual":
        return {"rel": 5e-4, "max": 0.01}  # as the first, after an fp32 norm
    return {"rel": 1.5e-2, "max": 0.2}     # bf16 activations through every layer: 3.3e-3 from 64 bits


# ---------------------------------------------------------------------------
# exact: 64-bit restatements
# ---------------------------------------------------------------------------
def _rotate(x: torch.Tensor, t, y, xx) -> torch.Tensor:
    """3D RoPE of rows x [n, 128] (float64) at index vectors t, y, xx [n]: the
    64 pairs split 22 / 21 / 21 over time, height and width."""
    ang = []
    for p, pairs in ((t, 22), (y, 21), (xx, 21)):
        inv = 10000.0 ** (-2.0 * torch.arange(pairs, dtype=torch.float64, device=x.device) / (2 * pairs))
        ang.append(p.double()[:, None] * inv)
    a = torch.cat(ang, dim=1)
    re, im = x[:, 0::2], x[:, 1::2]
    return torch.stack([re * a.cos() - im * a.sin(), re * a.sin() + im * a.cos()], dim=2).reshape(x.shape)


def _softmax_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    p = torch.softmax((q.double() @ k.double().t().contiguous()) * D ** -0.5, dim=1)
    return p @ v.double()


class _Frames:
    """Frames of one layer's rollout by time and head, and their 2x2 means."""

    def __init__(self, case, seed, layer, own=None):
        self.case, self.seed, self.layer, self.chunks = case, seed, layer, {}
        if own is not None:
            self.chunks[case["chunks"]] = own
        tok = torch.arange(_fs(case), device=DEV)
        self.y, self.x = tok // case["grid_w"], tok % case["grid_w"]
        self.cols = (case["grid_w"] + 1) // 2
        self.group = (self.y // 2) * self.cols + self.x // 2
        g = torch.arange(_groups(case), device=DEV)
        self.gy, self.gx = g // self.cols * 2, g % self.cols * 2

    def frame(self, t: int, h: int):
        F, FS = self.case["frames"], _fs(self.case)
        c = t // F
        if c not in self.chunks:
            self.chunks[c] = _chunk(self.case, self.seed, self.layer, c)
        k, v = self.chunks[c]
        s = slice((t % F) * FS, (t % F + 1) * FS)
        return k[s, h].double(), v[s, h].double()

    def mean(self, block: int, h: int):
        n = torch.bincount(self.group, minlength=_groups(self.case)).double() * BLOCK
        out = []
        for part in (0, 1):
            s = torch.zeros(_groups(self.case), D, dtype=torch.float64, device=DEV)
            for t in range(BLOCK * block, BLOCK * (block + 1)):
                s.index_add_(0, self.group, self.frame(t, h)[part])
            out.append(s / n[:, None])
        return out

    def keys(self, label: int, h: int, t_now: int, clean: bool):
        """Rotated K and V of one head for a query frame, in plan order."""
        sync = max(0, t_now - min(max(t_now, 18), 21))
        ks, vs = [], []
        for what, t in _held(self.case, label, t_now, clean):
            if what == "merge":
                k, v = (m.bfloat16().double() for m in self.mean(t[0], h))
                y, x, at = self.gy, self.gx, t[1]
            else:
                k, v = self.frame(t, h)
                y, x, at = self.y, self.x, t if what == "recent" else sync
            ks.append(_rotate(k, torch.full_like(y, at), y, x))
            vs.append(v)
        return torch.cat(ks), torch.cat(vs)

    def recent(self, labels):
        H, FS = self.case["heads"], _fs(self.case)
        k = torch.zeros(1, H, MAX_RECENT, FS, D, dtype=torch.float64, device=DEV)
        v = torch.zeros_like(k)
        seen = (self.case["chunks"] + 1) * self.case["frames"]
        for h, label in enumerate(labels):
            for i, t in enumerate(range(max(SINKS[label], seen - MAX_RECENT), seen)):
                k[0, h, i], v[0, h, i] = self.frame(t, h)
        return k, v


def _attend(case, frames: _Frames, labels, q: torch.Tensor) -> torch.Tensor:
    """q [frames * tokens, heads, D] over each head's held keys, per query frame."""
    F, FS, t0 = case["frames"], _fs(case), case["chunks"] * case["frames"]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for h, label in enumerate(labels):
        for f in range(F):
            k, v = frames.keys(label, h, t0 + f, False)
            out[f * FS:(f + 1) * FS, h] = _softmax_attention(q[f * FS:(f + 1) * FS, h], k, v)
    return out


def _exact_commit(case, seed):
    H, FS, labels, fr = case["heads"], _fs(case), _labels(case, 1)[0], _Frames(case, seed, 0)
    rk, rv = fr.recent(labels)
    mk = torch.zeros(1, H, MAX_MIDDLE, FS, D, dtype=torch.float64, device=DEV)
    mv = torch.zeros_like(mk)
    gk = torch.zeros(1, H, 6, GROUPS, D, dtype=torch.float64, device=DEV)
    gv = torch.zeros_like(gk)
    done = (case["chunks"] + 1) * case["frames"]
    for h, label in enumerate(labels):
        if label == 2:
            for slot, b in _veil_blocks(done // BLOCK)[0].items():
                gk[0, h, slot, :_groups(case)], gv[0, h, slot, :_groups(case)] = fr.mean(b, h)
            continue
        slots, count = {}, {}
        for t in range(done):
            phase = t % PERIOD
            if label == 1 and phase:
                continue
            i = count.get(phase, 0)
            slots[phase * BUCKET + i % BUCKET if label == -1 else i % RING] = t
            count[phase] = i + 1
        for slot, t in slots.items():
            mk[0, h, slot], mv[0, h, slot] = fr.frame(t, h)
    return dict(recent_k=rk, recent_v=rv, recent_pos=None, middle_k=mk, middle_v=mv, middle_pos=None, merge_k=gk,
                merge_v=gv, merge_pos=None, states=None, valid=None)


def _exact_evict(case, seed):
    H, F, G = case["heads"], case["frames"], _groups(case)
    k, v, w = _evict_inputs(case, seed)
    tok = torch.arange(_fs(case), device=DEV)
    group = tok // case["grid_w"] // 2 * ((case["grid_w"] + 1) // 2) + tok % case["grid_w"] // 2
    n = torch.bincount(group, minlength=G).double()[:, None]
    sums = torch.zeros(2, H, 2, GROUPS, D, dtype=torch.float64, device=DEV)
    means = torch.zeros(2, H, 6, GROUPS, D, dtype=torch.float64, device=DEV)
    active, wsum, count, finished = [None, None], [0.0, 0.0], [0, 0], 0
    for f in range(F):
        b = (f + 1) // BLOCK
        if b in active:
            a = active.index(b)
        else:
            a = active.index(None) if None in active else 0
            active[a], wsum[a], count[a] = b, 0.0, 0
            sums[:, :, a] = 0
        for i, x in enumerate((k, v)):
            s = torch.zeros(H, G, D, dtype=torch.float64, device=DEV)
            sums[i, :, a, :G] += s.index_add_(1, group, x[f].double() * float(w[f]))
        wsum[a] += float(w[f])
        count[a] += 1
        if count[a] == BLOCK:
            means[:, :, min(finished, 5), :G] = sums[:, :, a, :G] / (n * wsum[a])
            finished += 1
            active[a], count[a] = None, 0
    return dict(merge_k=means[0], merge_v=means[1], merge_pos=None, merge_count=None, sum_k=sums[0], sum_v=sums[1],
                states=None, desc=None)


def _rms(x, w=None):
    y = x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6)
    return y if w is None else y * w.double()


def _norm(x, mul=None, add=None):
    y = x - x.mean(1, keepdim=True)
    y = y * torch.rsqrt(y.square().mean(1, keepdim=True) + 1e-6)
    return y if mul is None else y * (1 + mul.double()) + add.double()


def _exact_dit(case, seed):
    """The forward in 64 bits on the model's random weights, drawn in the
    order in which the model draws them (biases are 0, norm weights 1)."""
    C, H, N, FS = D * case["heads"], case["heads"], case["frames"] * _fs(case), _fs(case)
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    lin = lambda i, o: (torch.randn(o, i, generator=g, device=DEV) * 0.02).to(torch.bfloat16).double().t().contiguous()
    gelu = lambda x: torch.nn.functional.gelu(x, approximate="tanh")
    text, latent = _dit_inputs(case, seed)
    w_patch, w_t0, w_t1, w_tproj = lin(64, C), lin(256, C), lin(C, C), lin(C, 6 * C)
    w_c0, w_c1 = lin(case["text_dim"], C), lin(C, C)
    blocks = []
    for _ in range(case["blocks"]):
        b = dict(mod=torch.randn(6, C, generator=g, device=DEV) / C ** 0.5)
        for name in ("q", "k", "v", "o", "cq", "ck", "cv", "co"):
            b[name] = lin(C, C)
        b["up"], b["down"] = lin(C, case["ffn"]), lin(case["ffn"], C)
        blocks.append(b)
    head_mod = torch.randn(2, C, generator=g, device=DEV) / C ** 0.5
    w_head = lin(C, 64)
    silu = torch.nn.functional.silu
    gh, gw, F = case["grid_h"], case["grid_w"], case["frames"]
    x = latent.double().view(16, F, gh, 2, gw, 2).permute(1, 2, 4, 0, 3, 5).reshape(N, 64) @ w_patch
    ang = 500.0 * 10000.0 ** (-torch.arange(128, dtype=torch.float64, device=DEV) / 128)
    e = silu(torch.cat([ang.cos(), ang.sin()])[None] @ w_t0) @ w_t1
    e0 = (silu(e) @ w_tproj).view(6, C)
    ctx = gelu(text.double() @ w_c0) @ w_c1
    tok = torch.arange(N, device=DEV)
    t0 = case["chunks"] * F
    qt, qy, qx = (p.repeat_interleave(H) for p in (t0 + tok // FS, tok % FS // gw, tok % gw))
    labels = _labels(case, case["blocks"])
    for l, b in enumerate(blocks):
        m = b["mod"].double() + e0
        xn = _norm(x, m[1], m[0])
        q = _rotate(_rms(xn @ b["q"]).reshape(N * H, D), qt, qy, qx).view(N, H, D)
        k, v = _rms(xn @ b["k"]).view(N, H, D), (xn @ b["v"]).view(N, H, D)
        y = _attend(case, _Frames(case, seed, l, own=(k, v)), labels[l], q)
        x = x + (y.reshape(N, C) @ b["o"]) * m[2]
        qc = _rms(_norm(x) @ b["cq"]).view(N, H, D)
        kc, vc = _rms(ctx @ b["ck"]).view(-1, H, D), (ctx @ b["cv"]).view(-1, H, D)
        y = torch.stack([_softmax_attention(qc[:, h], kc[:, h], vc[:, h]) for h in range(H)], dim=1)
        x = x + y.reshape(N, C) @ b["co"]
        x = x + (gelu(_norm(x, m[4], m[3]) @ b["up"]) @ b["down"]) * m[5]
    hm = head_mod.double() + e
    out = _norm(x, hm[1], hm[0]) @ w_head
    return out.view(F, gh, gw, 16, 2, 2).permute(3, 0, 1, 4, 2, 5).reshape(latent.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        labels, fr = _labels(case, 1)[0], _Frames(case, seed, 0)
        k, v = fr.recent(labels)
        out = _attend(case, fr, labels, _queries(case, seed)[0])
        return dict(out=out[None], recent_k=k, recent_v=v, recent_pos=None)
    if kind == "commit":
        return _exact_commit(case, seed)
    if kind == "cache":
        last = case["layers"] - 1
        labels, fr = _labels(case, case["layers"])[last], _Frames(case, seed, last)
        t0 = case["chunks"] * case["frames"]
        kv = [fr.keys(label, h, t0 + f, False) for f in range(case["frames"]) for h, label in enumerate(labels)]
        return dict(k=torch.cat([k for k, _ in kv]), v=torch.cat([v for _, v in kv]), pos=None, cu=None,
                    recent_k=None, recent_v=None)
    if kind == "attn":
        q, k, v, lens = _attn_inputs(case, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        at, R = 0, case["rows"]
        for i, n in enumerate(lens):
            b, h = divmod(i, case["heads"])
            out[b * R:(b + 1) * R, h] = _softmax_attention(q[b * R:(b + 1) * R, h], k[at:at + n], v[at:at + n])
            at += n
        return out
    if kind == "cross":
        q, k, v = _cross_inputs(case, seed)
        return torch.stack([_softmax_attention(q[:, h], k[:, h], v[:, h]) for h in range(case["heads"])], dim=1)
    if kind == "evict":
        return _exact_evict(case, seed)
    if kind == "qk":
        qkv, wq, wk, pos = _qk_inputs(case, seed)
        C = D * case["heads"]
        q = _rms(qkv[:, :C].double(), wq).reshape(-1, D)
        return dict(q=_rotate(q, pos[:, 0], pos[:, 1], pos[:, 2]), k=_rms(qkv[:, C:2 * C].double(), wk))
    if kind == "residual":
        x, y, gate, mul, add = _residual_inputs(case, seed)
        x = x.double() + y.double() * gate.double()
        return dict(x=x, out=_norm(x, mul, add))
    return dict(velocity=_exact_dit(case, seed), recent_k=None, recent_v=None)
