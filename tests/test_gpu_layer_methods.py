"""MegaCache's calls go through methods of the manager (update_layer,
attend_kv_layer, attend_layer): against the ops they stand for, with the same
state, bit for bit."""
from __future__ import annotations

import pytest
import torch

if torch.cuda.is_available():
    from gpu_util import DEV
    from pyramidkv import _mega_state_ops, _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,layer", [(1, 0), (3, 2)])
def test_methods_equal_ops(layers, layer):
    from pyramidkv import factory
    from pyramidkv._mega_cache import build_mega_caches
    from pyramidkv.rope import wan_freqs
    H, D, W, FS, F = 3, 128, 8, 64, 3
    make = lambda: build_mega_caches(layers, H, D, FS, 3, 24, 4,
                                     factory.shipped_compositions(layers, H, labels=[[-1, 1, 2]] * layers),
                                     device=DEV, freqs=wan_freqs(D), spatial_width=W, spatial_height=FS // W,
                                     **factory.PYRAMID_FORCING_REMAP)[layer]
    a, b = make(), make()
    g = torch.Generator(device=DEV)
    g.manual_seed(layers)
    rnd = lambda: torch.randn(1, F * FS, H, D, generator=g, device=DEV).to(torch.bfloat16)
    ops, ctx = _ops.ops(), b.ctx
    for blk in range(8):
        k, v, q = rnd(), rnd(), rnd()
        a.update(k, v, blk * F * FS, cache_update_mode="clean")
        if ctx.committed_vc is None:
            ctx.committed_vc = ctx.mgr.valid_count().clone()
        ops.cache_update(ctx.mgr, ctx.states_bytes[layer], ctx.sink_caps_per_head[layer], ctx.committed_vc[layer], k, v,
                         layer, blk * F, 1, 0, W, ctx.layer_merge_heads[layer])
        cu = ops.mega_attend_kv(ctx.mgr, ctx.states_bytes[layer], layer, torch.arange(blk * F, blk * F + F),
                                _mega_state_ops._SINK_MODE["window_clamp"], 18, 21, 0, *ctx.freq_parts_flat)
        cu_q = torch.arange(0, F * FS + 1, FS, dtype=torch.int32, device=DEV)
        want = _ops.ragged_attention(q[0], ctx.mgr.k_flat_out().view(-1, D), ctx.mgr.v_flat_out().view(-1, D), cu_q, cu,
                                     FS, max_seqlen_k=ctx.layer_max_keys[layer])
        assert torch.equal(a.attend_kv(blk * F * FS, F), cu)
        assert torch.equal(a.attend(q, blk * F * FS)[0], want)
        for name in ("recent_k_pool", "middle_v_pool", "merge_k_pool", "valid_count", "merge_token_count"):
            assert torch.equal(getattr(a.ctx.mgr, name)(), getattr(ctx.mgr, name)()), (blk, name)
        assert torch.equal(a.ctx.states_bytes, ctx.states_bytes)


# one token of positions more than a 16-byte multiple; a layer whose FIFO starts off one; several workgroups
@pytest.mark.parametrize("layers,heads,D,FS,recent", [(3, 1, 8, 5, 1), (2, 3, 128, 63, 3), (2, 4, 64, 700, 4),
                                                      (3, 1, 24, 341, 1)])
def test_recent_fifo_copy_and_restore(layers, heads, D, FS, recent):
    mgr = torch.classes.adahead.PyramidKVCacheManager(layers, heads, D, FS, 1, 1, recent, DEV, "bfloat16", 1)
    pools = (mgr.recent_k_pool(), mgr.recent_v_pool(), mgr.recent_pos_pool())
    g = torch.Generator(device=DEV)
    g.manual_seed(FS)
    for t in pools:
        t.copy_(torch.randint(-1000, 1000, t.shape, generator=g, device=DEV))
    want = [t.clone() for t in pools]
    for layer in range(layers):
        mine = [torch.zeros_like(t[layer]) for t in pools]
        mgr.recent_fifo_copy(layer, *mine, False)
        assert all(torch.equal(a, t[layer]) for a, t in zip(mine, want))
        for t in pools:
            t[layer].zero_()
        mgr.recent_fifo_copy(layer, *mine, True)
        assert all(torch.equal(a, b) for a, b in zip(pools, want))
