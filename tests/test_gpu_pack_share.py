"""MegaCache.attend's pack reads a segment that several query chunks hold
once (the plan's list, pkv_plan_pack_list): its flat K / V / positions and
offsets against the reference's op sequence (mega_plan_multi, layer offset,
pyramidkv_pack), which packs every chunk's segments by themselves, bit for bit
on the same cache, after noisy and clean passes."""
from __future__ import annotations

import pytest
import torch

if torch.cuda.is_available():
    from gpu_util import DEV

pytestmark = pytest.mark.gpu


# chunks below, at and past the four that share a read; two groups of them; more
# (chunk, head) pairs than the plan lists; head_dims with their own kernel and
# without; frames of a few tokens and of several 32-token tiles with a remainder
@pytest.mark.parametrize("chunks,heads,D,grid", [(1, 3, 128, (6, 9)), (2, 4, 128, (8, 16)), (4, 3, 64, (7, 9)),
                                                 (6, 3, 128, (3, 5)), (6, 12, 128, (8, 8)), (3, 5, 40, (11, 13)),
                                                 # the least tokens that are listed, and one token fewer per head
                                                 (4, 3, 64, (18, 19)), (4, 3, 64, (11, 31)), (6, 2, 128, (24, 32)),
                                                 (3, 4, 40, (12, 16)), (1, 13, 128, (15, 21)), (1, 16, 128, (16, 16))])
def test_shared_segments_pack_as_each_chunk_by_itself(chunks, heads, D, grid):
    from pyramidkv import factory
    from pyramidkv._mega_cache import build_mega_caches
    from pyramidkv.rope import wan_freqs
    FS, L, F = grid[0] * grid[1], 2, 3
    labels = [[(-1, 1, 2)[(h + l) % 3] for h in range(heads)] for l in range(L)]
    caches = build_mega_caches(L, heads, D, FS, 3, 24, 4, factory.shipped_compositions(L, heads, labels=labels),
                               max_attend_chunks=chunks + 8, device=DEV, freqs=wan_freqs(D), spatial_width=grid[1],
                               spatial_height=grid[0], **factory.PYRAMID_FORCING_REMAP)
    g = torch.Generator(device=DEV)
    g.manual_seed(chunks * 100 + heads)
    mgr = caches[0].ctx.mgr
    print(f"pack share: {chunks} chunks, {heads} heads of {D}, {FS} tokens", flush=True)
    for blk in range(9):
        for mode in ("noisy", "clean"):
            for cache in caches:
                k, v = (torch.randn(1, F * FS, heads, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
                cache.update(k, v, blk * F * FS, cache_update_mode=mode)
            if blk not in (0, 1, 8):
                continue
            for cache in caches:
                start = blk * F * FS
                cu = cache.attend_kv(start, chunks).clone()
                n = int(cu[-1])
                got = [t[:n].clone() for t in (mgr.k_flat_out(), mgr.v_flat_out(), mgr.pos_flat_out())]
                for t in (mgr.k_flat_out(), mgr.v_flat_out(), mgr.pos_flat_out()):
                    t[:n].zero_()
                want_cu = cache.pack(cache.plan(start, chunks))
                assert torch.equal(cu, want_cu)
                for name, a, b in zip(("k", "v", "pos"), got,
                                      (mgr.k_flat_out(), mgr.v_flat_out(), mgr.pos_flat_out())):
                    assert torch.equal(a.view(torch.int16) if a.dtype == torch.bfloat16 else a,
                                       b[:n].view(torch.int16) if b.dtype == torch.bfloat16 else b[:n]), (blk, mode, name)
