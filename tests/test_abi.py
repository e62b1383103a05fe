"""The C-ABI library loads without a GPU and exports every entry point that
include/pyramidkv_hip.h declares; pure host queries answer correctly.  No
compute call is made here."""
import ctypes

from pyramidkv import _abi as A


def test_library_exports_every_declared_symbol():
    lib = A.lib()
    declared = A.declared_symbols()
    assert len(declared) >= 13
    missing = [s for s in declared if not hasattr(lib, s)]
    assert not missing, missing


def test_host_queries():
    lib = A.lib()
    assert lib.pkv_abi_version() == 3
    assert lib.pkv_perhead_state_size() == 600
    g = A.make_geometry(30, 12, 128, 1560, 3, 24, 4, 8 * 12 * 37 * 1560)
    assert lib.pkv_cache_update_workspace_size(ctypes.byref(g), 3) > 8 * 36 * 4
    assert lib.pkv_merge_workspace_size(12, 3, 1560, 420) >= 36 * (1560 + 421) * 4


def test_argument_errors_are_reported_without_touching_the_device():
    lib = A.lib()
    rc = lib.pkv_ragged_attn_fwd(None, None)
    assert rc == A.PKV_ERR_INVALID
    assert b"NULL" in lib.pkv_last_error()
    rc = lib.pkv_plan_multi(None, None, None, None, None, 0, None, None, None, None)
    assert rc == A.PKV_ERR_INVALID


def test_plan_list_size_rule():
    """A list is offered where it pays: one chunk below 4,096 tokens of all
    heads, several from 256 tokens per chunk on, and never past what the plan
    can list."""
    size = lambda heads, fs, chunks: A.lib().pkv_plan_list_size(
        ctypes.byref(A.make_geometry(2, heads, 128, fs, 3, 24, 4, 1 << 20)), chunks)
    segs = 3 + 24 + 4 + 6
    assert size(3, 64, 1) == 64 + 3 * segs * 48 and size(13, 315, 1) > 0 and size(16, 256, 1) == 0
    for chunks in (2, 3, 4):
        assert size(1, 256 * chunks, chunks) == 64 + chunks * segs * 48 and size(1, 256 * chunks - 1, chunks) == 0
    assert size(12, 1560, 3) == 64 + 3 * 12 * segs * 48
    assert size(12, 1560, 5) == 0 and size(20, 1560, 3) == 0 and size(12, 1560, 0) == 0
