"""The C-ABI library: it loads, exports every entry point include/vortex_hip.h
declares, and rejects bad arguments on the host (these calls return before
any device work, so they run without a GPU)."""
import ctypes
import os
import re

import pytest

from vortex_torch import _hip

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "vortex_hip.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vtx_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _hip.load_library()
    declared = _declared()
    assert len(declared) >= 8
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in vortex_hip.h but not exported"
    assert set(declared) == set(_hip.EXPORTED_SYMBOLS)
    assert lib.vtx_version().startswith(b"vortex-mi355x")


def test_host_side_argument_errors():
    lib = _hip.load_library()
    rc = lib.vtx_plan_decode(None, -1, None, None, 0, None, None, 0, None, None, 0, 0, None, None, None, None,
                             0, None, None, 16, 8, 30, 1, 1, 64, 16, None, 0, 0, None)
    assert rc == -1 and b"batch_size" in lib.vtx_last_error()
    rc = lib.vtx_topk_select(None, 0, None, None, None, 0, None, 0, 1, 5000, 1, 1, 512, None)
    assert rc == -1 and b"exceeds" in lib.vtx_last_error()
    rc = lib.vtx_page_reduce(None, 0, 16, 128, None, 0, 0, None, 5, 8, 16, 3, 0, None)
    assert rc == -1 and b"dim" in lib.vtx_last_error()
    rc = lib.vtx_indexer_fused(None, 0, 2, None, None, None, 0, None, 0, None, None, None, 0, None, 0,
                               4, 30, 1, 1, 512, 100, None, 0, 0, None, 0, None)
    assert rc == -1 and b"head_dim" in lib.vtx_last_error()
    # well-formed (never dereferenced) addresses: the layout checks fail before any device work
    fake = [0x10000 * (i + 1) for i in range(9)]
    args = [fake[0], 4, 2, None, fake[1], fake[2], 100, fake[3], 100, fake[4], fake[5], fake[6], 100,
            fake[7], 100, 4, 30, 1, 1, 512, 128]
    rc = lib.vtx_indexer_fused(*args, None, 0, 7, None, 0, None)
    assert rc == -1 and b"unknown mode" in lib.vtx_last_error()
    rc = lib.vtx_indexer_fused(*args, fake[8], 3, _hip.FUSED_SPLIT, None, 0, None)
    assert rc == -1 and b"segment counters" in lib.vtx_last_error()
    assert lib.vtx_indexer_fused_supported(128) == 1 and lib.vtx_indexer_fused_supported(100) == 0


@pytest.mark.parametrize("types", [[_hip.REDUCE_MEAN], [_hip.REDUCE_MEAN, _hip.REDUCE_MAX],
                                   [_hip.REDUCE_MAX, _hip.REDUCE_MIN],
                                   [_hip.REDUCE_MEAN, _hip.REDUCE_MAX, _hip.REDUCE_MIN, _hip.REDUCE_L2NORM]])
@pytest.mark.parametrize("cols", [64, 128, 256, 512, 576])
def test_page_reduce_sharing_leaves_no_wave_a_queue(cols, types):
    """The workgroups that share a block of 256 loc entries take the tiles it
    closes in one round of what their waves really do at a time (several tiles
    only where the instance's registers fit), or there are sixteen; and sixteen
    while the grid is small, also where a whole page is wider than a block."""
    lib = _hip.load_library()
    rt = (ctypes.c_int32 * len(types))(*types)
    # statistics that the instance accumulates, times the levels of its fold over a wave's row groups
    stats = len(types) if types != [_hip.REDUCE_MAX, _hip.REDUCE_MIN] else 4
    lpr = cols // 8
    fits = lpr <= 64 and 64 % lpr == 0 and {8: 4, 16: 3, 32: 2, 64: 1}[lpr] * stats <= 8
    for page in (1, 8, 16, 17, 32, 256, 512):
        for heads in (1, 2, 3, 8):
            for nnz in (1, 256, 768, 769, 1024, 1025, 4096, 8192, 8193, 65536, 1 << 20):
                share, per = ctypes.c_int32(), ctypes.c_int32()
                assert lib.vtx_page_reduce_sharing(page, cols, len(types), rt, nnz, heads, page, share, per) == 0
                what = (page, heads, nnz, share.value, per.value)
                tiles, blocks = max(1, 256 // page) * heads, -(-nnz // 256)
                assert 1 <= share.value <= 16, what
                assert per.value == 1 or (per.value == 64 // lpr and fits and page <= 16 and blocks >= 4), what
                assert share.value == 16 or share.value * 4 * per.value >= tiles, what
                if blocks <= 32:
                    assert share.value == 16, what


@pytest.mark.parametrize("segments", [1, 170, 171, 200, 256, 257, 304, 341, 342, 511, 512, 600])
@pytest.mark.parametrize("dim", [64, 128, 256, 576])
def test_auto_layout_needs_the_staging_zone_for_four_wave_chunks(segments, dim):
    """On 256 compute units: the four-wave chunks that let AUTO split past two
    segments for three units exist only with the staging zone, so a workspace
    of counters alone, or none, never splits there."""
    lib = _hip.load_library()
    full = lib.vtx_indexer_fused_workspace_len(segments)
    for pages in (16, 512, 513, 600, 1024, 2046, 8192):
        for topk in (16, 32, 33, 64, 65):
            def split(entries):
                rc = lib.vtx_indexer_fused_auto_layout(segments, topk, 1, 1, pages, dim, entries, 256)
                assert rc in (_hip.FUSED_SEGMENT, _hip.FUSED_SPLIT)
                return rc == _hip.FUSED_SPLIT
            what = (segments, pages, topk, dim)
            idle = segments < 512 if dim >= 256 else pages > 512 and 3 * segments < 512
            chunks = -(-(pages - 2) // 256)
            quad = (dim == 128 and pages > 512 and topk <= 64 and chunks <= 16 and segments <= 512
                    and segments * chunks <= 1024 and (segments > 256 or topk > 32))
            assert split(full) == (idle or quad), what
            assert split(segments) == idle, what
            assert not split(segments - 1) and not split(0), what
    assert lib.vtx_indexer_fused_auto_layout(4, 30, 1, 1, 512, 100, 0, 256) == -1


def test_missing_library_fails_loudly(tmp_path):
    with pytest.raises(RuntimeError, match="not found"):
        _hip.load_library(tmp_path / "nope.so")
