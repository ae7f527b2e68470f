"""The C-ABI library loads on the CPU and exports every symbol the header declares."""

from __future__ import annotations

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "aoto_hip.h")


def _declared() -> list[str]:
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(aoto_hip_\w+)\s*\(", text)))


def test_header_declares_entry_points():
    names = _declared()
    assert "aoto_hip_w4_gemv" in names and "aoto_hip_load_code_object" in names


def test_library_exports_every_declared_symbol():
    from aotolith_amd import _lib

    lib = _lib.library()
    for name in _declared():
        assert hasattr(lib, name), name
        assert name in _lib.SIGNATURES, f"{name} has no ctypes signature"
    assert lib.aoto_hip_abi_version() == 19


def test_no_code_object_without_a_gpu():
    from aotolith_amd import _lib

    # No HIP device here: the loaded-check must say "not loaded" rather than crash.
    assert _lib.library().aoto_hip_code_object_loaded() == 0


def test_code_object_is_built_for_gfx950():
    from aotolith_amd import _lib

    image = _lib.default_code_object()
    assert image[:4] == b"\x7fELF"
    assert b"gfx950" in image


def test_launcher_rejects_bad_arguments_on_the_host():
    from aotolith_amd import _lib

    lib = _lib.library()
    status = lib.aoto_hip_w4_gemv(None, None, None, None, None, None, 0.0, None, 1.0, 1.0, None,
                                  896, 896, 64, 0, None)
    assert status == _lib.AOTO_ERR_ARGUMENT
    assert "null pointer" in _lib.last_error()


def test_wide_plan_matches_the_workspace_queries():
    """ops.wide_plan (the Python mirror of the automatic plan's rule) agrees with what the
    C ABI's workspace queries size: from ops.WIDE_ROWS rows (K % 256 == 0) a split plan
    needs splits * M * N f32 partials (twice that for the gate/up pair), an unsplit one
    none - host logic only, no device call."""

    from aotolith_amd import _lib, ops

    lib = _lib.library()
    seen = set()
    for m in (512, 640, 1024, 1100, 2048, 4096):
        assert ops.wide_plan(m, 896, 896) is None  # K % 256 != 0: the 16x16 kernel's plan
        for n, k in ((4096, 4096), (1152, 1024), (6144, 4096), (4096, 14336), (14336, 4096), (640, 2048),
                     (768, 512)):
            plan = ops.wide_plan(m, n, k)
            assert plan is not None, (m, n, k)
            tile, splits = plan
            seen.add(tile)
            want = splits * m * n * 4 if splits > 1 else 0
            assert ops.gemm_workspace_bytes(m, n, k) == want, (m, n, k, plan)
            ptile, psplits = ops.wide_plan(m, n, k, paired=True)
            assert ptile == 241
            assert ops.gate_up_workspace_bytes(m, n, k) == (2 * psplits * m * n * 4 if psplits > 1 else 0), (m, n, k)
        for hq, hkv, d, k in ((32, 8, 128, 4096), (8, 2, 128, 2048), (28, 4, 128, 3584)):
            n = (hq + 2 * hkv) * d
            tile, splits = ops.wide_plan(m, n, k)
            got = lib.aoto_hip_w4_gemm_qkv_rope_workspace(m, k, 0, 0, hq, hkv, d)
            assert got == (splits * m * n * 4 if splits > 1 else 0), (m, hq, k)
    assert seen == {241, 243, 441}, seen
    # below the wide rows, or K % 256 != 0, the 16x16 kernel's plan (no wide plan)
    assert ops.wide_plan(511, 4096, 4096) is None and ops.wide_plan(2048, 896, 896) is None
    # explicit codes are taken as given
    assert ops.gemm_workspace_bytes(2048, 4096, 4096, 28, 1) == 0
    assert ops.gemm_workspace_bytes(2048, 4096, 4096, 441, 2) == 2 * 2048 * 4096 * 4


def test_lds_plan_takes_the_full_rounds_at_long_prompts():
    """ops.lds_plan (the Python mirror of the C ABI's choice of the dequant-once kernel):
    at 2048 rows the Llama-3-8B o, down and paired gate/up projections (256 / 256 / 1792
    blocks: whole rounds of 256) take it, and q/k/v on 192-column blocks (384 blocks of 128
    columns would be 1.5 rounds, 256 of 192 are one); 1024-row o / down grids (128 blocks),
    8-bit codes, gate epilogues and odd group counts do not; at 32-256 rows the paired
    gate/up takes the 128-row forms (64 + 64 columns where that gives 128 blocks, else 32 +
    32 within one round), and single projections with K >= 2048 its split-K form, whose
    partials the automatic workspace query covers; its unsplit tiles need no split-K
    workspace - host logic only."""

    from aotolith_amd import ops

    assert ops.lds_plan(2048, 4096, 4096) == ops.LDS_TILE
    assert ops.lds_plan(2048, 4096, 14336) == ops.LDS_TILE
    assert ops.lds_plan(2048, 14336, 4096, paired=True) == ops.LDS_PAIRED_TILE
    assert ops.lds_plan(2048, 6144, 4096) == ops.LDS_WIDE_TILE
    assert ops.lds_plan(2048, 5120, 4096) is None  # 20 x 8 = 160 blocks of 256 x 128 columns
    assert ops.lds_plan(1024, 4096, 4096) is None and ops.lds_plan(1024, 14336, 4096, paired=True) is None
    assert ops.lds_plan(4096, 4096, 4096) == ops.LDS_TILE
    assert ops.lds_plan(2048, 4096, 4096, bits=8) is None
    assert ops.lds_plan(2048, 4096, 4096, gate=True) is None
    assert ops.lds_plan(2048, 4096, 4096 - 64, group_size=64) is None  # 63 groups per row
    assert ops.lds_plan(2048, 4096, 4096, group_size=96) is None
    # short prompts: the paired gate/up only, 128-row blocks
    assert ops.lds_plan(128, 4864, 896, paired=True) == ops.LDS_SHORT_NARROW_TILE  # 152 blocks of 32 + 32
    assert ops.lds_plan(64, 4864, 896, paired=True) == ops.LDS_SHORT_NARROW_TILE
    assert ops.lds_plan(256, 4864, 896, paired=True) == ops.LDS_SHORT_PAIRED_TILE  # 2 x 76 blocks of 64 + 64
    assert ops.lds_plan(128, 14336, 4096, paired=True) == ops.LDS_SHORT_PAIRED_TILE  # 224 blocks
    assert ops.lds_plan(64, 14336, 4096, paired=True) is None  # 448 blocks of 32 + 32: more than a round
    assert ops.lds_plan(16, 4864, 896, paired=True) is None and ops.lds_plan(300, 4864, 896, paired=True) is None
    assert ops.lds_plan(128, 4864, 896, paired=True, bits=8) is None
    # short prompts, single projections with K >= 2048 and no RoPE: the split-K form
    assert ops.lds_plan(128, 896, 4864) == ops.LDS_SPLIT_NARROW_TILE  # 28 column blocks of 32
    assert ops.lds_plan(128, 4096, 4096) == ops.LDS_SPLIT_TILE  # 64 column blocks of 64
    assert ops.lds_plan(128, 896, 896) is None and ops.lds_plan(128, 4864, 896) is None  # K < 2048
    assert ops.lds_plan(128, 6144, 4096, rope=True) is None and ops.lds_plan(16, 896, 4864) is None
    # the automatic workspace covers the split plan: 232 / 28 -> 8 slices of 10 steps (76 in all)
    assert ops.gemm_workspace_bytes(128, 896, 4864) == 8 * 128 * 896 * 4
    assert ops.gemm_workspace_bytes(128, 896, 4864, ops.LDS_SPLIT_NARROW_TILE, 1) == 128 * 896 * 4
    for tile in (ops.LDS_TILE, ops.LDS_WIDE_TILE, ops.LDS_PAIRED_TILE):
        assert ops.gemm_workspace_bytes(2048, 4096, 4096, tile, 0) == 0
        assert ops.gate_up_workspace_bytes(2048, 4096, 4096, tile, 0) == 0


def test_unload_is_refused_while_captured_graphs_are_held():
    """Host logic only: with a captured graph held, aoto_hip_unload_code_object refuses
    before touching any device (its modules would back the graph's kernel handles); a
    release below zero is refused; after the release the unload no longer names graphs."""

    from aotolith_amd import _lib

    lib = _lib.library()
    assert lib.aoto_hip_graph_holds() == 0
    assert lib.aoto_hip_hold_graphs(1) == _lib.AOTO_OK
    try:
        assert lib.aoto_hip_graph_holds() == 1
        assert lib.aoto_hip_unload_code_object() == _lib.AOTO_ERR_ARGUMENT
        assert "captured graphs still launch kernels" in _lib.last_error()
    finally:
        assert lib.aoto_hip_hold_graphs(-1) == _lib.AOTO_OK
    assert lib.aoto_hip_hold_graphs(-1) == _lib.AOTO_ERR_ARGUMENT
    assert lib.aoto_hip_graph_holds() == 0
    lib.aoto_hip_unload_code_object()  # no GPU here: a device error at most, never the graph refusal
    assert "captured graphs" not in _lib.last_error()


def test_hold_graph_is_released_when_the_graph_is_collected():
    import gc

    from aotolith_amd import _lib

    class Graph:  # stands in for torch.cuda.CUDAGraph (no GPU here)
        pass

    lib = _lib.library()
    graph = Graph()
    _lib.hold_graph(graph)
    assert lib.aoto_hip_graph_holds() == 1
    del graph
    gc.collect()
    assert lib.aoto_hip_graph_holds() == 0


def test_tiles_that_read_scale_pairs_refuse_scales_at_an_odd_element():
    """The dequant-once and wide kernels load scales as aligned 32-bit pairs: an explicit code with a base that is only
    2-byte aligned is an argument error before anything is launched (the addresses here are never read)."""

    from aotolith_amd import _lib, ops

    lib = _lib.library()
    at = 1 << 20
    for entry, tiles in ((lib.aoto_hip_w4_gemm, (241, 242, 243, 281, 441, 813, 814, 815, 822, 823, 825)),
                         (lib.aoto_hip_w8_gemm, (241, 242, 441, 833, 834, 845))):
        for tile in tiles:
            status = entry(at, at, at + 2, None, None, None, at, 256, 1024, 1024, 64, tile, 1, at, None)
            assert status == _lib.AOTO_ERR_ARGUMENT and "4-byte aligned" in _lib.last_error(), tile
    for tile in (ops.LDS_PAIRED_TILE, 811, 812, 241):
        for gate, up in ((at + 2, at), (at, at + 2)):
            status = lib.aoto_hip_w4_gemm_gate_up(at, at, gate, at, up, at, 256, 1024, 1024, 64, tile, 1, at, None)
            assert status == _lib.AOTO_ERR_ARGUMENT and "4-byte aligned" in _lib.last_error(), tile


def test_modelled_workspaces_are_what_a_plan_takes_and_at_most_32_mib():
    """The cost model's share of the automatic workspace queries: whole f32 copies of a plan it leads to, never past
    32 MiB, and nothing for shapes it leaves alone (more than 8M outputs in one copy, or N > K up to 256 rows) -
    beyond what the 16x16 kernel's own plan takes (from 129 rows that of tile 28) and the short prompts' split form."""

    from aotolith_amd import _lib, ops

    lib = _lib.library()
    for m, n, k in ((1024, 151936, 896), (2048, 4864, 896), (256, 151936, 896), (256, 8192, 896), (129, 16384, 640)):
        assert ops.gemm_workspace_bytes(m, n, k) == 0, (m, n, k)
        assert ops.gate_up_workspace_bytes(m, n, k) == 0, (m, n, k)
    modelled = 0
    for m in (129, 200, 256, 300, 333, 511, 700, 1030, 1900):
        for n in (128, 896, 1152, 2560, 4096, 6144, 11008, 14336, 28672, 151936):
            for k in (448, 896, 1088, 2048, 4096, 4864, 14336):
                fixed = max(ops.gemm_workspace_bytes(m, n, k, 28, 0), ops.gemm_workspace_bytes(m, n, k, 813, 0),
                            ops.gemm_workspace_bytes(m, n, k, 814, 0)) if m <= 256 else \
                    ops.gemm_workspace_bytes(m, n, k, 28, 0)
                if ops.wide_plan(m, n, k) is not None:
                    continue
                need = ops.gemm_workspace_bytes(m, n, k)
                assert need % (m * n * 4) == 0 and need <= max(fixed, 32 << 20), (m, n, k, need)
                modelled += need > fixed
                pair = ops.gate_up_workspace_bytes(m, n, k)
                fixed = ops.gate_up_workspace_bytes(m, n, k, 18, 0)
                assert pair % (2 * m * n * 4) == 0 and pair <= max(fixed, 32 << 20), (m, n, k, pair)
                rope = lib.aoto_hip_w4_gemm_qkv_rope_workspace(m, k, 0, 0, n // 64 - 2, 1, 64) if n >= 192 else 0
                fixed = ops.gemm_workspace_bytes(m, n, k, 28, 0)
                assert rope % (m * n // 64 * 64 * 4) == 0 and rope <= max(fixed, 32 << 20, need), (m, n, k, rope)
    assert modelled > 20  # (the model does add plans that need one)
