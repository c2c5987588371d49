"""The C-ABI library: it loads and exports every symbol the header declares.

No device work happens here: only calls that fail argument validation before
touching the HIP runtime, and the version query.
"""

from __future__ import annotations

import ctypes
import re
from pathlib import Path

import pytest
import torch

from dexter_amd.ops.gfx950 import _lib

from _util import (DECODE, DUAL, F32_EIGHT, F32_FOUR, F32_PAIR, GENERAL, PAIRED, SINGLE, WAVE, WIDE,
                   attention_kernel)

HEADER = Path(__file__).resolve().parents[1] / "include" / "dexter_gfx950.h"


def declared_functions() -> list[str]:
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(dx_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_path():
    names = declared_functions()
    for want in ("dx_qk_norm_rope", "dx_qk_norm_rope_append", "dx_kv_append",
                 "dx_blockwise_causal_attention", "dx_blockwise_causal_attention_varlen",
                 "dx_attention_workspace_bytes", "dx_last_error", "dx_abi_version",
                 "dx_adaln_modulate", "dx_gated_residual"):
        assert want in names


def test_library_exports_every_declared_symbol(built_lib):
    lib = ctypes.CDLL(str(built_lib))
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, f"not exported: {missing}"


def test_library_resolves_all_of_its_own_symbols(built_lib):
    """No kernel or stub of the library's own namespace is left undefined (a
    dropped template instantiation links, then fails at load on the GPU box)."""
    import shutil
    import subprocess
    if shutil.which("nm") is None:
        pytest.skip("nm not available")
    out = subprocess.run(["nm", "-D", "--undefined-only", str(built_lib)], capture_output=True,
                         text=True, check=True).stdout
    own = [line.split()[-1] for line in out.splitlines() if "_ZN2dx" in line]
    assert not own, f"undefined: {own}"


def test_product_library_carries_no_phase_stamps(built_lib):
    """The timeline build's readers (and so its stamp code) exist only in the measurement
    library that `build.py --timeline` writes beside this one."""
    lib = ctypes.CDLL(str(built_lib))
    stamped = [n for n in ("dx_timeline_words", "dx_timeline_read", "dx_timeline_clear")
               if hasattr(lib, n)]
    assert not stamped, f"product library exports {stamped}"


def test_loader_binds_exactly_the_header(built_lib):
    assert sorted(_lib.exported_symbols()) == declared_functions()


def test_abi_version(built_lib):
    lib = _lib.load()
    assert lib.dx_abi_version() == _lib.ABI_VERSION
    header_version = int(re.search(r"#define DX_ABI_VERSION (\d+)", HEADER.read_text()).group(1))
    assert header_version == _lib.ABI_VERSION


def test_overflow_is_reported_before_any_launch(built_lib):
    lib = _lib.load()
    rc = lib.dx_kv_append(16, 0, 0, 0, 16, 0, 0, 0, 16, 0, 0, 0, 0,
                          _lib.DX_BF16, 1, 5, 2, 64, 8, 4, None)
    assert rc == _lib.DX_EFULL
    assert lib.dx_last_error().decode() == "KV cache full: 4 + 5 > 8"
    with pytest.raises(RuntimeError, match="KV cache full: 4 \\+ 5 > 8"):
        _lib.check(rc, "kv_append")


def test_bad_arguments_are_rejected(built_lib):
    lib = _lib.load()
    rc = lib.dx_kv_append(16, 0, 0, 0, 16, 0, 0, 0, 16, 0, 0, 0, 0,
                          99, 1, 1, 2, 64, 8, 0, None)
    assert rc == _lib.DX_EINVAL and "dtype" in lib.dx_last_error().decode()
    args = [16, 0, 0, 0] * 3 + [None, 0, 0, 0, 0] + [16, 0, 0, 0]
    # (dtype, B, Lq, Lk, H, Hkv, D, cache_len, starts, starts dtype, n_blocks, causal, scale,
    #  workspace, bytes, stream)
    rc = lib.dx_blockwise_causal_attention(*args, _lib.DX_BF16, 1, 8, 8, 2, 2, 96, 0, None,
                                           _lib.DX_I32, 0, 0, 1.0, None, 0, None)
    assert rc == _lib.DX_EINVAL and "head_dim 96" in lib.dx_last_error().decode()
    # Lk != Lq is cross-attention, defined only without a causal or block mask.
    rc = lib.dx_blockwise_causal_attention(*args, _lib.DX_BF16, 1, 8, 9, 2, 2, 128, 0, None,
                                           _lib.DX_I32, 0, 1, 1.0, None, 0, None)
    assert rc == _lib.DX_EINVAL and "must equal q length" in lib.dx_last_error().decode()
    with pytest.raises(ValueError, match="must equal q length"):
        _lib.check(rc, "attention")
    rc = lib.dx_blockwise_causal_attention(*args, _lib.DX_BF16, 1, 8, 8, 6, 4, 128, 0, None,
                                           _lib.DX_I32, 0, 0, 1.0, None, 0, None)
    assert rc == _lib.DX_EINVAL and "not a multiple" in lib.dx_last_error().decode()
    rc = lib.dx_blockwise_causal_attention(*args, _lib.DX_BF16, 1, 8, 0, 2, 2, 128, 0, None,
                                           _lib.DX_I32, 0, 0, 1.0, None, 0, None)
    assert rc == _lib.DX_EINVAL and "no keys" in lib.dx_last_error().decode()


def test_norm_entry_points_validate_before_any_launch(built_lib):
    lib = _lib.load()
    bf, f32 = _lib.DX_BF16, _lib.DX_F32
    # Empty rows: success, nothing launched (null pointers are never touched).
    assert lib.dx_adaln_modulate(None, 0, 0, bf, None, 0, 0, None, 0, 0, bf,
                                 None, 0, 0, bf, 1, 0, 3072, 1e-6, None) == _lib.DX_OK
    assert lib.dx_gated_residual(None, 0, 0, None, 0, 0, bf, None, 0, 0, bf,
                                 None, 0, 0, bf, 0, 5, 3072, None) == _lib.DX_OK
    rc = lib.dx_adaln_modulate(None, 0, 0, 7, None, 0, 0, None, 0, 0, bf,
                               None, 0, 0, bf, 1, 1, 64, 1e-6, None)
    assert rc == _lib.DX_EINVAL and "dtype codes" in lib.dx_last_error().decode()
    rc = lib.dx_adaln_modulate(None, 0, 0, bf, None, 0, 0, None, 0, 0, f32,
                               None, 0, 0, bf, 1, 1, 64, 1e-6, None)
    assert rc == _lib.DX_EINVAL and "promotion" in lib.dx_last_error().decode()
    rc = lib.dx_gated_residual(None, 0, 0, None, 0, 0, bf, None, 0, 0, bf,
                               None, 0, 0, bf, 1, 1, 1 << 20, None)
    assert rc == _lib.DX_EINVAL and "exceeds" in lib.dx_last_error().decode()
    rc = lib.dx_gated_residual(None, 0, 0, None, 0, 0, bf, None, 0, 0, bf,
                               None, 0, 0, bf, 70000, 1, 64, None)
    assert rc == _lib.DX_EINVAL and "grid limits" in lib.dx_last_error().decode()
    with pytest.raises(ValueError, match="grid limits"):
        _lib.check(rc, "gated_residual")


def test_noalloc_refuses_a_call_beyond_its_scratch_before_any_launch(built_lib):
    """The no-allocation entry point plans first and refuses a call whose
    workspace exceeds the static scratch (64 MiB) without touching memory:
    128 heads x 16 forced splits need ~71 MB of partials."""
    lib = _lib.load()
    h, d, lq, c = 128, 128, 128, 4096
    row = h * d  # [B, L, H, D] contiguous: strides (L*H*D, H*D, D)
    qkv = [16, lq * row, row, d] * 3
    cache = [16, (c + lq) * row, (c + lq) * row, row, d]
    out = [16, lq * row, row, d]
    with _lib.tuning(_lib.TUNE_ATTN_SPLITS, 16):
        need = lib.dx_attention_workspace_bytes(1, lq, lq, h, d, c, None)
        rc = lib.dx_blockwise_causal_attention_noalloc(
            *qkv, *cache, *out, _lib.DX_BF16, 1, lq, lq, h, h, d, c, None, _lib.DX_I32, 0, 0,
            0.088, None)
    assert need > (64 << 20)
    assert rc == _lib.DX_EWORKSPACE
    assert "static scratch" in lib.dx_last_error().decode()


def test_planner_choices_at_the_measured_shapes(built_lib):
    """The launch plans at the benchmark shapes, read back through the workspace
    size (256 KiB of arrival counters, then per partial `rows` f16 values of D
    and a 16-byte record per row). Each split count was chosen by measurement:
    C1 8 splits of 128-row items, C3 3 splits of 256-row items, the C4 ragged
    batch 1/1/2/6 by length, cross-attention onto 257 image keys 5 splits of one
    tile and onto 512 text keys 4 of two; C2 (768 items) has none. Runs without
    a GPU, where the planner assumes MI355X's 256 CUs."""
    lib = _lib.load()
    counters, d = 256 << 10, 128

    def ws(partials, rows):
        return counters + partials * rows * (2 * d + 16)

    assert lib.dx_attention_workspace_bytes(1, 83, 83, 24, d, 1245, None) == ws(24 * 8, 128)
    assert lib.dx_attention_workspace_bytes(1, 8192, 8192, 24, d, 0, None) == 0
    assert lib.dx_attention_workspace_bytes(1, 913, 913, 40, d, 7304, None) == ws(40 * 4 * 3, 256)
    lens = (ctypes.c_int64 * 4)(0, 332, 1245, 3237)
    assert lib.dx_attention_workspace_bytes(4, 99, 99, 24, d, 0, lens) == ws(24 * (1 + 1 + 2 + 6), 128)
    assert lib.dx_attention_workspace_bytes(1, 83, 257, 24, d, 0, None) == ws(24 * 5, 128)
    assert lib.dx_attention_workspace_bytes(1, 83, 512, 24, d, 0, None) == ws(24 * 4, 128)


def test_general_kernel_plan(built_lib):
    """fp32 inputs and head dims 16, 32, 256 run on the general kernel, whose
    workspace is the counter region (never written by it) and then, per split
    of each 64-query item, 64 rows of D fp32 values and an 8-byte {m, l}
    record. About two items per CU (256 CUs without a GPU), at least two
    32-key tiles per split; none when the items alone fill the chip. The
    workspace query takes no dtype: at head dims 64 and 128 it reports the
    16-bit kernels' bytes, within which fp32 calls lower their split count."""
    lib = _lib.load()
    counters = 256 << 10

    def ws(items, d):
        return counters + items * 64 * (4 * d + 8)

    # 83 queries x 24 heads: 48 items, 512 // 48 = 10 splits over 42 tiles.
    assert lib.dx_attention_workspace_bytes(1, 83, 83, 24, 256, 1245, None) == ws(48 * 10, 256)
    assert lib.dx_attention_workspace_bytes(1, 83, 83, 24, 32, 1245, None) == ws(48 * 10, 32)
    # Few keys: at most one split per two tiles (40 keys: 2 tiles, 1 split).
    assert lib.dx_attention_workspace_bytes(1, 20, 20, 2, 16, 20, None) == 0
    # 3,072 items: no split.
    assert lib.dx_attention_workspace_bytes(1, 8192, 8192, 24, 32, 0, None) == 0
    lens = (ctypes.c_int64 * 2)(100, 3000)
    assert lib.dx_attention_workspace_bytes(2, 16, 16, 4, 256, 0, lens) == ws(8 * 16, 256)
    assert lib.dx_attention_workspace_bytes(1, 8, 8, 2, 96, 0, None) < 0
    # Dtype codes other than bf16, f16 and f32 are refused before any launch.
    args = [16, 0, 0, 0] * 3 + [None, 0, 0, 0, 0] + [16, 0, 0, 0]
    rc = lib.dx_blockwise_causal_attention(*args, 7, 1, 8, 8, 2, 2, 64, 0, None,
                                           _lib.DX_I32, 0, 0, 1.0, None, 0, None)
    assert rc == _lib.DX_EINVAL and "dtype code 7" in lib.dx_last_error().decode()


def test_kernel_choice(built_lib):
    """Which kernel a call takes, by shape and by override (256 CUs without a GPU)."""
    bf, f32 = torch.bfloat16, torch.float32
    assert attention_kernel(bf, 1, 83, 83, 24, 128, 1245) == DUAL
    assert attention_kernel(bf, 1, 8192, 8192, 24, 128, n_blocks=8) == PAIRED
    assert attention_kernel(bf, 1, 300, 300, 16, 128, causal=True) == WAVE
    assert attention_kernel(bf, 1, 2048, 2048, 16, 256) == WIDE
    assert attention_kernel(bf, 1, 83, 83, 24, 32, 1245) == GENERAL
    assert attention_kernel(f32, 1, 332, 332, 24, 128, 996, n_blocks=4) == F32_FOUR
    assert attention_kernel(f32, 1, 83, 83, 24, 16, 1245) == GENERAL
    assert attention_kernel(bf, 4, 99, 99, 24, 128, lens=[0, 332, 1245, 3237], n_blocks=2) == DUAL
    assert attention_kernel(bf, 1, 0, 0, 16, 256) == 0
    assert attention_kernel(bf, 1, 8, 8, 2, 96) < 0 and attention_kernel(bf, 1, 8, 8, 2, 64, -1) < 0
    for kernel in range(SINGLE, F32_PAIR + 1):
        with _lib.tuning(_lib.TUNE_ATTN_KERNEL, kernel):
            # An override of one class of calls leaves the other's choice alone.
            mine = attention_kernel(bf, 1, 83, 83, 24, 128, 1245)
            assert mine == (kernel if kernel <= WAVE else DUAL)
            wide = attention_kernel(bf, 1, 2048, 2048, 16, 256)
            assert wide == (GENERAL if kernel == GENERAL else WIDE)
            fp32 = attention_kernel(f32, 1, 332, 332, 24, 128, 996, n_blocks=4)
            assert fp32 == (kernel if kernel in (GENERAL, F32_EIGHT, F32_PAIR) else F32_FOUR)


def test_query_rows_past_a_descriptor(built_lib):
    """Kernels that fetch a work item's query rows through one buffer descriptor (2^31 bytes)
    take every call whose items fit it, however long q is, and no other."""
    bf = torch.bfloat16
    last = (2**30 - 1 - 256) // 127  # row stride at which 128 rows of 256 still fit
    assert attention_kernel(bf, 1, 131136, 128, 64, 256) == WIDE
    assert attention_kernel(bf, 1, 4096, 128, 64, 256, q_sl=last) == WIDE
    assert attention_kernel(bf, 1, 4096, 128, 64, 256, q_sl=last + 1) == GENERAL
    assert attention_kernel(bf, 1, 4096, 128, 64, 256, q_sl=2**40) == GENERAL
    assert attention_kernel(bf, 1, 4096, 128, 64, 256, q_sl=-256) == GENERAL
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, WIDE):
        assert attention_kernel(bf, 1, 128, 32, 64, 256, q_sl=last + 1) == GENERAL
        assert attention_kernel(bf, 512, 1, 32, 64, 256, q_sl=2**40) == WIDE  # one row: no stride
    last = (2**30 - 1 - 128) // 31
    assert attention_kernel(bf, 1, 300, 300, 16, 128, causal=True, q_sl=last) == WAVE
    assert attention_kernel(bf, 1, 300, 300, 16, 128, causal=True, q_sl=last + 1) == DUAL
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, WAVE):  # forced, it falls back to the same plan
        assert attention_kernel(bf, 1, 300, 300, 16, 128, causal=True, q_sl=last + 1) == DUAL
    last = (2**30 - 1 - 128) // 255
    assert attention_kernel(bf, 1, 262272, 64, 64, 128) == PAIRED
    assert attention_kernel(bf, 1, 300, 1000, 48, 128, q_sl=last) == PAIRED
    assert attention_kernel(bf, 1, 300, 1000, 48, 128, q_sl=last + 1) == SINGLE
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, DECODE):  # 96 rows
        assert attention_kernel(bf, 1, 300, 1000, 48, 128, q_sl=last + 1) == DECODE
        assert attention_kernel(bf, 1, 300, 1000, 48, 128, q_sl=4 * last) == SINGLE


def test_grids_past_the_launch_limit(built_lib):
    """A launch holds less than 2^32 threads: calls whose finer work items pass that stay on the
    general kernel, which has fewer of them."""
    f32, bf = torch.float32, torch.bfloat16
    assert attention_kernel(f32, 1, 2**23 - 32, 2048, 64, 32) == F32_PAIR
    assert attention_kernel(f32, 1, 2**23, 2048, 64, 32) == GENERAL
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, WIDE):
        assert attention_kernel(bf, 1 << 10, 1, 32, (1 << 13) - 1, 256) == WIDE
        assert attention_kernel(bf, 1 << 10, 1, 32, 1 << 13, 256) == GENERAL
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, WAVE):
        assert attention_kernel(bf, 1 << 11, 1, 32, (1 << 13) - 1, 128) == WAVE
        assert attention_kernel(bf, 1 << 11, 1, 32, 1 << 13, 128) != WAVE


def test_head_dim_256_choice_counts_items_and_rounds(built_lib):
    """Batches of short queries stay on the general kernel, whose items hold 64 queries, also past
    one 128-query item per CU; prefill-shaped calls go to the 128-query kernel (both measured)."""
    bf = torch.bfloat16
    for b, lq, h, cache in [(8, 64, 16, 8000), (8, 16, 16, 2000), (17, 16, 16, 500),
                            (17, 64, 16, 8000), (12, 64, 24, 2000), (4, 1, 24, 1000),
                            (1, 300, 24, 2000), (32, 64, 16, 500)]:
        assert attention_kernel(bf, b, lq, lq, h, 256, cache) == GENERAL, (b, lq, h, cache)
    for b, lq, h, cache in [(8, 83, 16, 500), (17, 83, 16, 8000), (32, 128, 16, 2000),
                            (1, 400, 16, 0), (1, 2048, 16, 0), (1, 4100, 16, 0), (2, 1000, 24, 0)]:
        assert attention_kernel(bf, b, lq, lq, h, 256, cache) == WIDE, (b, lq, h, cache)
    assert attention_kernel(bf, 1, 1000, 1000, 24, 256, causal=True) == WIDE
    assert attention_kernel(bf, 1, 1000, 1000, 8, 256, causal=True) == GENERAL
    # A ragged batch: its longest sequence's items bound the launch.
    assert attention_kernel(bf, 4, 200, 200, 16, 256, lens=[100, 100, 100, 8000]) == GENERAL
    assert attention_kernel(bf, 4, 200, 200, 16, 256, lens=[500, 400, 500, 600]) == WIDE


def test_fp32_form_leaves_no_empty_query_tile(built_lib):
    """Two query tiles per item past 2.75 16-query items per CU, one where the second is empty."""
    f32 = torch.float32
    assert attention_kernel(f32, 32, 16, 16, 24, 128, 500) == F32_FOUR
    assert attention_kernel(f32, 64, 1, 1, 16, 64, 2000) == F32_FOUR
    assert attention_kernel(f32, 32, 17, 17, 24, 128, 500) == F32_PAIR
    assert attention_kernel(f32, 1, 664, 664, 24, 128) == F32_PAIR
    assert attention_kernel(f32, 1, 16 * 44, 500, 16, 128) == F32_FOUR  # 704 items on 256 CUs
    assert attention_kernel(f32, 1, 16 * 44 + 1, 500, 16, 128) == F32_PAIR


def test_fp32_choice_counts_items_and_rounds(built_lib):
    """Short key ranges, and batches whose 16-query items take more rounds, stay on the general
    kernel; the others go to the fp32 wave split (both measured)."""
    f32 = torch.float32
    for b, lq, lk, h, d, cache in [(4, 300, 64, 24, 128, 0), (1, 4000, 16, 64, 128, 0),
                                   (32, 64, 64, 16, 128, 1000), (32, 40, 40, 16, 64, 4000),
                                   (32, 40, 40, 16, 256, 1000), (1, 1, 1, 24, 64, 1000),
                                   (2, 1, 1, 24, 32, 4000), (1, 83, 83, 24, 128, 4000)]:
        assert attention_kernel(f32, b, lq, lk, h, d, cache) == GENERAL, (b, lq, lk, h, d, cache)
    for b, lq, lk, h, d, cache in [(1, 83, 512, 24, 128, 0), (1, 332, 332, 24, 128, 996),
                                   (1, 400, 400, 24, 128, 500), (1, 2500, 2500, 12, 128, 0),
                                   (32, 16, 16, 24, 128, 2000), (1, 200, 200, 40, 64, 4000),
                                   (17, 40, 40, 16, 32, 1000), (2, 16, 16, 24, 256, 1000)]:
        assert attention_kernel(f32, b, lq, lk, h, d, cache) > GENERAL, (b, lq, lk, h, d, cache)


def test_wave_split_choice_counts_cached_keys_and_rounds(built_lib):
    """A mask makes room for the wave split by the new keys that it hides: not over a long cache,
    and not in batches whose items pass three per CU (both sides measured)."""
    bf = torch.bfloat16
    causal = lambda *a: attention_kernel(bf, *a, causal=True)  # noqa: E731
    blocks = lambda *a: attention_kernel(bf, *a, n_blocks=-(-a[1] // 83))  # noqa: E731
    assert causal(1, 332, 332, 24, 128, 700) == WAVE
    assert causal(1, 332, 332, 24, 128, 1300) == DUAL
    assert causal(1, 1200, 1200, 8, 128, 700) == DUAL
    assert causal(1, 600, 600, 40, 128) == WAVE and causal(1, 600, 600, 40, 128, 300) == PAIRED
    assert causal(2, 300, 300, 24, 128, 500) == WAVE
    assert causal(4, 332, 332, 24, 128) == PAIRED and causal(6, 500, 500, 16, 128) == PAIRED
    assert blocks(4, 332, 332, 24, 128) == PAIRED and blocks(2, 332, 332, 24, 128) == WAVE
    assert blocks(4, 700, 700, 16, 64) == PAIRED and causal(1, 1400, 1400, 24, 64) == WAVE
    ragged = lambda h, d, lens: attention_kernel(bf, len(lens), 99, 99, h, d, lens=lens,  # noqa: E731
                                                 n_blocks=2)
    assert ragged(24, 128, [0, 100, 200, 300]) == WAVE and ragged(40, 128, [0, 100, 200, 300]) == DUAL
    assert ragged(24, 64, [0, 0, 83, 400, 200, 100, 300, 50]) == DUAL
