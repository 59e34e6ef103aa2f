"""The C-ABI shared library: builds, loads, exports every symbol include/castle_hip.h
declares, and validates arguments on the host (no kernel is launched here)."""
import ctypes
import os
import re

import pytest

from lookahead_keys_attention_amd import _native as N

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "castle_hip.h")


@pytest.fixture(scope="module")
def lib():
    if not N.is_built():
        from lookahead_keys_attention_amd.build import build

        build()
    return N.lib()


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(castle_[a-z_0-9]+)\s*\(", text)))


def test_header_symbols_are_exported(lib):
    names = declared_functions()
    assert sorted(N.EXPORTED_SYMBOLS) == names
    raw = ctypes.CDLL(N.LIB_PATH)
    for name in names:
        assert hasattr(raw, name), f"{name} missing from libcastle_hip.so"


def test_every_native_source_is_built():
    """Nothing lies beside the sources that the build does not read."""
    from lookahead_keys_attention_amd import build as B

    files = set(os.listdir(B.CSRC))
    headers = {f for f in files if f.endswith(".h")}
    assert files - headers == {*B.SOURCES, B.HOST_SOURCE}
    text = "".join(open(os.path.join(B.CSRC, f)).read() for f in files)
    assert headers <= set(re.findall(r'#include "([^"/]+)"', text))


@pytest.mark.parametrize("complaint, again", [("clang (LLVM option parsing): Unknown command line argument '{}'.", True), ("error: no such thing as {}", False)])
def test_a_compiler_without_an_internal_option_builds_all_the_same(monkeypatch, complaint, again):
    from lookahead_keys_attention_amd import build as B

    option, commands = B.VECTOR_RESULTS[1], []

    def run(cmd):
        commands.append(cmd)
        if option in cmd:
            raise RuntimeError(complaint.format(option))
        return ""

    monkeypatch.setattr(B, "_run", run)
    if not again:
        with pytest.raises(RuntimeError):
            B.build(jobs=1)
        return
    B.build(jobs=1)
    for src in (*B.SOURCES, B.HOST_SOURCE):
        tried = [c for c in commands if os.path.join(B.CSRC, src) in c]
        assert option not in tried[-1] and len(tried) == 1 + (src in B.SOURCE_FLAGS)


def test_version_and_error_strings(lib):
    assert lib.castle_abi_version() == 5
    assert lib.castle_error_string(0) == b"ok"
    for code in (-1, -2, -3, -4, -5, -6):
        assert len(lib.castle_error_string(code)) > 3


def test_workspace_sizes(lib):
    # B4 H8 L4096 d64 bf16.  Kept for backward (O(L d)): header + lse + three T arrays (T', T'^T, cross quarter) +
    # six operand copies; state buffer (O(L^2 d / 128)): snapshots, 64 * nblk*(nblk-1)/2 rows per head
    n = lib.castle_fwd_workspace_bytes(4, 8, 4096, 64, 1)
    BH, Lp, nblk = 32, 4096, 64
    header = 256 + 4 * 256   # status / scale header + partial maxima
    snaps = BH * 64 * nblk * (nblk - 1) // 2 * 64 * 2
    assert n == header + BH * Lp * 4 + 3 * BH * Lp * 64 * 2 + 6 * BH * Lp * 64 * 2
    assert lib.castle_fwd_state_bytes(4, 8, 4096, 64, 1) == snaps
    bwd = header + snaps + BH * Lp * 4 + BH * Lp * 64 * 2 + 2 * BH * Lp * Lp * 2
    assert lib.castle_bwd_workspace_bytes(4, 8, 4096, 64, 1, 0) == bwd
    assert lib.castle_bwd_workspace_bytes(4, 8, 4096, 64, 1, N.FLAG_RECOMPUTE_STATE) == bwd + snaps
    assert lib.castle_bwd_workspace_bytes(4, 8, 4096, 64, 1, N.FLAG_RECOMPUTE_SCORES) == bwd - 2 * BH * Lp * Lp * 2
    # fp32 asks for nothing else, with and without its score tiles
    bwd32 = header + 2 * snaps + BH * Lp * 4 + BH * Lp * 64 * 4
    assert lib.castle_fwd_workspace_bytes(4, 8, 4096, 64, 0) == header + BH * Lp * 4 + 3 * BH * Lp * 64 * 4 + 6 * BH * Lp * 64 * 4
    assert lib.castle_bwd_workspace_bytes(4, 8, 4096, 64, 0, 0) == bwd32 + 2 * BH * Lp * Lp * 4
    assert lib.castle_bwd_workspace_bytes(4, 8, 4096, 64, 0, N.FLAG_RECOMPUTE_SCORES) == bwd32
    # ragged L rounds up to 128 rows
    assert lib.castle_fwd_workspace_bytes(1, 1, 129, 64, 0) == lib.castle_fwd_workspace_bytes(1, 1, 256, 64, 0)
    assert lib.castle_decode_workspace_bytes(32, 8, 64, 4096) > 0


def test_state_size_formula_of_the_python_callers_matches_the_library(lib):
    from lookahead_keys_attention_amd import ops

    for B, H, L, d, dtype, es in ((4, 8, 4096, 64, 1, 2), (1, 16, 16384, 128, 1, 2), (2, 2, 100, 32, 0, 4), (1, 1, 129, 16, 2, 2),
                                  (3, 5, 128, 64, 0, 4)):
        assert ops.state_bytes_formula(B, H, L, d, es) == lib.castle_fwd_state_bytes(B, H, L, d, dtype)


def test_rejects_bad_shapes_and_types(lib):
    assert lib.castle_fwd_workspace_bytes(1, 1, 16, 48, 1) == -2      # head dim not supported
    assert lib.castle_fwd_workspace_bytes(1, 1, 16, 128, 0) == -2     # fp32 needs d <= 64
    assert lib.castle_fwd_workspace_bytes(1, 1, 16, 64, 7) == -1      # unknown dtype
    assert lib.castle_fwd_workspace_bytes(0, 1, 16, 64, 1) == -2
    assert lib.castle_decode_workspace_bytes(1, 1, 24, 8) == -2


def test_null_and_misaligned_views_are_rejected_on_the_host(lib):
    ok = N.View4(4096, 64, 64, 64)
    null = N.View4(None, 0, 0, 0)
    odd = N.View4(4098, 64, 64, 64)          # not 16-byte aligned
    bad_stride = N.View4(4096, 64, 64, 3)    # rows not 16-byte aligned
    args = lambda v: ([ok] * 5 + [v], [1, 1, 16, 64, 1, 0.125, 0, ok, null, 4096, 1 << 30, 8192, 1 << 30, None])
    for bad in (null, odd, bad_stride):
        a, b = args(bad)
        assert lib.castle_fwd(*a, *b) == -5
    a, b = args(ok)
    b[9] = None                                # no workspace
    assert lib.castle_fwd(*a, *b) == -4
    b[9], b[10] = 4096, 16                     # too small
    assert lib.castle_fwd(*a, *b) == -4
    b[10], b[11] = 1 << 30, None               # no state buffer
    assert lib.castle_fwd(*a, *b) == -4


def test_no_backward_pass_behind_a_forward_pass_by_itself(lib):
    ok = N.View4(4096, 64, 64, 64)
    for flags, code in ((N.FLAG_FORWARD_ONLY, -5), (0, -4)):   # (no workspace)
        assert lib.castle_bwd(*[ok] * 8, 1, 1, 16, 64, 1, 0.125, flags, *[ok] * 6, None, 0, None, 0, None, 0, None) == code


def test_small_linear_and_static_step_validate_on_the_host(lib):
    assert lib.castle_small_linear(4096, 4096, 4096, 4, 64, 30, 64, 64, 64, 1, None) == -2     # K % 8
    assert lib.castle_small_linear(4096, 4096, 4096, 4, 64, 32, 64, 64, 64, 0, None) == -1     # fp32 not offered
    assert lib.castle_small_linear(None, 4096, 4096, 4, 64, 32, 64, 64, 64, 1, None) == -5
    assert lib.castle_small_linear(4100, 4096, 4096, 4, 64, 32, 64, 64, 64, 1, None) == -5     # misaligned x
    # castle_decode_step_static: partials beyond the 4 MiB array, and a row beyond the capacity
    v = N.View4(4096, 128, 128, 128)
    rc = lib.castle_decode_step_static(v, v, v, v, 5, None, 8, v, v, v, v, v, v, 9000, 1, 128, 1, 0.1, 0, v, None, None)
    assert rc == -6 and b"static scratch" in lib.castle_error_string(rc)
    assert lib.castle_decode_step_static(v, v, v, v, 8, None, 8, v, v, v, v, v, v, 1, 1, 128, 1, 0.1, 0, v, None, None) == -2
    assert lib.castle_decode_step(v, v, v, v, 8, 8, v, v, v, v, v, v, 1, 1, 128, 1, 0.1, 0, v, None, 4096, 1 << 30, None) == -2


def test_products_refuse_operands_beyond_32_bit_offsets(lib):
    vp, i, i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    lib.castle_gemm.argtypes = [vp, i64, i, vp, i64, i, vp, i64, i, i, i, i, i, vp, vp, vp, i64, vp]
    lib.castle_gemm_operand_ok.argtypes = [i64, i64]

    def gemm(lda, a_t, ldb, b_t, M=40000, N=64, K=64):
        return lib.castle_gemm(4096, lda, a_t, 4096, ldb, b_t, 4096, N, M, N, K, 1, 0, None, None, 4096, 1 << 40, None)

    for ld in (65536, 1 << 31, (1 << 32) + 64, 1 << 40):   # 40000 rows of 65536: 2.6e9 elements; the others do not fit 32 bits themselves
        assert gemm(ld, 0, 64, 0) == -2
        assert gemm(64, 0, ld, 0, M=64, N=40000) == -2
        assert gemm(64, 0, ld, 1, M=64, K=40000) == -2
        assert gemm(ld, 1, 64, 1, M=64, K=40000) == -2
        assert not lib.castle_gemm_operand_ok(40000, ld)
    # the last element at 2^31 and just inside, with the room that the kernels' first steps want
    assert lib.castle_gemm_operand_ok(32767 - 192, 65536) and not lib.castle_gemm_operand_ok(32768 - 192, 65536)


def test_layer_steps_go_in_one_launch_only_where_that_was_measured_ahead(lib):
    ok = lib.castle_decode_layer_once_ok   # (B, H, d, dtype, t, dim)
    f32, bf16, f16 = 0, 1, 2
    for B, H, d, t, dim in ((1, 8, 64, 300, 512), (1, 16, 64, 300, 512), (4, 8, 64, 300, 512), (8, 8, 64, 300, 512), (16, 4, 64, 300, 512), (64, 2, 32, 100, 512),
                            (1, 2, 64, 3000, 512), (1, 4, 128, 700, 512), (1, 1, 16, 0, 8)):
        assert ok(B, H, d, bf16, t, dim) and ok(B, H, d, f16, t, dim)
    assert ok(1, 4, 64, f32, 300, 256) and ok(2, 4, 64, f32, 300, 256) and ok(1, 4, 64, f32, 900, 256)
    # contractions that a job reads in more than one round, also where the weights are few
    for dtype, dim in ((bf16, 520), (bf16, 768), (f16, 1024), (bf16, 2048), (bf16, 4096), (f32, 260), (f32, 512)):
        assert not ok(1, 4, 64, dtype, 300, dim)
    # more than two jobs a CU before the output projection, two thirds of one in fp32
    for B, H, dtype, t, dim in ((8, 16, bf16, 40, 512), (16, 8, bf16, 100, 512), (64, 4, bf16, 40, 512), (1, 32, bf16, 300, 512), (16, 4, f32, 100, 256), (1, 16, f32, 300, 256), (1, 5, f32, 600, 256)):
        assert not ok(B, H, 64, dtype, t, dim)
    # more than 10 MB of cached rows, more than 32 partial results of a head
    assert not ok(8, 8, 64, bf16, 1000, 512) and ok(1, 1, 128, bf16, 32 * 48, 512) and not ok(1, 1, 128, bf16, 32 * 48 + 1, 512)
    for B, H, d, dtype, t, dim in ((0, 8, 64, bf16, 1, 512), (1, 0, 64, bf16, 1, 512), (1, 8, 48, bf16, 1, 512), (1, 8, 64, 7, 1, 512), (1, 8, 64, bf16, -1, 512),
                                   (1, 8, 64, bf16, 1, 0), (65536, 1, 64, bf16, 1, 512), (1 << 30, 1 << 30, 128, bf16, 1 << 30, 1 << 30)):
        assert not ok(B, H, d, dtype, t, dim)


def test_check_raises_with_message(lib):
    with pytest.raises(RuntimeError, match="unsupported shape"):
        N.check(-2, "castle_fwd")
