"""CPU-only checks of the drop-in boundary: the C-ABI library loads and exports every symbol the header declares,
argument validation rejects bad calls before any device work, and the torch operator surface (schemas, python
shims, error behaviour) matches the reference's (kernels/*/pkg/*_unified/csrc/*_kernel.cpp, ops.py)."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "mi355_serving.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mi355_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol(lib):
    names = declared_functions()
    assert names == sorted(lib.EXPORTED_SYMBOLS)
    cdll = lib.load()
    for n in names:
        assert getattr(cdll, n) is not None
    assert cdll.mi355_serving_version() == 200
    # the test / tuning hooks are exported but stay out of the public header, and no process-wide switch exists any more
    for n in lib.INTERNAL_SYMBOLS:
        assert n not in names and getattr(cdll, n) is not None
    assert not any("debug" in n for n in names)
    assert not hasattr(cdll, "mi355_debug_set_gemm_variant") and not hasattr(cdll, "mi355_debug_set_fmha_variant")


def test_profiling_twin_exports_the_library_plus_its_readers(lib):
    # libmi355_serving_timeline.so (bench.py --timeline) is the same library with time stamps compiled into the tiled GEMM and the
    # attention kernels: every public symbol, plus the readers of the records and the read-only yardstick kernel; the product
    # library carries none of those
    twin = ctypes.CDLL(os.path.join(os.path.dirname(lib.LIB_PATH), "libmi355_serving_timeline.so"))
    for n in declared_functions():
        assert getattr(twin, n) is not None
    extra = ("mi355_timeline_read_hgemm", "mi355_timeline_read_fmha_fwd", "mi355_timeline_read_fmha_decode",
             "mi355_timeline_stream_read")
    cdll = lib.load()
    for n in extra:
        assert getattr(twin, n) is not None
        assert not hasattr(cdll, n)
    assert twin.mi355_timeline_stream_read(None, ctypes.c_size_t(64), None, None) != 0   # null pointers: refused, nothing launched


def test_a_refused_step_kernel_leaves_no_error_text(lib):
    """The decoder layer offers its first two products to the step's kernels and goes on with the single calls where they refuse:
    a forward pass that succeeds leaves the text of the caller's last failure as it was. (Refused before anything is launched.)"""
    cdll = lib.load()
    p = ctypes.c_void_p(0x1000)

    def qkv(B, S, hidden, norm=p):
        return cdll.mi355_internal_step_qkv(p, norm, 1e-5, p, p, p, B, S, 8, 2, hidden, S * 1536, 1536, 128, p, p, p, 0, 16, 0, None)

    assert cdll.mi355_hgemm(None, None, None, 4, 4, 4, 4, 4, 4, 0, None) == lib.ERR_BAD_ARGUMENT
    text = cdll.mi355_last_error()
    for rows, hidden in ((65, 1024), (9, 1024), (8, 4096), (1, 1000), (1, 512)):     # beyond 64 rows, 8, a CU's LDS; widths
        assert qkv(rows, 1, hidden) == qkv(1, rows, hidden) == lib.ERR_UNSUPPORTED
    for rows, hidden in ((9, 1024), (8, 4096), (1, 1000), (1, 512)):
        assert cdll.mi355_internal_step_gate_up(p, p, 1e-5, p, p, rows, 2816, hidden, 0, None) == lib.ERR_UNSUPPORTED
    assert cdll.mi355_last_error() == text
    assert qkv(0, 1, 1024) == lib.ERR_BAD_ARGUMENT and b"step_qkv" in cdll.mi355_last_error()


def test_capi_rejects_bad_arguments_without_a_gpu(lib):
    cdll = lib.load()
    assert cdll.mi355_hgemm(None, None, None, 4, 4, 4, 4, 4, 4, 0, None) == 10001
    assert b"null pointer" in cdll.mi355_last_error()
    p = ctypes.c_void_p(0x1000)
    p2 = ctypes.c_void_p(0x100000)
    assert cdll.mi355_hgemm(p, p, p, 0, 4, 4, 4, 4, 4, 0, None) == 10001
    assert cdll.mi355_hgemm(p, p, p, 4, 4, 4, 4, 4, 4, 7, None) == 10001
    assert b"layout" in cdll.mi355_last_error()
    assert cdll.mi355_hgemm(p, p, p, 4, 8, 4, 4, 4, 4, 0, None) == 10001  # ldb < N
    assert cdll.mi355_fmha_fwd(p, p, p, p, None, 1, 4, 1, 8, 8, 64, 0.1, 0, 8, None) == 10002  # head_dim != 128
    assert b"128" in cdll.mi355_last_error()
    assert cdll.mi355_fmha_fwd(p, p, p, p, None, 1, 5, 2, 8, 8, 128, 0.1, 0, 8, None) == 10001  # Hq % Hkv
    assert cdll.mi355_fmha_fwd(p, p, p, p, None, 1, 4, 2, 8, 8, 128, 0.1, 0, 9, None) == 10001  # kv_valid > Sk
    assert cdll.mi355_fmha_fwd(p, p, p, p, None, 1, 4, 2, 8, 8, 128, -1.0, 0, 8, None) == 10001  # scale <= 0
    def strided(st):
        arr = (ctypes.c_int64 * 12)(*st)
        return cdll.mi355_fmha_fwd_strided(p, p, p, p, None, 2, 4, 2, 8, 8, 128, 0.1, 0, 8, arr, None)
    good = [4096, 128, 512] * 4
    assert strided(good[:2] + [516] + good[3:]) == 10001  # q row stride not a multiple of 8 elements
    assert b"stride 2" in cdll.mi355_last_error()
    assert strided(good[:5] + [-512] + good[6:]) == 10001  # negative stride
    assert strided(good[:11] + [64]) == 10001              # rows of O overlap
    assert b"overlap" in cdll.mi355_last_error()
    assert cdll.mi355_fmha_fwd_strided(p, p, p, p, None, 2, 4, 2, 8, 8, 128, 0.1, 0, 8, None, None) == 10001
    # caller-owned workspace: size query and the checks that run before any launch
    wsb = cdll.mi355_fmha_fwd_workspace_bytes
    assert wsb(1, 32, 8, 4096, 4096, 4096) == 0 and wsb(1, 32, 8, 1, 400, 400) == 0     # prefill, short cache: no split-KV
    need = wsb(1, 32, 8, 1, 8192, 8192)
    assert 0 < need <= 16 << 20 and need % 16 == 0
    assert wsb(8, 32, 8, 1, 8192, 8192) > 0 and wsb(1, 32, 8, 1, 8192, 9000) == 0         # invalid sizes report 0
    assert wsb(1, 32, 8, 128, 8192, 8192) == 8 * 32 * 128 * 260 and wsb(1, 32, 8, 512, 8192, 8192) == 4 * 32 * 512 * 260   # key ranges
    assert wsb(1, 32, 8, 512, 2048, 2048) == 0 and wsb(1, 32, 8, 128, 8192, 2047) == 0
    ws_call = lambda ptr, nbytes, dtype=0: cdll.mi355_fmha_fwd_ws(p, p, p, p, None, 1, 32, 8, 1, 8192, 128, 0.1, 0, 8192, None,
                                                                  dtype, ptr, nbytes, None)
    assert ws_call(None, 0) == 10001 and b"workspace" in cdll.mi355_last_error()
    assert ws_call(p2, need - 16) == 10001
    assert ws_call(ctypes.c_void_p(0x100008), need) == 10001                                 # misaligned
    assert ws_call(p2, need, dtype=5) == 10001 and b"dtype" in cdll.mi355_last_error()
    # layer glue
    assert cdll.mi355_rmsnorm(p, None, None, p, p, 4, 100, 104, 0, 0, 104, 1e-5, None) == 10001   # hidden % 8
    assert cdll.mi355_rmsnorm(p, p, None, p, p, 4, 128, 128, 128, 128, 128, 1e-5, None) == 10001   # residual without residual_out
    assert cdll.mi355_rmsnorm(p, None, None, p, p, 4, 128, 64, 0, 0, 128, 1e-5, None) == 10001     # ldx < hidden
    assert cdll.mi355_rope(p, p, 1, 4, 2, 0, 64, 1024, 256, 1024, 256, p, p, p, 0, 16, None) == 10002    # head_dim != 128
    assert cdll.mi355_rope(p, p, 1, 4, 1, 1, 128, 1024, 128, 1024, 256, p, p, p, 0, 16, None) == 10001   # row stride < heads * 128
    assert cdll.mi355_rope(p, p, 1, 4, 2, 0, 128, 1024, 256, 1024, 256, p, p, None, 0, 16, None) == 10001
    assert cdll.mi355_rope_qkv(p, p, 1, 4, 4, 1, 128, 4096, 512, 1024, 256, 128, p, p, p, 0, 16, None) == 10001   # x_row < (4 + 2) * 128
    assert cdll.mi355_rope_qkv(p, p, 1, 4, 4, 1, 128, 4096, 768, 1024, 128, 128, p, p, p, 0, 16, None) == 10001   # token-major row too short for k | v
    assert cdll.mi355_rope_qkv(p, p, 1, 4, 4, 1, 128, 4096, 768, 1024, 128, 256, p, p, p, 0, 16, None) == 10001   # head-major: head stride < 4 rows
    assert cdll.mi355_rope_qkv(p, p, 1, 4, 4, 1, 128, 4096, 768, 1024, 256, 64, p, p, p, 0, 16, None) == 10001    # out_head < 128
    assert cdll.mi355_rope_qkv(p, p, 1, 4, 4, 0, 128, 4096, 768, 1024, 256, 128, p, p, p, 0, 16, None) == 10001   # no kv heads
    assert cdll.mi355_rope_qkv(p, None, 1, 4, 4, 1, 128, 4096, 768, 1024, 256, 128, p, p, p, 0, 16, None) == 10001
    assert cdll.mi355_rope_qkv_bf16(p, p, 1, 4, 4, 1, 64, 4096, 768, 1024, 256, 128, p, p, p, 0, 16, None) == 10002   # head_dim != 128
    assert cdll.mi355_silu_mul(p, p, 4, 64, 0, 64, 64, None) == 10001                               # ld_in < 2 * inter
    assert cdll.mi355_silu_mul(p, p, 0, 64, 0, 128, 64, None) == 10001
    assert cdll.mi355_silu_mul(p, p, 4, 64, 12, 128, 64, None) == 10001                             # interleave % 8
    assert cdll.mi355_hgemm_silu_mul(p, p, p, 256, 128, 64, 64, 64, 128, 2, None) == 10002          # TN has no fused epilogue
    assert cdll.mi355_hgemm_silu_mul(p, p, p, 256, 128, 64, 64, 64, 64, 1, None) == 10001           # ldc < N
    assert cdll.mi355_hgemm_silu_mul(p, p, p, 32, 128, 96, 96, 96, 128, 1, None) == 10002           # K not a multiple of 64: product + silu_mul
    assert b"mi355_silu_mul" in cdll.mi355_last_error()
    assert cdll.mi355_hgemm_add(p, p, None, p, 64, 64, 64, 64, 64, 64, 64, 0, None) == 10001            # residual missing
    assert cdll.mi355_hgemm_add(p, p, p2, p, 64, 64, 64, 64, 64, 32, 64, 0, None) == 10001              # ldr < N
    assert b"ldr" in cdll.mi355_last_error()
    assert cdll.mi355_hgemm_add(p, p, p, p, 64, 64, 64, 64, 64, 128, 64, 0, None) == 10001              # in place with ldr != ldc
    assert cdll.mi355_gemm_add_bf16(p, p, p2, p, 64, 64, 0, 64, 64, 64, 64, 0, None) == 10001           # K < 1
    with pytest.raises(lib.Mi355Error):
        lib.hgemm_raw(0, 0, 0, 4, 4, 4, 4, 4, 4, 0)


def test_operator_schemas_match_reference():
    import fmha_unified  # noqa: F401
    import gemm_unified  # noqa: F401
    for i in range(17):  # gemm_kernel.cpp:10-26
        op = getattr(torch.ops.gemm_unified, f"finegemm_{i}").default
        assert str(op._schema) == f"gemm_unified::finegemm_{i}(Tensor a, Tensor b) -> Tensor"
    for i in range(8):  # fmha_kernel.cpp:10-17
        op = getattr(torch.ops.fmha_unified, f"finefmha_{i}").default
        assert str(op._schema) == (f"fmha_unified::finefmha_{i}(Tensor q, Tensor k, Tensor v, bool causal, "
                                   "bool is_decode, int decode_length) -> Tensor")
    assert "-> (Tensor, Tensor)" in str(torch.ops.fmha_unified.finefmha_fwd_lse.default._schema)


def test_gemm_operator_validation_errors():
    import gemm_unified
    a = torch.randn(8, 8).half()
    with pytest.raises(RuntimeError, match="GPU tensors"):
        gemm_unified.ops.fine_gemm(a, a, 0)
    with pytest.raises(RuntimeError, match="float16"):
        gemm_unified.ops.fine_gemm(a.float(), a, 0)
    with pytest.raises(RuntimeError, match="inner dimensions"):
        gemm_unified.ops.fine_gemm(a[:, :4], a, 0)
    with pytest.raises(RuntimeError, match="inner dimensions"):  # index 13 reads b as [N, K]
        gemm_unified.ops.fine_gemm(a, a[:, :4], 13)
    with pytest.raises(RuntimeError, match="2-D"):
        gemm_unified.ops.fine_gemm(a[None], a, 0)
    with pytest.raises(AttributeError):
        gemm_unified.ops.fine_gemm(a, a, 17)
    assert gemm_unified.ops.LAYOUT_OF_INDEX[16] == "TN" and gemm_unified.ops.LAYOUT_OF_INDEX[14] == "NT"


def test_fmha_operator_validation_errors():
    import fmha_unified
    q = torch.randn(1, 4, 8, 128).half()
    kv = torch.randn(1, 2, 8, 128).half()
    with pytest.raises(RuntimeError, match="GPU tensors"):
        fmha_unified.ops.fine_fmha(q, kv, kv, True, False, 2)
    with pytest.raises(RuntimeError, match="128"):
        fmha_unified.ops.fine_fmha(q[..., :64], kv[..., :64], kv[..., :64], True, False, 2)
    with pytest.raises(RuntimeError, match="float16"):
        fmha_unified.ops.fine_fmha(q.float(), kv, kv, True, False, 2)
    with pytest.raises(RuntimeError, match="decode"):  # semi/fmha_2_amd.cpp:331-333
        fmha_unified.ops.fine_fmha(q, kv, kv, True, True, 2)
    with pytest.raises(RuntimeError, match="multiple of kv heads"):
        fmha_unified.ops.fine_fmha(q[:, :3], kv, kv, False, False, 2)
    with pytest.raises(RuntimeError, match="decode_length"):
        torch.ops.fmha_unified.finefmha_2.default(q, kv, kv, False, False, 9)
    with pytest.raises(RuntimeError, match="v shape"):
        fmha_unified.ops.fine_fmha(q, kv, kv[:, :, :4], False, False, 2)


def test_product_code_does_not_touch_the_oracle():
    pkg = os.path.join(ROOT, "understanding-gpu-architecture-implications-on-llm-serving-workloads_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".cpp", ".hip", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert "serving_oracle" not in text and "oracle/" not in text, os.path.join(dirpath, f)


def test_generation_step_partial_results_fit_where_256_workgroups_would(lib):
    # The number of key ranges is chosen by a model of their time. No call may need more than the 4 MiB static array (what
    # mi355_fmha_fwd_noalloc has, and the smallest buffer a captured call finds) that would fit it cut into ranges of at least
    # eight 32-key tiles, one per CU in all; and no call that would then need no memory at all may need some.
    wsb = lib.load().mi355_fmha_fwd_workspace_bytes
    limit = 4 << 20
    for pairs in list(range(1, 40)) + list(range(40, 256, 7)):
        for cols in (1, 4, 8, 12, 16, 24, 32):
            for tiles in list(range(16, 64, 5)) + [64, 100, 141, 256, 257, 400, 1000]:
                even = max(1, min((256 + pairs // 2) // pairs, (tiles + 7) // 8, 256))
                per = -(-tiles // even)
                even = -(-tiles // per)
                need = wsb(pairs, cols, 1, 1, tiles * 32, tiles * 32)
                if 65536 + pairs * even * cols * 528 <= limit:
                    assert need <= limit, (pairs, cols, tiles, need)
                if even == 1:
                    assert need == 0, (pairs, cols, tiles, need)


def decode_plan(lib, B, Hq, Hkv, Sq, kv):
    splits, waves = ctypes.c_int(), ctypes.c_int()
    assert lib.load().mi355_internal_fmha_decode_plan(B, Hq, Hkv, Sq, kv, ctypes.byref(splits), ctypes.byref(waves)) == 0
    return splits.value, waves.value


def even_cut(pairs, tiles):
    """Ranges of the even cut: about 256 workgroups of at least eight 32-key tiles."""
    even = max(1, min((256 + pairs // 2) // pairs, (tiles + 7) // 8, 256))
    return -(-tiles // -(-tiles // even))


def test_generation_step_has_no_fewer_key_ranges_and_waves_than_its_precision_needs(lib):
    # A wave rounds its probabilities against the maximum of its first tile; with fewer ranges or waves than the even cut on
    # four waves the pieces get longer and the error of O against float64 grows by up to 5 %.
    for pairs in list(range(1, 40)) + list(range(40, 256, 7)) + [300, 512, 1024]:
        for cols in (1, 4, 8, 32):
            for kv in (1, 32, 64, 65, 128, 300, 511, 512, 513, 700, 1000, 2208, 2336, 4500, 8191, 8192, 16384, 32768):
                splits, waves = decode_plan(lib, pairs, cols, 1, 1, kv)
                tiles = (kv + 31) // 32
                if splits == 0:      # the prefill kernel's
                    assert kv < 512, (pairs, cols, kv)
                    continue
                assert splits >= (even_cut(pairs, tiles) if kv >= 512 and pairs < 256 else 1), (pairs, cols, kv, splits)
                assert waves == 4 or (splits == 1 and kv <= 64), (pairs, cols, kv, waves)
    assert decode_plan(lib, 1, 32, 8, 1, 8191) == (32, 4)      # one sequence, 8 kv heads: the even cut itself


@pytest.mark.parametrize("B,Hq,Hkv", [(1, 8, 2), (1, 32, 8), (3, 32, 8), (16, 32, 8), (20, 32, 8), (13, 16, 4), (1, 64, 8), (2, 32, 1)])
def test_workspace_asked_for_at_the_longest_cache_serves_the_shorter_ones(lib, B, Hq, Hkv):
    # a generation loop asks once for mi355_fmha_fwd_ws. Where the even cut of the shorter cache has no more ranges than that
    # of the longer one, the shorter one must not need more (the even cut alone may: 32 ranges of 8 tiles, 29 of 9).
    wsb = lib.load().mi355_fmha_fwd_workspace_bytes
    lengths = list(range(512, 12000, 32)) + [16384, 16416, 32768]
    need = [wsb(B, Hq, Hkv, 1, 32768, kv) for kv in lengths]
    cuts = [even_cut(B * Hkv, (kv + 31) // 32) for kv in lengths]
    most_need = most_cut = 0
    for kv, n, c in zip(lengths, need, cuts):
        assert (n > 0) == (c > 1), (kv, n, c)      # memory is asked for exactly where the even cut takes some
        if c >= most_cut:
            assert n >= most_need, (kv, n, most_need)
        splits, _ = decode_plan(lib, B, Hq, Hkv, 1, kv)
        assert n >= (65536 + B * Hkv * splits * (Hq // Hkv) * 528 if splits > 1 else 0), (kv, n, splits)
        most_need, most_cut = max(most_need, n), max(most_cut, c)


def test_short_caches_take_the_kernel_that_is_done_first(lib):
    # several queries over a short cache: the prefill kernel, until its query heads need several rounds of workgroups
    for B, Hq, Hkv, Sq, kv in ((1, 32, 8, 8, 32), (1, 32, 8, 8, 64), (8, 32, 8, 8, 511), (4, 32, 32, 32, 128), (4, 32, 32, 20, 300), (1, 64, 8, 2, 64),
                               (32, 32, 32, 32, 511), (1, 8, 2, 5, 128)):
        assert decode_plan(lib, B, Hq, Hkv, Sq, kv)[0] == 0, (B, Hq, Hkv, Sq, kv)
    for B, Hq, Hkv, Sq, kv in ((1, 32, 8, 1, 300), (1, 8, 2, 1, 301), (1, 32, 32, 1, 128), (16, 32, 8, 2, 300), (64, 32, 8, 5, 64), (128, 32, 8, 8, 300),
                               (32, 32, 32, 1, 64), (1, 32, 8, 8, 512), (4, 32, 32, 32, 700)):
        assert decode_plan(lib, B, Hq, Hkv, Sq, kv)[0] > 0, (B, Hq, Hkv, Sq, kv)


def test_short_caches_of_many_sequences_take_the_generation_step_kernel(lib):
    # 17 to 32 columns, or up to 64 keys of more (sequence, kv head) pairs than CUs, where the prefill kernel's items need several rounds
    for B, Hq, Hkv, Sq, kv in ((16, 32, 1, 1, 100), (32, 16, 2, 4, 65), (16, 32, 8, 8, 65), (16, 32, 8, 8, 128), (8, 64, 8, 4, 128), (20, 32, 32, 12, 8),
                               (64, 32, 32, 12, 33), (32, 32, 32, 16, 8)):
        assert decode_plan(lib, B, Hq, Hkv, Sq, kv) == (1, 2 if kv <= 64 else 4), (B, Hq, Hkv, Sq, kv)
    for B, Hq, Hkv, Sq, kv in ((1, 32, 8, 8, 300), (8, 32, 32, 17, 128), (4, 32, 8, 5, 64), (1, 32, 1, 1, 480), (2, 32, 32, 28, 448)):
        assert decode_plan(lib, B, Hq, Hkv, Sq, kv)[0] == 0, (B, Hq, Hkv, Sq, kv)


@pytest.mark.parametrize("layout,few_rows,shapes", [
    # up to 16 rows against an nn.Linear weight: the small-M kernels, which stream it fastest, also beyond a layer's widths
    ("NT", (1, 4, 8), [(50304, 4096), (50257, 4096), (128256, 2048), (28672, 8192), (14336, 14336), (14336, 4096), (4096, 14336), (4096, 4096)]),
    ("NT", (16,), [(50304, 4096), (32000, 4096), (28672, 4096), (28672, 8192), (14336, 4096), (4096, 14336), (8192, 8192), (4096, 4096)]),
    # a short K, where a kernel that starts fast is done first
    ("NT", (1, 4, 11), [(3520, 448), (4096, 384), (576, 320), (1024, 192)]), ("NN", (1, 8), [(1088, 448), (320, 384)]),
    ("NN", (1, 16), [(14336, 4096)])])
def test_products_of_few_rows_that_the_small_m_kernels_finish_first(lib, layout, few_rows, shapes):
    for M in few_rows:
        for N, K in shapes:
            choice = lib.load().mi355_internal_hgemm_choice(M, N, K, K if layout == "NT" else N, lib.LAYOUTS[layout], None)
            assert choice == 8, (M, N, K, layout, choice)


@pytest.mark.parametrize("M,N,K,layout", [(20, 220928, 128, "NT"), (45, 258816, 128, "TN"), (64, 10240, 8192, "NN"), (12, 13494, 12872, "NT"),
                                          (16, 50264, 4096, "NN"), (16, 28672, 4096, "NN"), (64, 14336, 4096, "NT")])
def test_products_of_few_rows_that_the_tiles_finish_first(lib, M, N, K, layout):
    assert lib.load().mi355_internal_hgemm_choice(M, N, K, K if layout == "NT" else N, lib.LAYOUTS[layout], None) != 8


def test_128_columns_and_ranges_of_k_are_taken_where_they_are_done_first(lib):
    ranges = lambda M, N, K, layout: lib.load().mi355_internal_hgemm_wide_ranges(M, N, K, N, lib.LAYOUTS[layout])
    for M, N, K, layout, want in ((16, 14336, 4096, "NN", 2), (16, 4096, 4096, "NN", 8), (8, 6144, 4096, "TN", 5), (16, 4096, 14336, "NN", 8),
                                  (1, 1024, 4096, "NN", 8), (16, 12288, 4096, "TN", 2)):
        assert ranges(M, N, K, layout) == want, (M, N, K, layout)
    # a short K, where the merge costs more than it gives; more rows or columns; an nn.Linear weight
    for M, N, K, layout in ((16, 8192, 1024, "NN"), (16, 4096, 512, "TN"), (17, 4096, 4096, "NN"), (16, 28672, 4096, "NN"), (16, 4096, 4096, "NT")):
        assert ranges(M, N, K, layout) == 0, (M, N, K, layout)


def test_aligned_copies_of_large_operands_are_asked_for_only_where_they_are_repaid(lib):
    # unaligned dense operands, bytes of the copies asked for: nothing where reading and writing a large operand takes longer than
    # the product takes without copies
    ask = lambda M, N, K, lay: lib.load().mi355_gemm_workspace_bytes(4096, 1 << 40, M, N, K, M if lay == "TN" else K, K if lay == "NT" else N, lib.LAYOUTS[lay])
    for M, N, K, lay in ((1, 128257, 512, "NN"), (1, 256001, 1024, "TN"), (4, 128257, 512, "NN"), (2, 53001, 102, "NN")):
        assert ask(M, N, K, lay) == 0, (M, N, K, lay)
    for M, N, K, lay in ((64, 50257, 4096, "NN"), (16, 14337, 4096, "NN"), (16, 128256, 4099, "NT"), (1999, 3001, 2503, "NN"), (256, 4097, 4096, "TN")):
        assert ask(M, N, K, lay) >= N * K * 2 * (lay != "TN" or N % 8 != 0), (M, N, K, lay)


def test_the_copies_of_a_call_never_take_more_than_is_asked_for_and_often_nothing(lib):
    # what the operators allocate (the bytes that the call uses) against what the public query asks for
    import random
    args = lambda M, N, K, lay: (4096, 1 << 40, M, N, K, M if lay == "TN" else K, K if lay == "NT" else N, lib.LAYOUTS[lay])
    ask = lambda *c: lib.load().mi355_gemm_workspace_bytes(*args(*c))
    use = lambda *c: lib.load().mi355_internal_gemm_copy_bytes(*args(*c))
    for c in ((8, 50257, 4096, "NN"), (64, 50257, 4096, "NN"), (62, 19578, 5867, "NT"), (16, 14337, 4096, "NN")):
        assert use(*c) == 0 and ask(*c) > 100 << 20, c       # read where they lie
    for c in ((1999, 3001, 2503, "NN"), (2169, 2399, 1727, "NT"), (4097, 4097, 4097, "TN")):
        assert use(*c) == ask(*c) > 0, c
    rng = random.Random(1)
    for _ in range(3000):
        c = tuple(int(lo * (hi / lo) ** rng.random()) for lo, hi in ((1, 8192), (16, 100000), (8, 16384))) + (rng.choice(("NN", "NT", "TN")),)
        assert use(*c) in (0, ask(*c)), c


def test_the_direct_kernel_leaves_no_cu_of_an_xcd_with_twice_the_work_of_the_others(lib):
    # an XCD's 32 CUs take an eighth of the tiles of every range, rounded up: 84 tiles in 3 ranges are 33 workgroups on most XCDs
    for M, N, K, layout in ((751, 385, 8595, "NN"), (1029, 261, 6005, "NN"), (561, 551, 5443, "NT"), (1287, 221, 5129, "NT")):
        variant = lib.load().mi355_internal_hgemm_direct_choice(M, N, K, lib.LAYOUTS[layout], None)
        tile, ranges = {10: 64, 11: 128}[variant & 15], max(1, variant >> 4)
        tiles = -(-M // tile) * -(-N // tile)
        assert -(-tiles // 8) * ranges <= 32, (M, N, K, layout, tile, ranges)
