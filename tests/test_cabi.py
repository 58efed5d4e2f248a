"""The C-ABI library loads and exports every symbol include/mi8.h declares (no GPU work is launched)."""

import ctypes
import re
from pathlib import Path

import pytest

import helpers
from olmo_core_amd import _C

ROOT = Path(__file__).resolve().parent.parent


def _declared_symbols(header="mi8.h"):
    text = (ROOT / "include" / header).read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mi8_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    assert _declared_symbols() == sorted(_C.EXPORTED_SYMBOLS)


def test_library_exports_every_declared_symbol():
    assert _C.is_built(), "libmi8.so is not built: run `python -m olmo_core_amd.build`"
    handle = ctypes.CDLL(str(_C.LIB_PATH))
    for name in _declared_symbols():
        assert hasattr(handle, name), f"libmi8.so does not export {name}"


def test_diagnostics_live_in_their_own_library():
    """The measurement kernels are no part of the drop-in boundary: mi8.h / libmi8.so do not carry them,
    mi8_diag.h / libmi8_diag.so do."""
    diag_syms = _declared_symbols("mi8_diag.h")
    assert diag_syms == sorted(_C.DIAG_EXPORTED_SYMBOLS)
    assert not set(diag_syms) & set(_declared_symbols())
    assert _C.DIAG_LIB_PATH.exists(), "libmi8_diag.so is not built: run `python -m olmo_core_amd.build`"
    main, diag = ctypes.CDLL(str(_C.LIB_PATH)), ctypes.CDLL(str(_C.DIAG_LIB_PATH))
    for name in diag_syms:
        assert hasattr(diag, name), f"libmi8_diag.so does not export {name}"
        assert not hasattr(main, name), f"libmi8.so exports the diagnostic {name}"
    assert _C.diag().mi8_probe_mfma_loop(7, 0, 1, 1, None, None) == -1  # argument check, nothing launched
    assert b"sink" in _C.diag().mi8_diag_last_error()


def test_host_only_entry_points():
    L = _C.lib()
    assert L.mi8_version() == 100
    assert L.mi8_gemm_num_variants() >= 1
    assert L.mi8_gemm_variant_name(0)
    assert L.mi8_gemm_variant_name(999) is None
    assert L.mi8_amax_slots_for(1) == 1
    assert L.mi8_amax_slots_for(1 << 40) == _C.AMAX_SLOTS
    assert L.mi8_colamax_workspace_slots(16384, 4096) % 4096 == 0
    # split-K planning: large problems are not split, a few rows go to the kernel that streams the weight once,
    # few output tiles with a long K are cut so that no slice is empty and each keeps at least four K steps
    assert L.mi8_gemm_splitk_suggest(16384, 11008, 4096) == 1
    assert L.mi8_gemm_splitk_suggest(16, 4096, 4096) == 1
    assert L.mi8_gemm_splitk_suggest(256, 256, 512) == 1
    for (m, n, k) in ((256, 4096, 11008), (100, 200, 1040), (384, 1024, 4096), (64, 11008, 4096)):
        s = L.mi8_gemm_splitk_suggest(m, n, k)
        steps = -(-k // 128)
        per = -(-steps // s)
        assert 2 <= s <= 32 and per >= 4 - 1 and (s - 1) * per < steps, (m, n, k, s)
    assert L.mi8_gemm_splitk_workspace_bytes(100, 30, 4) == 4 * 100 * 32 * 4
    assert L.mi8_gemm_splitk_workspace_bytes(0, 30, 4) == 0


def test_few_rows_slices():
    """17 to 64 rows: either no split, or the non-empty eighths of K - never another order of summation."""
    L = _C.lib()
    for m in (17, 32, 33, 64):
        for n in (8, 1024, 4096, 11008, 27648, 50304):
            for steps in list(range(1, 90)) + [216, 1000]:
                per = -(-steps // 8)
                assert L.mi8_gemm_splitk_suggest(m, n, 128 * steps - 16) in (1, -(-steps // per)), (m, n, steps)


def test_few_rows_swiglu_on_ring_tiles_only_where_offsets_fit():
    """Ring tiles have 32-bit offsets into a tile's rows (a partial maximum per 32 columns of h); rows that are further apart stay
    on the kernel with 64-bit addresses (one per 16)."""
    slots = lambda m, k: _C.lib().mi8_few_rows_swiglu_slots(m, 64, k, 1)  # noqa: E731
    assert slots(64, 4096) == slots(64, (1 << 26) - 16) == slots(32, (1 << 27) - 16) == 2
    assert slots(64, 1 << 26) == slots(33, 1 << 27) == slots(32, 1 << 27) == slots(9, 1 << 27) == 4


def test_variant_for():
    """The kernel a product runs on: few rows, tiles too few or of the wrong kind for the persistent kernel, and its own."""
    L = _C.lib()
    name = lambda m, n, k, dt=_C.MI8_BF16, acc=0: L.mi8_gemm_variant_name(L.mi8_gemm_variant_for(m, n, k, dt, acc)).decode()  # noqa: E731
    assert name(16, 4096, 4096) == "rows64x16_k8_m16x128" and name(64, 4096, 4096) == "64x64_ring4_eighths"
    assert name(16384, 4096, 4096) == name(16384, 4096, 4096, acc=1) == name(16384, 4100 // 8 * 8, 4096) == "256x256_dma_w4x128_m16x128"
    for args in ((300, 272, 144), (16384, 4096, 4112), (16384, 4096, 4096, _C.MI8_F32), (16383, 4096, 4096, _C.MI8_BF16, 1),
                 (16384, 4104, 4096, _C.MI8_BF16, 1), (16384, 4100, 4096)):
        assert "ring" in name(*args) and "eighths" not in name(*args), args
    # ... those of them that are large on the tiles with the persistent kernel's operand traffic
    for args in ((16384, 11008, 4112), (16384, 4096, 11024), (8192, 5120, 27648, _C.MI8_F32), (16383, 4096, 11008, _C.MI8_BF16, 1)):
        assert name(*args) == "256x256_ring2", args
    assert L.mi8_gemm_variant_for(0, 256, 256, _C.MI8_BF16, 0) == -1


def test_host_only_shape_helpers():
    """Sizes and shape predicates the callers plan with (no GPU work)."""
    L = _C.lib()
    # one code per 64 columns of a row, ragged last segment included
    assert L.mi8_rowseg_code_count(16384, 11008) == 16384 * 172
    assert L.mi8_rowseg_code_count(3, 65) == 6 and L.mi8_rowseg_code_count(0, 64) == 0
    assert L.mi8_swiglu_amax_state_words(16384, 11008) >= 4 and L.mi8_swiglu_amax_state_words(0, 0) == 0
    # the GEMM that records codes is the persistent tile kernel: full tiles, K in 128-byte steps, whole segments
    assert L.mi8_gemm_fp8_codes_supported(16384, 11008, 4096) == 1
    for shape in ((128, 11008, 4096), (16384, 11008, 4000), (16384, 11000, 4096)):
        assert L.mi8_gemm_fp8_codes_supported(*shape) == 0, shape
    # the fused SwiGLU launch replaces the separate GEMMs only where both run on that kernel
    assert L.mi8_gemm_fp8_swiglu_matches_separate(16384, 11008, 4096) == 1
    assert L.mi8_gemm_fp8_swiglu_matches_separate(64, 11008, 4096) == 0
    # the padded token axis of the grouped transposed copies: groups whose sizes sum to T fill at most
    # ceil(T / 128) + groups - 1 tiles of 128 rows
    assert L.mi8_grouped_padded_rows(131072, 64) == 131072 + 63 * 128
    assert L.mi8_grouped_padded_rows(5, 2) == 2 * 128


def test_argument_validation_happens_before_any_gpu_call():
    L = _C.lib()
    assert L.mi8_cast_rowwise(None, 0, 4, 16, 0, 0, None, 16, None, None) == -1
    assert "null" in _C.last_error()
    assert L.mi8_gemm_fp8(None, 0, 16, None, 0, 16, 1, 1, 16, None, 0, None, 0, None, 0, 16, -1, None) == -1
    assert L.mi8_gemm_fp8_splitk(None, 0, 16, None, 0, 16, 1, 1, 16, None, 0, None, 0, None, 0, 16, 2, None, 0, None) == -1
    assert L.mi8_amax_partials_batch(None, None, 1, 0, None, None, None) == -1
    ptrs, ns = (ctypes.c_void_p * 9)(), (ctypes.c_int64 * 9)()
    assert L.mi8_amax_partials_batch(ptrs, ns, 9, 0, ctypes.c_void_p(16), None, None) == -1 and "9 tensors" in _C.last_error()
    assert L.mi8_amax_partials_batch(ptrs, ns, 2, 0, ctypes.c_void_p(16), None, None) == -1 and "tensor 0 is null" in _C.last_error()
    with pytest.raises(Exception):
        _C.check(-2, "x")


def test_sums_are_not_rounded_to_bf16_values():
    """MI8_F32_OF_BF16 holds what a bf16 output would; of a sum that is a value rounded twice, which no entry point that adds forms."""
    L, p = _C.lib(), 1 << 20  # (16-byte aligned; never read: refused before any launch)
    args = (p, _C.MI8_E4M3, 256, p, _C.MI8_E4M3, 256, 128, 128, 256, p, 0, p, 0, p, _C.MI8_F32_OF_BF16, 128)
    assert L.mi8_gemm_fp8_accumulate(*args, None) == -2
    assert L.mi8_gemm_fp8_splitk_accumulate(*args, 2, p, 1 << 30, None) == -2
    chain = (_C.GemmProduct * 2)(*(_C.GemmProduct(p, 256, p, 256, 128, 128, 256, p, p, p, 128, 0, 0, _C.MI8_F32_OF_BF16, i) for i in range(2)))
    assert L.mi8_gemm_fp8_batch(chain, 2, _C.MI8_E4M3, _C.MI8_E4M3, None) == -2 and not L.mi8_gemm_fp8_batch_pays(chain, 2)
    assert L.mi8_gemm_variant_for(512, 512, 256, _C.MI8_F32_OF_BF16, 1) == -1 != L.mi8_gemm_variant_for(512, 512, 256, _C.MI8_F32_OF_BF16, 0)


def test_few_rows_entry_points_refuse():
    """What the two launches of a generation step do not take, by their numbers alone (the pointers are never followed)."""
    L, p, odd = _C.lib(), ctypes.c_void_p(256), ctypes.c_void_p(264)
    n = ctypes.c_int32(0)

    def swiglu(x=p, fp8=1, lda=256, sx=p, ldb=256, m=4, h=64, k=256, out=p):
        return L.mi8_few_rows_swiglu(x, fp8, lda, sx, p, p, ldb, m, h, k, p, p, 0, out, p, n, None)

    def cast_gemm(x=p, lda=256, slots=16, b=p, ldb=256, m=4, cols=64, k=256, out=p, ldc=64):
        return L.mi8_few_rows_cast_gemm(x, lda, p, slots, b, ldb, m, cols, k, p, 0, out, ldc, None)

    for call, code, kw, text in (
        (swiglu, -1, dict(x=None), "null"), (swiglu, -1, dict(sx=None), "null"), (swiglu, -1, dict(out=None), "null"),
        (swiglu, -2, dict(m=0), "rows"), (swiglu, -2, dict(m=65), "rows"), (swiglu, -2, dict(h=60), "H"), (swiglu, -2, dict(k=248), "K"),
        (swiglu, -2, dict(h=16 * _C.AMAX_SLOTS + 8), "H"), (swiglu, -2, dict(lda=240), "pitches"), (swiglu, -2, dict(ldb=264), "pitches"),
        (swiglu, -2, dict(x=odd), "aligned"), (swiglu, -2, dict(out=odd), "aligned"),
        (swiglu, -2, dict(fp8=0, m=17, k=16, lda=16, ldb=16), "bf16"), (swiglu, -2, dict(fp8=0, lda=272, ldb=272), "bf16"),
        (swiglu, -2, dict(fp8=0, m=16, k=1040, lda=1040, ldb=1040), "bf16"),
        (cast_gemm, -1, dict(x=None), "null"), (cast_gemm, -1, dict(slots=0), "n_slots"), (cast_gemm, -1, dict(slots=_C.AMAX_SLOTS + 1), "n_slots"),
        (cast_gemm, -2, dict(m=17), "rows"), (cast_gemm, -2, dict(cols=60), "N"), (cast_gemm, -2, dict(k=248), "K"),
        (cast_gemm, -2, dict(m=16, k=4112, lda=4112, ldb=4112), "elements"), (cast_gemm, -2, dict(lda=252), "lda"),
        (cast_gemm, -2, dict(ldb=264), "ldb"), (cast_gemm, -2, dict(ldc=56), "ldc"), (cast_gemm, -2, dict(ldc=66), "ldc"),
        (cast_gemm, -2, dict(x=odd), "aligned"), (cast_gemm, -2, dict(b=odd), "aligned"),
    ):
        assert call(**kw) == code and text in _C.last_error(), (call.__name__, kw, _C.last_error())


def test_grouped_pitch_limits():
    """T * lda below 4 GiB or lda below 2^27: refused by the numbers alone (the pointers are never followed)."""
    L, p = _C.lib(), ctypes.c_void_p(256)

    rc = L.mi8_grouped_gemm_fp8(p, 0, 1 << 27, p, 0, 256, 0, p, 1, 32, 1, 256, p, p, 0, p, 1, 1, None)
    assert rc == -2 and "2^27" in _C.last_error()


def _plan(M, N, K, swiglu=0, accumulate=0, units=256):
    """How the persistent kernel cuts a product: names and counts as mi8_diag.h lists them."""
    counts = (ctypes.c_int32 * 7)()
    assert _C.diag().mi8_diag_gemm_plan(M, N, K, swiglu, accumulate, units, ctypes.addressof(counts)) == 0
    return dict(zip(("rows", "whole", "halves", "split_halves", "quarters", "split_quarters", "blocks"), counts))


@pytest.mark.parametrize("units", [256, 304])
def test_partial_maxima_of_the_fused_swiglu_launch_have_room(units):
    """Four words per workgroup, MI8_AMAX_SLOTS in all, whatever mix of tiles a plan has and whatever rounds its launch up."""
    for M in (*range(256, 6000, 192), 5952, 777, 1999):
        for tiles in (*range(1, 140, 3), 49, 96):
            for K in (128, 512, 4096, 28672):
                plan = _plan(M, 128 * tiles, K, swiglu=1, units=units)
                assert 4 * plan["blocks"] <= _C.AMAX_SLOTS, (M, tiles, K, plan)


def test_slots_that_the_counting_sort_takes():
    """Its second launch reads every workgroup's counts in every workgroup: what passes 3e8 of them is for the caller's sort."""
    words = _C.lib().mi8_moe_sort_workspace_words
    for n, experts in ((8193, 1), (131072, 64), (1 << 20, 256), (1 << 21, 64), (1 << 22, 8)):
        assert words(n, experts) >= -(-n // 1024) * (experts + 2 + 1024), (n, experts)
    for n, experts in ((1 << 21, 256), (1 << 22, 64), (1 << 24, 1), ((1 << 30) - 1, 1), (1 << 30, 8), (131072, 257), (0, 8), (8193, 0)):
        assert words(n, experts) == 0, (n, experts)


@pytest.mark.parametrize("plans,how", [("HALF_PLANS", {}), ("QUARTER_PLANS", {}), ("HALF_SWIGLU_PLANS", dict(swiglu=1)),
                                       ("QUARTER_SWIGLU_PLANS", dict(swiglu=1)), ("ACCUMULATE_PLANS", dict(accumulate=1))], ids=str)
def test_sizes_of_the_tile_tests_have_the_tiles_they_are_for(plans, how):
    for (M, N, K), kinds in getattr(helpers, plans).items():
        p = _plan(M, N, K, **how)
        end = 256 * p["rows"]  # where the rows at the end start
        found = ["W"] * (p["whole"] > 0) + ["h"] * (p["split_halves"] > 0) + ["q"] * (p["split_quarters"] > 0) + ["+"] * (end > M)
        if p["halves"] > p["split_halves"]:
            found.append("H" if end + 128 <= M else "H-")
            end += 128
        if p["quarters"] > p["split_quarters"]:
            found.append("Q" if end + 64 <= M else "Q-")
        assert " ".join(sorted(found)) == kinds, (M, N, K, p)
