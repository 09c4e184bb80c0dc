"""CPU-side checks of the native boundary: the library loads and exports every
symbol that include/odl_fp8.h declares (no compute calls: there is no GPU here)."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "odl_fp8.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(odl_fp8_\w+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    syms = declared_symbols()
    for must in ("odl_fp8_amax", "odl_fp8_cast", "odl_fp8_cast_transpose", "odl_fp8_gemm_nt",
                 "odl_fp8_scale_from_amax", "odl_fp8_delayed_update"):
        assert must in syms


def test_library_exports_every_declared_symbol():
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("libodl_fp8.so not built here (run `python -m optimus_dl_amd.build`)")
    lib = native.load()
    for sym in declared_symbols():
        assert hasattr(lib, sym), f"{sym} is declared in include/odl_fp8.h but not exported"
    assert sorted(native.EXPORTS) == declared_symbols()
    assert lib.odl_fp8_abi_version() == native.ABI_VERSION
    assert lib.odl_fp8_gemm_num_variants() >= 2
    assert b"generic" in lib.odl_fp8_gemm_variant_name(0)


def torch_equal(a, b):
    import torch

    return torch.equal(a, b)


def test_multi_tensor_planner_counts_work_and_refuses_bad_tables():
    """odl_fp8_multi_plan is host code: blocks of the amax pass (one per 64 KB, at most 512 per tensor), tiles of the
    cast (128 x 64), and the checks on shapes and pointers."""
    import numpy as np

    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    table = np.zeros((3, 9), dtype=np.int64)       # x, out, out_t, parts, dyn_out, scale, rows, cols, {src_dtype, reserved}
    table[0] = (4096, 8192, 16384, 32768, 64, 0, 1024, 1024, native.DT_BF16)           # 2 MB: 32 blocks, 8 x 16 tiles
    table[1] = (4096, 8192, 16384, 32768, 64, 0, 3072, 1024, native.DT_F32)            # 12 MB: 192 blocks, 24 x 16 tiles
    table[2] = (4096, 8192, 16384, 32768, 64, 0, 16384, 16384, native.DT_BF16)         # 512 MB: capped at 512 blocks
    amax, cast = native.MultiTensorPlan.plan_work(table, 0), native.MultiTensorPlan.plan_work(table, 1)
    assert amax.shape == (32 + 192 + 512, 2) and cast.shape == (128 + 384 + 128 * 256, 2)
    assert amax[:32, 0].eq(0).all() and amax[:32, 1].tolist() == list(range(32)) and amax[32, :].tolist() == [1, 0]
    assert cast[-1].tolist() == [2, 128 * 256 - 1]
    for col, bad in ((6, 1000), (7, 1020), (8, 5), (0, 0), (2, 16392), (1, 8196), (3, 0)):
        t = table.copy()
        t[1, col] = bad
        with pytest.raises(native.NativeError, match="odl_fp8_multi_plan"):
            native.MultiTensorPlan.plan_work(t, 0)
    with pytest.raises(native.NativeError, match="needs `scale`"):                      # the delayed phase reads *scale
        native.MultiTensorPlan.plan_work(table, 2)
    table[:, 5] = 128
    assert torch_equal(native.MultiTensorPlan.plan_work(table, 2), cast)
    assert native.load().odl_fp8_multi_plan(None, 0, 0, None, 0) == 0
    assert native.load().odl_fp8_multi_plan(table.ctypes.data, 3, 7, None, 0) == -1


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from optimus_dl_amd import native

    monkeypatch.setattr(native, "_lib", None)
    monkeypatch.setattr(native, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(native.NativeError, match="no fallback"):
        native.load()


@pytest.mark.parametrize("why", ["missing", "not a module", "other header", "other torch"])
def test_library_is_usable_without_the_cpp_side_of_its_wrappers(monkeypatch, tmp_path, caplog, why):
    """The extension belongs to one torch and one header.  Without a fitting one the library still loads, says so once, and
    every wrapper goes the long way; nothing of a module that does not fit is bound or called."""
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    native.load()
    monkeypatch.setattr(native, "_lib", None)
    monkeypatch.setattr(native, "_host", None)
    monkeypatch.setattr(native, "_HERE", str(tmp_path))
    if why == "not a module":
        (tmp_path / "_host.so").write_bytes(b"not an ELF file")
    elif why != "missing":
        bound = []

        class Module:
            abi_version = native.ABI_VERSION - (why == "other header")
            torch_version = "1.0.0" if why == "other torch" else __import__("torch").__version__.split("+")[0]
            bind = bound.append

        spec = type("Spec", (), {"loader": type("L", (), {"exec_module": lambda self, m: None})()})()
        monkeypatch.setattr(native.importlib.util, "spec_from_file_location", lambda *a: spec)
        monkeypatch.setattr(native.importlib.util, "module_from_spec", lambda s: Module)
    with caplog.at_level("WARNING"):
        assert native.load() is native.load() and native.is_built()
    assert [r for r in caplog.records if "rebuild" in r.message] and len(caplog.records) == 1
    assert native._host.amax_parts("anything", 0) is None and native._host.gemm_swiglu() is None
    assert why in ("missing", "not a module") or not bound


def test_cpp_side_of_the_wrappers_is_the_one_in_use():
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    native.load()
    assert native._host.abi_version == native.ABI_VERSION and callable(native._host.gemm_nt)


def test_cpu_tensors_are_refused_not_emulated():
    import torch

    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    with pytest.raises(native.NativeError):
        native.amax(torch.zeros((4, 4), dtype=torch.bfloat16))


def test_every_wrapper_refuses_cpu_tensors_with_an_error_of_its_own():
    """Also where no GPU is visible, where asking torch for the current stream would raise something else."""
    import torch

    from optimus_dl_amd import native as N

    x, codes, one = torch.zeros((128, 128), dtype=torch.bfloat16), torch.zeros((128, 512), dtype=torch.uint8), torch.ones(1)
    parts, row = torch.ones(N.AMAX_PARTS), torch.ones(128)
    scales = torch.zeros((4, 128, 4), dtype=torch.uint8)
    calls = {
        "amax_parts": (x,), "amax_parts_colsum": (x,), "cast_dynamic": (x, parts, N.E4M3), "quantise_small": (x, N.E4M3),
        "swiglu_amax_parts": (x, x), "swiglu_bwd_amax_parts": (x, x, x), "rmsnorm_amax_parts": (x, row, 1e-5), "rmsnorm_bwd": (x, x, row, row),
        "layernorm_amax_parts": (x, row, row, 1e-5), "layernorm_bwd": (x, x, row, row, row), "gelu_amax_parts": (x,), "gelu_bwd_amax_parts": (x, x),
        "quantize_rowcol": (x, N.E4M3), "cast_delayed": (x, one, N.E4M3), "gemm_nt": (codes, codes, N.E4M3, N.E4M3, one, one),
        "gemm_layouts": (codes, codes, N.E4M3, N.E4M3, N.K_FAST, N.K_FAST, one, one), "gemm_swiglu": (codes, codes, codes, N.E4M3, N.E4M3, one, one, one),
        "mx_cast": (x, N.E4M3), "block_cast": (x, N.E4M3), "mx_gemm_nt": (codes, scales, codes, scales, N.E4M3, N.E4M3),
        "swiglu_mx_cast": (x, x, N.E4M3, N.MX_CEIL), "swiglu_block_cast": (x, x, N.E4M3), "swiglu_cast_delayed": (x, x, one, N.E4M3, parts),
    }
    for name, args in calls.items():
        with pytest.raises(N.NativeError):
            getattr(N, name)(*args)
            raise AssertionError(name)


def test_build_rejects_asm_that_reads_a_scalar_too_soon_after_a_vector_write():
    from optimus_dl_amd.build import check_asm_hazards

    bad = """
	v_readlane_b32 s0, v180, 14
	;;#ASMSTART
	buffer_store_dwordx4 v[60:63], v0, s[16:19], s0 offen
	;;#ASMEND
"""
    good = bad.replace("\tbuffer_store", "\ts_nop 4\n\tbuffer_store")
    other_register = bad.replace("s_readlane", "s_readlane").replace("v_readlane_b32 s0", "v_readlane_b32 s7")
    in_descriptor = bad.replace("v_readlane_b32 s0", "v_readlane_b32 s18")
    assert len(check_asm_hazards(bad, "x.s")) == 1
    assert check_asm_hazards(good, "x.s") == []
    assert check_asm_hazards(other_register, "x.s") == []
    assert len(check_asm_hazards(in_descriptor, "x.s")) == 1
    # instructions the compiler emitted itself are its own business
    assert check_asm_hazards("\tv_readlane_b32 s0, v1, 2\n\tbuffer_load_dword v1, v0, s[16:19], s0 offen\n", "x.s") == []


def test_build_rejects_scaled_conversions_that_run_before_the_saturation_mode_is_set():
    from optimus_dl_amd.build import check_saturating_conversions

    mode = "\ts_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 1\n"
    cvt = "\tv_cvt_scalef32_pk_fp8_bf16 v3, v1, s2\n"
    assert check_saturating_conversions("_Z1kv:\n" + mode + "\tv_mov_b32 v0, 0\n" + cvt, "x.s") == []
    assert len(check_saturating_conversions("_Z1kv:\n" + cvt + mode, "x.s")) == 1
    # the mode belongs to the wave that set it: the next function starts without it
    assert len(check_saturating_conversions("_Z1kv:\n" + mode + cvt + "_Z1lv:\n" + cvt + cvt, "x.s")) == 1
    assert check_saturating_conversions("_Z1kv:\n\tv_cvt_pk_fp8_f32 v3, v1, v2\n", "x.s") == []


def test_split_count_is_a_host_side_decision_with_the_documented_shape_rules():
    """odl_fp8_gemm_split_count launches nothing; without a GPU it plans for 256 compute units."""
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    raw = native.load().odl_fp8_gemm_split_count
    count = lambda M, N, K, k_slow=0: raw(M, N, K, k_slow)
    assert count(8192, 14336, 4096) == 1                    # enough tiles: one launch
    assert count(8192, 1024, 4096) == 1                     # 128 tiles, short contraction
    assert count(1024, 4096, 8192) == 1 and count(1024, 4096, 8192, 1) >= 2      # no 128 x 128 alternative for K-slow operands
    for M, N, K in ((768, 768, 16384), (2304, 768, 16384), (1024, 1024, 16384), (8192, 1024, 151936), (8192, 768, 50304)):
        s = count(M, N, K)
        assert 2 <= s <= 16
        assert ((M + 255) // 256) * ((N + 255) // 256) * s <= 256             # the runs fit the chip at once
        steps, per = K // 128, ((-(-(K // 128) // s)) + 1) & ~1
        assert per >= 8 and steps - (s - 1) * per >= 4                        # no run shorter than 512
    for M, N, K in ((300, 512, 8192), (768, 768, 1024), (768, 776, 16384), (768, 768, 16400), (0, 768, 16384)):
        assert count(M, N, K) == 1                          # not multiples of 128, or too short to split


def test_whole_k_steps_never_run_the_generic_kernel():
    """Neither a whole product nor the rows of its last round that go to a second launch: over every remainder of tiles that
    the rows and columns can leave, the shapes among them whose rest is few 128 x 128 tiles and many of 256 x 256."""
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    generic = next(i for i, name in enumerate(native.gemm_variants()) if name.startswith("generic"))
    tails = 0
    shapes = [(4224, 5632, 4096), (16384, 1408, 4096), (612, 50304, 4096), (25088, 896, 4864), (8064, 3072, 4096), (32640, 768, 50304)]
    for shape in shapes:
        assert native.gemm_route(*shape)[1] > 0, "meant to have a second launch"
    for N in (384, 768, 896, 1024, 1408, 2944, 3072, 4096, 5632, 14336, 50304):
        for K in (128, 2048, 4096):
            shapes += [(M, N, K) for M in [*range(16, 20000, 336), *range(25088, 33000, 128)]]
    for M, N, K in shapes:
        for dtype in native._OUT_DTYPES:
            variant, rest, second = native.gemm_route(M, N, K, dtype)
            tails += rest > 0
            assert variant != generic and (rest == 0 or second != generic), (M, N, K, dtype)
    assert tails > 1000
    with pytest.raises(native.NativeError):
        native.gemm_route(16, 16, 20)


def test_short_contractions_of_few_tiles_keep_the_four_stage_kernel():
    """At most one 128 x 128 tile per compute unit: the tiled kernel below 16 K steps, the pipelined one from there on; more tiles
    in 128 x 192 from 8 steps on."""
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    names = native.gemm_variants()
    deep, wide = (next(i for i, n in enumerate(names) if n.startswith(tile) and "three stages" in n) for tile in ("128x128x128", "128x192x128"))
    tiled = next(i for i, n in enumerate(names) if n.startswith("128x128x128") and "three stages" not in n)
    for M, N in ((512, 768), (1024, 1024), (2048, 2048), (130, 16), (4016, 768)):
        for K in (128, 512, 1920):
            assert native.gemm_route(M, N, K) == (tiled, 0, 0), (M, N, K)
        assert native.gemm_route(M, N, 2048, accumulate=True)[0] in (deep, 8)
    assert native.gemm_route(1024, 1024, 2048) == (deep, 0, 0)
    assert native.gemm_route(1024, 5632, 512)[0] == tiled and native.gemm_route(1024, 5632, 1024)[0] == wide


def test_gate_up_and_product_in_one_launch_only_where_that_is_faster():
    """Up to 32 rows four rounds of 16-column blocks, up to 64 rows one round and a short contraction; never more than the entry
    takes (operands under 4 GiB): what it would refuse goes to the separate products, as it always has."""
    from optimus_dl_amd.native import gemm_swiglu_pays as pays

    assert pays(32, 14336, 4096) and pays(16, 16384, 128) and pays(64, 3072, 1024) and pays(48, 4096, 1920) and pays(32, 14336, 8192)
    assert not pays(16, 16388, 128) and not pays(32, 28672, 8192) and not pays(64, 4112, 1024) and not pays(48, 3072, 2048)
    assert not pays(48, 5632, 2048) and not pays(64, 14336, 4096) and not pays(33, 14336, 1024)
    assert not pays(65, 3072, 1024) and not pays(0, 3072, 1024) and not pays(32, 3074, 1024) and not pays(32, 3072, 1040)
    assert not pays(16, 16384, 2**18)


def test_data_gradient_sums_run_in_one_launch_only_for_whole_wave_tiles():
    """Whether the members' products are rounded once or one by one depends on the token count like this and no other way:
    multiples of 128 with more than 128 output tiles go in one launch."""
    from optimus_dl_amd import native

    qkv = [4096, 1024, 1024]
    assert native.dgrad_sum_in_one_launch(4096, 4096, qkv) and native.dgrad_sum_in_one_launch(4224, 4096, qkv)
    for tokens in (4016, 4112, 4095, 8176):
        assert not native.dgrad_sum_in_one_launch(tokens, 4096, qkv)
    assert not native.dgrad_sum_in_one_launch(2048, 4096, qkv)                  # 128 tiles
    assert not native.dgrad_sum_in_one_launch(4096, 4096, [4096]) and not native.dgrad_sum_in_one_launch(4096, 4096, [4096, 640])


def test_block_scaled_entry_points_refuse_bad_arguments_before_touching_a_device():
    """Argument and shape checks of the MXFP8 / blockwise entry points are host code that runs before any HIP call: they
    answer with an error code and a message here, where no GPU exists."""
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    L = native.load()
    err = lambda: L.odl_fp8_last_error().decode()
    p = 4096                                                     # any aligned non-null address: it is never dereferenced
    # cast: negative shape, unknown format, scale bytes without codes, blocked axis not a multiple of 32 / of 128
    assert L.odl_fp8_mx_cast(p, 0, -1, 64, 0, p, p, 0, None, None, 0, 0, None) != 0 and "negative" in err()
    assert L.odl_fp8_mx_cast(p, 0, 64, 64, 7, p, p, 0, None, None, 0, 0, None) != 0 and "fmt" in err()
    assert L.odl_fp8_mx_cast(p, 0, 64, 64, 0, p, None, 0, None, None, 0, 0, None) != 0 and "go together" in err()
    assert L.odl_fp8_mx_cast(p, 0, 64, 48, 0, p, p, 0, None, None, 0, 0, None) != 0 and "multiple of 32" in err()
    assert L.odl_fp8_mx_cast(p, 0, 64, 64, 0, p, p, 1, None, None, 0, 0, None) != 0 and "multiple of 128" in err()
    assert L.odl_fp8_mx_cast(p, 0, 0, 64, 0, None, None, 0, None, None, 0, 0, None) == 0        # nothing to do
    assert L.odl_fp8_mx_cast(p, 0, 64, 64, 0, p, p, 0, None, None, 0, 2, None) != 0 and "scale_rule" in err()
    # GEMM: K not a multiple of 32, unknown layout, K-step-major scales with K % 128 != 0, misaligned operand
    assert L.odl_fp8_mx_gemm_nt(p, p, p, p, 0, 64, 64, 48, 0, 0, None, p, 0, 0, None) != 0 and "multiple of 32" in err()
    assert L.odl_fp8_mx_gemm_nt(p, p, p, p, 5, 64, 64, 64, 0, 0, None, p, 0, 0, None) != 0 and "scales_layout" in err()
    assert L.odl_fp8_mx_gemm_nt(p, p, p, p, 1, 64, 64, 64, 0, 0, None, p, 0, 0, None) != 0 and "128" in err()
    assert L.odl_fp8_mx_gemm_nt(p + 8, p, p, p, 0, 64, 64, 64, 0, 0, None, p, 0, 0, None) != 0 and "aligned" in err()
    assert L.odl_fp8_mx_gemm_nt(p, p, p, p, 0, 0, 64, 64, 0, 0, None, p, 0, 0, None) == 0           # empty output
    # split over K: too few steps per run, workspace too small
    assert L.odl_fp8_mx_gemm_splitk(p, p, p, p, 256, 256, 1024, 0, 0, None, p, 0, 0, 4, p, 1 << 30, None) != 0 and "shorter than 512" in err()
    assert L.odl_fp8_mx_gemm_splitk(p, p, p, p, 256, 256, 8192, 0, 0, None, p, 0, 0, 4, p, 64, None) != 0 and "workspace" in err()
    # blockwise cast: sizes must be multiples of 128, margin in range
    assert L.odl_fp8_block_cast(p, 0, 128, 192, 0, 0, 0, p, p, None, None, None) != 0 and "multiples of 128" in err()
    assert L.odl_fp8_block_cast(p, 0, 128, 128, 0, 1000, 0, p, p, None, None, None) != 0 and "margin" in err()


def test_small_weight_gradients_read_dy_as_stored_only_where_that_is_no_slower():
    """The line in output elements and tokens that the measurements beside the rule draw."""
    from optimus_dl_amd.native import wgrad_direct_pays as pays

    assert not pays(768, 512, 1024) and not pays(512, 768, 8192) and pays(768, 512, 16384) and pays(512, 512, 16384)
    assert not pays(512, 256, 16384) and not pays(256, 256, 32768)
    assert not pays(768, 768, 8064) and pays(768, 768, 8192) and pays(2304, 768, 8192) and not pays(2048, 1024, 16384)
    assert pays(4096, 4096, 512) and pays(14336, 4096, 8192)


def test_a_split_that_one_launch_beats_is_dropped_before_its_workspace_is_made():
    """128 x 192 tiles in place of two runs, for every caller; the split entry itself runs what it is asked for."""
    from optimus_dl_amd import native

    if not native.is_built():
        pytest.skip("library not built")
    proposed = native.load().odl_fp8_gemm_split_count
    for M, N, K in ((8192, 768, 50304), (16384, 384, 50304)):
        assert proposed(M, N, K, 0) == 2 and native.gemm_split_count(M, N, K) == 1
    for M, N, K in ((8192, 1024, 151936), (3072, 1536, 50304), (768, 768, 16384), (8192, 14336, 4096), (300, 512, 8192)):
        assert native.gemm_split_count(M, N, K) == proposed(M, N, K, 0)
    assert native.gemm_split_count(8192, 768, 50304, True) == proposed(8192, 768, 50304, 1)
