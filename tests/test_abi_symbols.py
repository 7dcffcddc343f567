"""The shipped library loads without a GPU and exports exactly the C ABI that
include/w4_abi.h declares (no compute calls here)."""
import copy
import ctypes
import inspect
import os
import pickle
import re
import subprocess
import sys
import sysconfig

import pytest

import w4amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "w4_abi.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(w4_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported_and_bound():
    capi = w4amd.capi()
    lib = ctypes.CDLL(capi.LIB_PATH)
    names = _declared()
    assert len(names) >= 20
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in w4_abi.h but not exported"
    assert set(capi.SIGNATURES) == set(names), "the ctypes view and the header disagree"


def test_validation_runs_without_a_device():
    capi = w4amd.capi()
    v = capi.packed_view(2, 32, 7, 4, 1, 1, 1)
    try:
        capi.gemm(v, 1, 1, 1)
    except ValueError as e:
        assert "gs must be a multiple of 8" in str(e)
    else:
        raise AssertionError("a malformed view was accepted")
    assert capi.load().w4_dispatch_mma_min_m() >= 1
    lib = capi.load()
    # one constant, lowered only for large matrices whose rows are not 16-byte aligned
    assert lib.w4_dispatch_mma_min_m_for(4096, 4096) == lib.w4_dispatch_mma_min_m()
    assert lib.w4_dispatch_mma_min_m_for(64, 4104) == lib.w4_dispatch_mma_min_m()
    assert lib.w4_dispatch_mma_min_m_for(11008, 4104) == 2
    assert lib.w4_dispatch_mma_min_m_for(4096, 11008) == 3
    assert lib.w4_dispatch_mma_min_m_for(4096, 4128) == 3
    assert lib.w4_dispatch_mma_min_m_for(4096, 6144) == 2
    assert lib.w4_dispatch_mma_min_m_for(11008, 4096) == 3
    assert lib.w4_dispatch_mma_min_m_for(8192, 4096) == lib.w4_dispatch_mma_min_m()
    assert lib.w4_dispatch_mma_min_m_for_gs(11008, 4096, 128) == 3
    assert lib.w4_dispatch_mma_min_m_for_gs(11008, 4096, 32) == 3
    assert lib.w4_dispatch_mma_min_m_for_gs(11008, 4096, 48) == lib.w4_dispatch_mma_min_m()
    assert lib.w4_dispatch_mma_min_m_for_gs(11008, 4104, 8) == 2
    assert lib.w4_dispatch_mma_min_m_for_mx(4096, 14336) == 2
    assert lib.w4_dispatch_mma_min_m_for_mx(4096, 8192) == 3
    assert lib.w4_dispatch_mma_min_m_for_mx(4096, 4096) == lib.w4_dispatch_mma_min_m()


def test_flash_plan_of_short_caches_shares_nothing():
    """Caches of up to 512 positions, and 512 slabs and more, on the matrix cores: one split per slab, so
    neither scratch nor arrival counters are touched and calls on several streams may overlap."""
    capi = w4amd.capi()
    for kind in (0, 1, 2):
        for D, gs in ((64, 32), (128, 32), (128, 128)):
            for H in (1, 8, 64, 300, 5000):
                for group in (1, 4, 16, 64):
                    for S in (1, 127, 128, 300, 384, 511, 512):
                        splits, length, direct, route = capi.flash_plan_for(kind, H, group, S, D, gs)
                        assert (splits, direct) == (1, 1) and length >= S and route >= 1, (kind, H, group, S, D)
            for H in (512, 520, 560, 608, 700, 1030):
                for S in (513, 1500, 4096, 6000, 32768):
                    assert capi.flash_plan_for(kind, H, 4, S, D, gs)[0] == 1, (kind, H, S, D, gs)
    for bad in [(3, 8, 1, 100, 128, 32), (1, 8, 65, 100, 128, 32), (1, 8, 1, 100, 128, 12), (1, 0, 1, 100, 128, 32),
                (0, 8, 1, 100, 128, 32, 16)]:
        with pytest.raises(ValueError):
            capi.flash_plan_for(*bad)


def test_flash_splits_of_grids_past_one_round():
    """260 to 325 slabs, a little more than one workgroup per compute unit, are split: with one each,
    most units would idle while a few work on two.  FP8 with D = 64: two workgroups per unit."""
    capi = w4amd.capi()
    for kind in (1, 2):
        for D in (64, 128):
            for H in (260, 288, 300, 325):
                for S in (4096, 8192):
                    assert capi.flash_plan_for(kind, H, 4, S, D, 64)[0] >= 2, (kind, D, H, S)
    assert capi.flash_plan_for(2, 16, 4, 32768, 64, 64)[:2] == (32, 1024)


def test_flash_long_splits_keep_tiles_in_registers():
    """Many tiles per wave go through registers: W4 and FP8 with D = 64 from 13 on, FP8 with D = 128 from 16
    on where no compute unit has two workgroups."""
    capi = w4amd.capi()
    seen = set()
    for kind, gs in ((1, 32), (2, 32), (2, 64)):
        for D in (64, 128):
            for H in (1, 16, 100, 256, 300, 512, 700):
                for S in (700, 1500, 1700, 1900, 2100, 4096, 8192, 20000, 32768):
                    splits, length, _, route = capi.flash_plan_for(kind, H, 4, S, D, gs)
                    tiles = length // 128
                    lds = tiles <= 12 if kind == 1 or D == 64 else tiles <= 15 or H * splits > 256
                    assert route == (2 if lds else 1), (kind, D, H, S, splits, length, route)
                    seen.add((kind, D, lds))
    assert len(seen) == 8


def test_flash_partials_stay_inside_the_fixed_scratch():
    """Calls whose partials fit the array of the entry that allocates nothing with fewer splits are not
    split beyond it (260 slabs x 16 heads: one split of 4096 positions)."""
    capi = w4amd.capi()
    for H, group, S, D in [(260, 16, 4096, 128), (88, 48, 1300, 64), (91, 64, 2048, 64), (300, 11, 4096, 128),
                           (200, 24, 1500, 128)]:
        splits = capi.flash_plan_for(1, H, group, S, D, 32)[0]
        assert H * group * splits * (D + 2) * 4 <= 4 << 20, (H, group, S, D, splits)


def test_flash_plan_of_many_heads():
    """More than 12 query heads per slab: from four splits on a kernel of its own merges them."""
    capi = w4amd.capi()
    for kind in (0, 1, 2):
        for S in (900, 1000, 1024, 2000, 5000, 16384):
            for H in (8, 37, 64, 71, 128, 200):
                for group in (4, 12, 13, 16, 19):
                    splits, _, one_launch, _ = capi.flash_plan_for(kind, H, group, S, 128, 32)
                    heads = min(group, 16)
                    assert one_launch == (splits == 1 or heads * splits <= (48 if heads > 12 else 64))


def test_flash_scale_dwords_end_with_their_array():
    """Tiles through LDS fetch row scales as dwords: caches whose scale arrays hold an odd number of
    halves (one group per row, odd slabs times odd positions) take the register kernels."""
    capi = w4amd.capi()
    for kind in (1, 2):
        for D in (64, 128):
            for H in (1, 2, 3, 5, 8):
                for S in (1, 77, 600, 601, 1500, 1501):
                    for gs in (D, D // 2, D // 4):
                        route = capi.flash_plan_for(kind, H, 1, S, D, gs)[3]
                        assert route == (1 if gs == D and H * S % 2 else 2), (kind, H, S, D, gs, route)


def test_mx_plan():
    """Which kernel multiplies two scaled operands: grids of few eight-wave tiles are left to the skinny
    kernel (4-bit X, N = 13824, K = 5120, M = 5: 10.7 us, with tiles 15.9)."""
    plan = w4amd.capi().gemm_mx_plan_for
    skinny = [(0, 5, 13824, 5120), (0, 16, 13824, 5120), (1, 7, 13824, 5120), (0, 1, 22016, 4096), (0, 37, 8192, 8192),
              (0, 83, 352, 5120), (0, 202, 528, 5120), (0, 127, 4096, 14336), (0, 16, 4096, 4096), (1, 1, 14336, 4096), (0, 5, 100, 1000)]
    assert [a for a in skinny if plan(*a) != 0] == []
    eight_waves = [(0, 33, 14336, 4096), (1, 8, 14336, 4096), (1, 64, 14336, 4096), (0, 17, 4096, 11008),
                   (0, 1, 28672, 4096), (1, 192, 14336, 4096), (0, 101, 4096, 4096)]
    assert [a for a in eight_waves if plan(*a) not in (1, 2, 3, 4)] == []
    # K a multiple of 256 and not of 512
    assert [plan(0, M, 20480, 2816) for M in (2, 3, 4, 5)] == [0, 1, 1, 1] and plan(0, 5, 13000, 2816) == plan(1, 7, 13000, 7424) == 0
    assert plan(0, 2048, 4096, 4096) == plan(1, 2048, 4096, 4096) == 8
    for bad in [(0, 0, 8, 64), (0, 8, 0, 64), (1, 8, 8, 0)]:
        with pytest.raises(ValueError):
            plan(*bad)


def test_gemm_plan_contracts():
    """Bad sizes and formats are refused before the device is asked for its compute units."""
    plan = w4amd.capi().gemm_plan_for
    for bad in [(0, 0, 8, 64), (0, 8, 0, 64), (1, 8, 8, 0), (3, 8, 8, 64), (-1, 8, 8, 64), (0, 8, 8, 64, 12), (1, 8, 8, 64, 0)]:
        with pytest.raises(ValueError):
            plan(*bad)
    if os.path.exists("/dev/kfd"):
        assert plan(0, 1, 64, 64, 32) == plan(2, 1, 64, 64) == 0
    else:
        with pytest.raises(RuntimeError):
            plan(0, 8, 64, 64, 32)


def test_quantize_contracts():
    """Malformed calls are rejected before the device is touched (pack.hpp:64-72,
    mx.hpp:71-76, kvcache.hpp:60-68, kvfp8.hpp:70-79)."""
    c = w4amd.capi()
    one = 8  # any non-null address: nothing is dereferenced
    for view, text in [(c.packed_view(0, 32, 8, 4, 1, one, one), "bad dims"),
                       (c.packed_view(2, 32, 12, 3, 1, one, one), "multiple of 8"),
                       (c.packed_view(2, 32, 8, 5, 1, one, one), "G inconsistent"),
                       (c.packed_view(2, 32, 8, 4, 0, one, one, 0), "asymmetric without zeros"),
                       (c.packed_view(2, 32, 8, 4, 1, one, one, one), "symmetric carries no zeros"),
                       (c.packed_view(2, 32, 8, 4, 1, 0, one), "null pointer")]:
        with pytest.raises(ValueError, match=text):
            c.quantize(view, one, one)
    with pytest.raises(ValueError, match="null pointer"):
        c.quantize(c.packed_view(2, 32, 8, 4, 1, one, one), one, 0)
    with pytest.raises(ValueError, match="B inconsistent"):
        c.quantize_mx(c.packed_mx_view(2, 64, 3, one, one), one, one)
    with pytest.raises(ValueError, match="bad dims"):
        c.quantize_mx(c.packed_mx_view(2, 0, 0, one, one), one, one)
    with pytest.raises(ValueError, match="multiple of 8"):
        c.quantize_cache(c.kv_view(1, 1, 64, 20, 4, 1, one, one, 0, one, one, 0), one, one, one)
    with pytest.raises(ValueError, match="asymmetric without zeros"):
        c.quantize_cache(c.kv_view(1, 1, 64, 16, 4, 0, one, one, 0, one, one, 0), one, one, one)
    with pytest.raises(ValueError, match="null pointer"):
        c.quantize_cache_f8(c.kv_f8_view(1, 1, 64, 16, 4, one, one, one, one), 0, one, one)
    with pytest.raises(ValueError, match="G inconsistent"):
        c.quantize_cache_f8(c.kv_f8_view(1, 1, 64, 16, 3, one, one, one, one), one, one, one)
    # W4A4: both views checked, K must agree
    w, x = c.packed_mx_view(8, 64, 2, one, one), c.packed_mx_view(2, 32, 1, one, one)
    with pytest.raises(ValueError, match="disagree on K"):
        c.gemm_mx_w4a4(w, x, one)
    with pytest.raises(ValueError, match="null pointer"):
        c.gemm_mx_w4a4(w, c.packed_mx_view(2, 64, 2, one, one), 0)
    with pytest.raises(ValueError, match="B inconsistent"):
        c.gemm_mx_w4a4(w, c.packed_mx_view(2, 64, 3, one, one), one)
    with pytest.raises(ValueError, match="null pointer"):
        c.quantize_mx_f16(c.packed_mx_view(2, 64, 2, one, one), 0, one)
    # W4A8
    x8 = c.act_mx8_view(2, 64, 2, 16, one)
    with pytest.raises(ValueError, match="disagree on K"):
        c.gemm_mx_w4a8(c.packed_mx_view(8, 32, 1, one, one), x8, one)
    with pytest.raises(ValueError, match="multiple of 32"):
        c.gemm_mx_w4a8(c.packed_mx_view(8, 40, 2, one, one), c.act_mx8_view(2, 40, 2, 16, one), one)
    with pytest.raises(ValueError, match="16-byte aligned"):
        c.gemm_mx_w4a8(w, c.act_mx8_view(2, 64, 2, 8, one), one)
    with pytest.raises(ValueError, match="B inconsistent"):
        c.gemm_mx_w4a8(w, c.act_mx8_view(2, 64, 3, 16, one), one)
    with pytest.raises(ValueError, match="null pointer"):
        c.quantize_mx8_f16(x8, 0, one)


def test_noalloc_entry_contracts_without_a_device():
    """The entry point that allocates nothing validates like w4_attention_w4_flash_gqa
    and rejects partials beyond its built-in array before any device call."""
    c = w4amd.capi()
    one = 256
    with pytest.raises(ValueError, match="null pointer"):
        c.attention_w4_flash_noalloc(c.kv_view(1, 64, 128, 32, 4, 1, one, one, 0, one, one, 0), 0, one)
    with pytest.raises(ValueError, match="G inconsistent"):
        c.attention_w4_flash_noalloc(c.kv_view(1, 64, 128, 32, 3, 1, one, one, 0, one, one, 0), one, one)
    with pytest.raises(ValueError, match="bad query group"):
        c.attention_w4_flash_noalloc(c.kv_view(1, 64, 128, 32, 4, 1, one, one, 0, one, one, 0), one, one, group=65)
    # 512 splits x 64 query heads x 130 floats = 17 MB of partials
    with pytest.raises(ValueError, match="exceed the built-in scratch"):
        c.attention_w4_flash_noalloc(c.kv_view(1, 1 << 19, 128, 32, 4, 1, one, one, 0, one, one, 0), one, one, group=64)


def test_native_calls_take_and_refuse_what_ctypes_does():
    """The callables behind the Python entry points: positional, keyword and missing arguments, None and wrong types, each
    against the ctypes function that stands behind (validation fails in every call: nothing reaches a device)."""
    capi = w4amd.capi()
    lib = capi.load()
    assert all(hasattr(getattr(capi, n), "__wrapped__") for n in capi._NATIVE)
    v, kv = capi.packed_view(2, 32, 7, 4, 1, 1, 1), capi.kv_f8_view(1, 1, 128, 7, 1, 1, 1, 1, 1)
    calls = [("gemm", (v, 1, 1, 1), {}), ("gemm", (v, 1, 1), {"M": 1, "stream": None}), ("gemm", (v, 1, 1), {}),
             ("gemm", (v, 1, 1, 1), {"M": 2}), ("gemm", (v, 1, 1, 1), {"other": 2}), ("gemm", (v, 1, 1, 1, 0, 0, 0), {}),
             ("gemm", (3, 1, 1, 1), {}), ("gemm", (kv, 1, 1, 1), {}), ("gemm", (v, 2.0, 1, 1), {}), ("gemm", (v, None, 1, 1), {}),
             ("gemm", (), {}), ("gemm", (v, 1, 1, "1"), {}), ("attention_f8_flash", (kv, 1, 1), {"scale_mode": 1, "group": 3}),
             ("quantize_cache_f8", (kv, 1, 1, 1), {"src_f16": True}), ("quantize_cache_f8", (kv, 1, 1), {"status": None}),
             ("attention_fp16_flash", (1, 1, 1, 1, 0, 1, 128), {"group": 0}),
             # None stands for a null address only
             ("gemm", (v, 1, 1, None), {}), ("gemm_mma", (v, 1, 1), {"M": None}), ("attention_f8_flash", (kv, 1, 1), {"scale_mode": None}),
             ("attention_f8_flash", (kv, 1, 1), {"group": None}), ("quantize_cache_f8", (kv, 1, 1, 1), {"src_f16": None}),
             ("attention_fp16_flash", (1, 1, 1, 1, None, 1, 128), {}), ("attention_fp16_flash", (1, 1, 1, 1, 1, 1, 128, None, None), {})]
    for name, args, options in calls:
        said = []
        for f in (getattr(capi, name), getattr(capi, name).__wrapped__):
            with pytest.raises(Exception) as e:
                f(*args, **options)
            said.append((e.type, str(e.value)))
        assert said[0] == said[1], (name, args, options)
    # arguments in the C functions' order: a validator that names what it found
    with pytest.raises(ValueError, match="group"):
        capi.attention_w4_flash(capi.kv_view(1, 64, 128, 32, 4, 1, 16, 16, 0, 16, 16, 0), 16, 16, group=-1)
    assert lib.w4_last_error()


def test_entry_points_without_the_native_callables():
    """No extension for this Python: every entry point is its ctypes call; and one built for another Python is not loaded."""
    capi = w4amd.capi()
    assert capi.CALLS_PATH.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and os.path.exists(capi.CALLS_PATH)
    code = ("import w4amd; c = w4amd.capi(); c.CALLS_PATH += '.absent'; lib = c.load()\n"
            "assert not any(hasattr(getattr(c, n), '__wrapped__') for n in c._NATIVE)\n"
            "try: c.gemm(c.packed_view(2, 32, 7, 4, 1, 1, 1), 1, 1, 1)\n"
            "except ValueError as e: print('refused:', e)\n")
    run = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.abspath(__file__)), capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout.startswith("refused:"), run.stderr


def test_native_callables_are_named_copied_and_pickled_as_functions_are():
    capi = w4amd.capi()
    capi.load()
    for n in capi._NATIVE:
        f, behind = getattr(capi, n), getattr(capi, n).__wrapped__
        assert (f.__name__, f.__qualname__, f.__module__, f.__doc__) == (n, n, behind.__module__, behind.__doc__)
        assert inspect.signature(f) == inspect.signature(behind)
        assert pickle.loads(pickle.dumps(f)) is f and copy.deepcopy(f) is f
