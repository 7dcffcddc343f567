"""Flash decode without hooks on every route a quantized cache can take (csrc/flash_mfma.hip): tiles
through LDS or through registers.  Both do the same arithmetic on the same values, so a call without
hooks returns the bytes of the hooked one, whose kernel always goes through registers; the
outputs stay within the oracle gate of test_gpu_attention.py.  The plan query pins the route and the
number of splits, so that a change of the cost rule cannot move a shape elsewhere unseen."""
import numpy as np
import pytest

import orc
import w4amd
from devutil import DevKV, DevKVF8, bits, f64, halves, ptr, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-3
LDS, REG = 2, 1


def _cache(kind, H, S, D, gs, sym, seed):
    rng = np.random.default_rng(seed)
    k, v = rng.standard_normal(H * S * D), rng.standard_normal(H * S * D)
    return orc.quantize_cache(k, v, H, S, D, gs, sym) if kind == 1 else orc.quantize_cache_f8(k, v, H, S, D, gs)


def _reference(kind, c, q, group):
    deq = orc.dequant_cache if kind == 1 else orc.dequant_cache_f8
    return orc.attention_f16(q, deq(c, False), deq(c, True), c.H, group, c.S, c.D)


# (kind 1 W4 / 2 FP8, slabs, positions, D, group size, heads per slab, symmetric, route)
ROUTES = [
    # several groups per row, short and long splits
    (2, 520, 1300, 128, 32, 1, True, LDS), (2, 600, 1100, 64, 64, 1, True, LDS), (2, 4, 700, 128, 32, 5, True, LDS),
    # one group per row: with an odd S every other slab's scales begin in the middle of a dword
    (2, 2, 77, 128, 128, 1, True, LDS), (2, 4, 601, 128, 128, 4, True, LDS), (2, 6, 1333, 64, 64, 2, True, LDS),
    (1, 4, 601, 128, 128, 4, True, LDS), (1, 2, 1333, 128, 128, 1, False, LDS), (1, 6, 77, 64, 64, 3, False, LDS),
    # an odd number of scales in all: no dword may end behind the array
    (2, 3, 77, 128, 128, 1, True, REG), (2, 5, 1501, 128, 128, 4, True, REG), (2, 1, 1, 64, 64, 1, True, REG),
    (1, 3, 601, 128, 128, 4, False, REG), (1, 1, 1333, 64, 64, 2, True, REG),
]


@pytest.mark.parametrize("case", ROUTES, ids=str)
def test_every_route_gives_the_hooked_bytes(case):
    kind, H, S, D, gs, group, sym, route = case
    capi = w4amd.capi()
    assert capi.flash_plan_for(kind, H, group, S, D, gs)[3] == route
    c = _cache(kind, H, S, D, gs, sym, 0x0DD + H * S)
    q = orc.normal_activations(H * group * D, 0x0DE + S)
    dk, q_d = (DevKV if kind == 1 else DevKVF8)(c), to_dev(q)
    call = capi.attention_w4_flash if kind == 1 else capi.attention_f8_flash
    n = H * group * D
    out, hooked, ko, vo = halves(n, 0x7E00), halves(n, 0x7E00), halves(H * S * D), halves(H * S * D)
    call(dk.view, ptr(q_d), ptr(out), group=group)
    call(dk.view, ptr(q_d), ptr(hooked), 0, ptr(ko), ptr(vo), group=group)
    assert np.array_equal(bits(out), bits(hooked))
    assert orc.rel_l2(f64(out), _reference(kind, c, q, group)) <= TOL


@pytest.mark.parametrize("H,S,D,group", [(1, 77, 128, 1), (3, 600, 128, 4), (5, 2001, 64, 2)])
def test_f8_scale_per_slab_odd_slabs(H, S, D, group):
    """Scales of an odd number of slabs, and scale arrays that begin two bytes past a dword."""
    capi = w4amd.capi()
    c = _cache(2, H, S, D, D, True, 0x51AB + S)
    rng = np.random.default_rng(S)
    slab = rng.uniform(0.002, 0.02, (2, H)).astype(np.float16).view(np.uint16)
    full = orc.KVCacheF8()
    full.__dict__.update(c.__dict__)
    full.s_k, full.s_v = np.repeat(slab[0], S * c.G), np.repeat(slab[1], S * c.G)
    q = orc.normal_activations(H * group * D, 0x51AC)
    ref, q_d, n = _reference(2, full, q, group), to_dev(q), H * group * D
    got = []
    for shift in (0, 1):  # halves in front of the scales
        d8 = DevKVF8(c, np.concatenate([np.full(shift, 0x7E00, np.uint16), slab[0]]),
                     np.concatenate([np.full(shift, 0x7E00, np.uint16), slab[1]]))
        d8.view.s_k, d8.view.s_v = ptr(d8.t[1]) + 2 * shift, ptr(d8.t[3]) + 2 * shift
        out = halves(n, 0x7E00)
        capi.attention_f8_flash(d8.view, ptr(q_d), ptr(out), group=group, scale_mode=1)
        got.append(bits(out).copy())
        assert orc.rel_l2(f64(out), ref) <= TOL
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("kind,H,S,D,gs", [(1, 4, 700, 128, 32), (2, 4, 700, 128, 128), (2, 8, 1301, 64, 32)])
def test_scales_off_dwords(kind, H, S, D, gs):
    """Row scales that begin two bytes past a dword: the register kernels, same bytes."""
    capi = w4amd.capi()
    c = _cache(kind, H, S, D, gs, True, 0x0FF + S)
    q = orc.normal_activations(H * 2 * D, 0x0FE)
    q_d, n = to_dev(q), H * 2 * D
    call = capi.attention_w4_flash if kind == 1 else capi.attention_f8_flash
    got = []
    for shift in (0, 1):
        dk = (DevKV if kind == 1 else DevKVF8)(c)
        pad = np.full(shift, 0x7E00, np.uint16)
        s_k, s_v = to_dev(np.concatenate([pad, np.ravel(c.s_k)])), to_dev(np.concatenate([pad, np.ravel(c.s_v)]))
        dk.view.s_k, dk.view.s_v = ptr(s_k) + 2 * shift, ptr(s_v) + 2 * shift
        out = halves(n, 0x7E00)
        call(dk.view, ptr(q_d), ptr(out), group=2)
        got.append(bits(out).copy())
    assert np.array_equal(got[0], got[1])
    assert orc.rel_l2(got[0].view(np.float16), _reference(kind, c, q, 2)) <= TOL
