"""Split-S flash decode whose last workgroup of every slab merges the slab's splits
(csrc/flash_mfma.hip): numbers of splits and heads at the edges of the rule that chooses it
(64 splits and more, 64 (head, split) partials in one workgroup and more, several passes of 16
heads) for every kind of cache, called again and in between calls with other numbers of splits: the
arrival counters have to be back at zero after each.  The plan query pins the number of splits and
where they are merged.  kvflash.cuh:350-363 is the reference's entry for these shapes."""
import numpy as np
import pytest

import orc
import w4amd
from devutil import DevKV, DevKVF8, bits, halves, ptr, to_dev
from test_gpu_attention import _paged_pool

pytestmark = pytest.mark.gpu
TOL = 1e-3  # rel L2 against the FP64 oracle, as in test_gpu_attention.py
F16, W4, F8 = 0, 1, 2

# (cache, slabs, positions, head dim, query heads per slab, symmetric, page; splits, merged in place)
SHAPES = [(W4, 1, 16384, 128, 1, True, 0, 64, True),    # 64 splits, one per lane of the merging wave
          (W4, 8, 16384, 128, 1, True, 0, 64, True),    # the same for several slabs
          (W4, 1, 16793, 128, 4, False, 0, 66, False),  # more splits than that
          (W4, 1, 24000, 128, 1, False, 16, 63, True),
          (W4, 4, 4000, 128, 4, True, 0, 16, True),     # 64 partials per slab
          (W4, 4, 4000, 128, 5, False, 0, 32, False),   # more
          (W4, 4, 4000, 128, 4, True, 16, 16, True),
          (W4, 8, 600, 64, 7, True, 0, 5, True),        # few splits, heads that do not divide over the waves
          (W4, 80, 650, 128, 17, True, 0, 3, True),    # two passes over the heads, one after the other
          (W4, 60, 1000, 128, 19, True, 0, 4, False),   # more than 12 heads in a pass: up to three splits
          (W4, 130, 700, 128, 2, False, 48, 3, True),   # a slab count past one per compute unit and XCD round
          (F8, 1, 16384, 64, 1, True, 0, 64, True),
          (F8, 4, 4000, 128, 4, True, 0, 16, True),
          (F8, 4, 4000, 128, 5, True, 0, 32, False),
          (F8, 100, 600, 128, 17, True, 0, 3, True),
          (F16, 1, 16384, 128, 1, True, 0, 64, True),
          (F16, 4, 4000, 128, 4, True, 0, 32, False),
          (F16, 8, 600, 64, 7, True, 0, 5, True),
          (F16, 100, 600, 128, 17, True, 0, 3, True)]


class _Case:
    def __init__(self, i):
        self.c = c = w4amd.capi()
        self.kind, self.H, self.S, self.D, self.group, sym, self.page, splits, merged = SHAPES[i]
        H, S, D = self.H, self.S, self.D
        plan = c.flash_plan_for(self.kind, H, self.group, S, D, 32, self.page)
        assert (plan[0], plan[2]) == (splits, merged), plan
        k, v = orc.normal_weights(H * S * D, 71 + i), orc.normal_weights(H * S * D, 171 + i)
        if self.kind == F8:
            cache = orc.quantize_cache_f8(k, v, H, S, D, 32)
            self.kd, self.vd = orc.dequant_cache_f8(cache, False), orc.dequant_cache_f8(cache, True)
            self.dk = DevKVF8(cache)
        else:
            cache = orc.quantize_cache(k, v, H, S, D, 32, sym)
            self.kd, self.vd = orc.dequant_cache(cache, False), orc.dequant_cache(cache, True)
            if self.kind == F16:
                self.k16, self.v16 = to_dev(self.kd), to_dev(self.vd)
            elif self.page:
                self.npages = (S + self.page - 1) // self.page
                bt = np.random.default_rng(i).permutation(self.npages).astype(np.int32)
                self.keep, self.view = _paged_pool(cache, self.page, bt)
                self.bt = to_dev(bt)
            else:
                self.dk = DevKV(cache)
        self.q = orc.normal_activations(H * self.group * D, 271 + i)
        self.q_d = to_dev(self.q)

    def run(self):
        c, H, S, D, group = self.c, self.H, self.S, self.D, self.group
        out = halves(H * group * D, 0x7E00)
        if self.kind == F16:
            c.attention_fp16_flash(ptr(self.q_d), ptr(self.k16), ptr(self.v16), ptr(out), H, S, D, group=group)
        elif self.kind == F8:
            c.attention_f8_flash(self.dk.view, ptr(self.q_d), ptr(out), group=group)
        elif self.page:
            c.attention_w4_flash_paged_batched(self.view, ptr(self.bt), 1, self.npages, self.page, self.npages,
                                               group, ptr(self.q_d), ptr(out))
        else:
            c.attention_w4_flash(self.dk.view, ptr(self.q_d), ptr(out), group=group)
        return bits(out).copy()


@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_merge_in_place(i):
    a, b = _Case(i), _Case((i + 1) % len(SHAPES))
    runs = [x.run() for x in (a, b) * 3]  # three times each, in turn
    for r in (2, 4):
        assert np.array_equal(runs[r], runs[0]) and np.array_equal(runs[r + 1], runs[1])
    ref = orc.attention_f16(a.q, a.kd, a.vd, a.H, a.group, a.S, a.D)
    assert orc.rel_l2(runs[0].view(np.float16), ref) <= TOL


def test_entries_with_their_own_scratch_overlap():
    """The entry that allocates nothing and the other one keep their partials apart, so calls of the
    two may overlap on different streams: their arrivals have to be counted apart as well."""
    import torch
    c = w4amd.capi()
    H, S, D, group = 64, 3000, 128, 4
    c4 = orc.quantize_cache(orc.normal_weights(H * S * D, 81), orc.normal_weights(H * S * D, 82), H, S, D, 32, True)
    dk = DevKV(c4)
    qs = [to_dev(orc.normal_activations(H * group * D, 83 + i)) for i in range(2)]
    want = []
    for q in qs:
        out = halves(H * group * D, 0x7E00)
        c.attention_w4_flash(dk.view, ptr(q), ptr(out), group=group)
        want.append(bits(out).copy())
    entries = (c.attention_w4_flash, c.attention_w4_flash_noalloc)
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [[halves(H * group * D, 0x7E00) for _ in range(20)] for _ in range(2)]
    torch.cuda.synchronize()
    for n in range(20):
        for i in range(2):
            entries[i](dk.view, ptr(qs[i]), ptr(outs[i][n]), streams[i].cuda_stream, group=group)
    torch.cuda.synchronize()
    for i in range(2):
        for n in range(20):
            assert np.array_equal(bits(outs[i][n]), want[i]), (i, n)


def test_short_caches_overlap_on_two_streams():
    """One split per slab: no scratch, so calls of one entry may be in flight on several streams."""
    import torch
    c = w4amd.capi()
    H, S, D, group = 16, 512, 128, 4
    c4 = orc.quantize_cache(orc.normal_weights(H * S * D, 91), orc.normal_weights(H * S * D, 92), H, S, D, 32, True)
    dk = DevKV(c4)
    assert c.flash_plan_for(1, H, group, S, D, 32)[0] == 1
    qs = [to_dev(orc.normal_activations(H * group * D, 93 + i)) for i in range(2)]
    want = []
    for q in qs:
        out = halves(H * group * D, 0x7E00)
        c.attention_w4_flash(dk.view, ptr(q), ptr(out), group=group)
        want.append(bits(out).copy())
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [[halves(H * group * D, 0x7E00) for _ in range(20)] for _ in range(2)]
    torch.cuda.synchronize()
    for n in range(20):
        for i in range(2):
            c.attention_w4_flash(dk.view, ptr(qs[i]), ptr(outs[i][n]), streams[i].cuda_stream, group=group)
    torch.cuda.synchronize()
    for i in range(2):
        for n in range(20):
            assert np.array_equal(bits(outs[i][n]), want[i]), (i, n)


@pytest.mark.parametrize("H,S,D,group,splits", [(1, 2000, 64, 5, 16), (1, 8666, 64, 3, 68), (1, 33108, 64, 2, 130), (3, 2000, 128, 5, 16),
                                                (1, 8666, 128, 3, 68), (1, 16443, 128, 2, 129), (1, 64000, 128, 2, 250)])
def test_second_launch_that_merges(H, S, D, group, splits):
    """The kernel that merges what the last workgroup does not: fewer splits than waves times rows, one load a row and wave
    and more than that, one to four maxima a lane."""
    c = w4amd.capi()
    plan = c.flash_plan_for(F16, H, group, S, D, 32, 0)
    assert (plan[0], plan[2]) == (splits, 0), plan
    k, v = (orc.normal_activations(H * S * D, 91 + i) for i in range(2))
    q = orc.normal_activations(H * group * D, 93)
    k_d, v_d, q_d, out = to_dev(k), to_dev(v), to_dev(q), halves(H * group * D + 16, 0x7E00)
    runs = []
    for _ in range(2):
        c.attention_fp16_flash(ptr(q_d), ptr(k_d), ptr(v_d), ptr(out), H, S, D, group=group)
        runs.append(bits(out).copy())
    assert np.array_equal(*runs) and (runs[0][H * group * D:] == 0x7E00).all()
    ref = orc.attention_f16(q, k, v, H, group, S, D)
    assert orc.rel_l2(runs[0][: H * group * D].view(np.float16), ref) <= TOL


# D = 64: a wave of that kernel takes two splits at a time.  (cache, positions, query heads, page, splits): odd numbers of
# splits whose last one is held by a lane of the upper half (33 .. 63, 97 .. 127) or of the lower (65 .. 95, 129)
@pytest.mark.parametrize("kind,S,group,page,splits", [(F16, 4111, 4, 0, 33), (F16, 7954, 3, 0, 63), (F16, 8198, 2, 0, 65), (F16, 12346, 2, 0, 97),
                                                      (F16, 32293, 2, 0, 127), (F16, 32781, 2, 0, 129), (W4, 4111, 8, 0, 33), (W4, 14359, 4, 0, 57),
                                                      (W4, 4111, 8, 16, 33), (W4, 24607, 2, 0, 65), (F8, 10760, 3, 0, 43), (F8, 24607, 2, 0, 97)])
def test_second_launch_takes_an_odd_last_split(kind, S, group, page, splits):
    """The values of the last split are thirty times the others', so that its share of 1 / splits is a good part of the result."""
    c = w4amd.capi()
    D = 64
    plan = c.flash_plan_for(kind, 1, group, S, D, 32, page)
    assert (plan[0], plan[2]) == (splits, 0), plan
    k, v = orc.normal_weights(S * D, 95), orc.normal_weights(S * D, 96)
    v.reshape(S, D)[(splits - 1) * plan[1]:] *= 30
    q, out = orc.normal_activations(group * D, 97), halves(group * D + 16, 0x7E00)
    q_d = to_dev(q)
    if kind == F8:
        cache = orc.quantize_cache_f8(k, v, 1, S, D, 32)
        kd, vd = orc.dequant_cache_f8(cache, False), orc.dequant_cache_f8(cache, True)
        dk = DevKVF8(cache)
        c.attention_f8_flash(dk.view, ptr(q_d), ptr(out), group=group)
    else:
        cache = orc.quantize_cache(k, v, 1, S, D, 32, True)
        kd, vd = orc.dequant_cache(cache, False), orc.dequant_cache(cache, True)
        if kind == F16:
            k_d, v_d = to_dev(kd), to_dev(vd)
            c.attention_fp16_flash(ptr(q_d), ptr(k_d), ptr(v_d), ptr(out), 1, S, D, group=group)
        elif page:
            npages = (S + page - 1) // page
            bt = np.random.default_rng(S).permutation(npages).astype(np.int32)
            keep, view = _paged_pool(cache, page, bt)
            bt_d = to_dev(bt)
            c.attention_w4_flash_paged_batched(view, ptr(bt_d), 1, npages, page, npages, group, ptr(q_d), ptr(out))
        else:
            dk = DevKV(cache)
            c.attention_w4_flash(dk.view, ptr(q_d), ptr(out), group=group)
    got = bits(out)
    assert (got[group * D:] == 0x7E00).all()
    assert orc.rel_l2(got[: group * D].view(np.float16), orc.attention_f16(q, kd, vd, 1, group, S, D)) <= TOL


@pytest.mark.parametrize("S,D,group,splits", [(4200, 64, 5, 33), (4096, 64, 5, 32), (16443, 128, 2, 129), (8666, 128, 3, 68)])
def test_second_launch_keeps_infinities(S, D, group, splits):
    """Infinite values in the last split and in the first: their columns are infinite in the result, NaN comes from NaN alone."""
    c = w4amd.capi()
    plan = c.flash_plan_for(F16, 1, group, S, D, 32, 0)
    assert (plan[0], plan[2]) == (splits, 0), plan
    k, v, q = (orc.normal_activations(n * D, 98 + i) for i, n in enumerate((S, S, group)))
    k, q = ((a.view(np.float16) * np.float16(0.1)).view(np.uint16) for a in (k, q))
    rows = v.view(np.float16).reshape(S, D)
    rows[S - 2, 3], rows[7, 6], rows[S - 3, 9] = np.inf, -np.inf, np.nan
    k_d, v_d, q_d, out = to_dev(k), to_dev(v), to_dev(q), halves(group * D)
    c.attention_fp16_flash(ptr(q_d), ptr(k_d), ptr(v_d), ptr(out), 1, S, D, group=group)
    got = bits(out).view(np.float16).reshape(group, D)
    assert (got[:, 3] == np.inf).all() and (got[:, 6] == -np.inf).all() and np.isnan(got[:, 9]).all()
    others = np.delete(np.arange(D), [3, 6, 9])
    assert np.isfinite(got[:, others]).all()
