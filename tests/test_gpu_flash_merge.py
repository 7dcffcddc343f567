"""Split-S flash decode whose last workgroup of every slab merges the slab's splits
(csrc/flash_mfma.hip): numbers of splits and heads at the edges of the rule that chooses it
(2 and 64 splits, 64 (head, split) partials in one workgroup, just past both, several passes of 16
heads), called again and in between calls with other numbers of splits: the arrival counters have
to be back at zero after each.  kvflash.cuh:350-363 is the reference's entry for these shapes."""
import numpy as np
import pytest

import orc
import w4amd
from devutil import DevKV, bits, halves, ptr, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-3  # rel L2 against the FP64 oracle, as in test_gpu_attention.py

# (slabs, positions, head dim, query heads per slab, symmetric)
SHAPES = [(1, 16384, 128, 1, True),    # 64 splits, one per lane of the merging wave
          (1, 17000, 128, 1, False),   # more splits than that: the merge kernel
          (4, 4000, 128, 4, True),     # 64 partials per slab
          (4, 4000, 128, 5, False),    # more
          (8, 600, 64, 7, True),       # few splits, heads that do not divide over the waves
          (2, 1000, 128, 19, True),    # two passes over the heads, one merged in place, one not
          (130, 700, 128, 2, False)]   # a slab count past one per compute unit and XCD round


@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_merge_in_place(i):
    c = w4amd.capi()
    cases = []
    for j in (i, (i + 1) % len(SHAPES)):
        H, S, D, group, sym = SHAPES[j]
        c4 = orc.quantize_cache(orc.normal_weights(H * S * D, 71 + j), orc.normal_weights(H * S * D, 171 + j),
                                H, S, D, 32, sym)
        cases.append((c4, orc.normal_activations(H * group * D, 271 + j), group))
    runs = []
    for c4, q, group in cases * 3:  # three times each, in turn
        out = halves(c4.H * group * c4.D, 0x7E00)
        dk, q_d = DevKV(c4), to_dev(q)
        c.attention_w4_flash(dk.view, ptr(q_d), ptr(out), group=group)
        runs.append(bits(out).copy())
    for r in (2, 4):
        assert np.array_equal(runs[r], runs[0]) and np.array_equal(runs[r + 1], runs[1])
    c4, q, group = cases[0]
    ref = orc.attention_f16(q, orc.dequant_cache(c4, False), orc.dequant_cache(c4, True), c4.H, group, c4.S, c4.D)
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
