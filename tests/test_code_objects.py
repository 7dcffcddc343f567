"""What the compiler says about every kernel of the built library (the metadata notes of
its code objects; nothing is disassembled).

No kernel may use scratch memory: an instantiation that spills registers runs several
times slower than the next smaller one that fits (a scale pick that the compiler put in
scratch cost 1.8 us of a 10.5 us call once), so the launchers cap what they ask for at
what fits and do not compile the rest -- this test is what keeps the two in step.  The
kernels that write registers with hand-placed loads and waits must not have
any of them parked in the AGPR half of the register file either: the compiler does not
know when such a register lands, and a copy made before the wait copies stale bits."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "w4a16-dequant-gemm_amd"))
import codeobj  # noqa: E402

LIB = codeobj.default_lib()


@pytest.fixture(scope="module")
def kernels():
    assert os.path.exists(LIB), "libw4amd.so is not built (python __graft_entry__.py)"
    ks = codeobj.kernels(LIB)
    assert len(ks) > 100, "the code objects of the library were not found"
    return ks


def _demangle(names):
    try:
        out = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True).stdout
        return out.split("\n")[:len(names)]
    except OSError:
        return names


def test_every_kernel_is_gfx950(kernels):
    assert {k["target"].split("-")[-1] for k in kernels} == {"gfx950"}


def test_no_kernel_uses_scratch_memory(kernels):
    # (.vgpr_spill_count also counts registers the compiler parks in AGPRs, which costs a
    # copy and no memory traffic; what is policed here is the per-lane scratch segment)
    bad = [k for k in kernels if k.get(".private_segment_fixed_size", 0)]
    names = _demangle([k[".name"] for k in bad])
    assert not bad, "kernels with scratch memory:\n" + "\n".join(
        "%5d B, %d spilled VGPRs: %s" % (k[".private_segment_fixed_size"], k.get(".vgpr_spill_count", 0), n)
        for k, n in zip(bad, names))


def test_asm_loaded_registers_are_never_parked(kernels):
    """(also flash decode with tiles through LDS: query rows and slab scales are loaded ahead of the wait
    that covers them)"""
    rows4 = [k for k in kernels if "simt_rows4_kernel" in k[".name"]]
    flash = [k for k in kernels if re.search(r"flash_mfma_phase1ILi\dELi\d+ELb\dELi\dELb\dELb1EE", k[".name"])]
    assert rows4, "the four-rows vector kernel is missing from the library"
    assert len(flash) == 12, "W4 contiguous and paged, FP8; two head dimensions; two scale / zero-point forms"
    bad = [k for k in rows4 + flash if k.get(".agpr_count", 0) or k.get(".vgpr_spill_count", 0)]
    assert not bad, "\n".join(_demangle([k[".name"] for k in bad]))


def test_flash_kernels_without_hooks_for_every_route(kernels):
    """Calls without hooks run kernels without them: through registers for every cache kind (FP16,
    W4, FP8), head dimension and scale / zero-point form, through LDS for the quantized kinds."""
    names = [k[".name"] for k in kernels if "flash_mfma_phase1" in k[".name"]]
    for kind in (0, 1, 2):
        for D in (64, 128):
            for alt in ((0,) if kind == 0 else (0, 1)):
                for lds in ((0,) if kind == 0 else (0, 1)):
                    tag = "flash_mfma_phase1ILi%dELi%dELb0ELi0ELb%dELb%dEE" % (kind, D, alt, lds)
                    assert any(tag in n for n in names), tag


def test_wave64_and_workgroup_sizes(kernels):
    for k in kernels:
        assert k[".wavefront_size"] == 64
        assert k[".max_flat_workgroup_size"] <= 1024
        assert k.get(".group_segment_fixed_size", 0) <= 160 * 1024


def test_direct_to_lds_loads_wait_for_m0():
    """A load to LDS takes its address from M0, which needs one wait state between a scalar write and the load on
    this architecture: the compiler puts an s_nop between its own, and knows nothing of the ones inside an asm."""
    csrc = os.path.join(ROOT, "w4a16-dequant-gemm_amd", "csrc")
    found = 0
    for name in sorted(os.listdir(csrc)):
        text = open(os.path.join(csrc, name)).read()
        for m in re.finditer(r"s_\w+ m0, %\d(?:, %\d)?(.{0,20})", text):
            assert m.group(1).startswith("\\n\\ts_nop 0\\n"), (name, m.group(0))
            found += 1
    assert found >= 13
