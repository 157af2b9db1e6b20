"""The kernels that wait for an operand in another assembly statement than the one that asked for it must
hold every register from one to the other: the build refuses one that spills, and the library that is
there has none (its own kernel metadata)."""
import pytest

from logismos_amd import build, kernels


def _kernels(path):
    """name -> metadata of every kernel in the code objects of a library (their AMDGPU notes: the sizes of
    name and description, type 32, the name, a msgpack map)"""
    msgpack = pytest.importorskip("msgpack")
    blob, out, at = open(path, "rb").read(), {}, 0
    while (at := blob.find(b"\x07\0\0\0", at)) >= 0:
        size = int.from_bytes(blob[at + 4:at + 8], "little")
        if blob[at + 8:at + 20] == b"\x20\0\0\0AMDGPU\0\0":
            note = msgpack.unpackb(blob[at + 20:at + 20 + size], strict_map_key=False)
            out.update((k[".name"], k) for k in note["amdhsa.kernels"])
        at += 4
    return out


def test_built_kernels_hold_what_is_in_flight():
    found = _kernels(kernels.LIB_PATH)
    for name in build.READS_IN_FLIGHT:
        mine = {k: v for k, v in found.items() if name in k}
        assert mine
        for k, v in mine.items():
            assert v[".vgpr_spill_count"] == 0 and v[".private_segment_fixed_size"] == 0, k


@pytest.mark.parametrize("kernel,refused", [("qgemm_q4g128_tallp_kernelILi2", 2), ("some_other_kernel", 0)])
def test_the_build_sees_a_spill(kernel, refused):
    remarks = "\n".join(f"a.hip:1:1: remark: {x} [-Rpass-analysis=kernel-resource-usage]" for x in (
        "Function Name: _ZN2lg23matmul_ring_fp16_kernelE", "    ScratchSize [bytes/lane]: 0",
        "    VGPRs Spill: 0", f"Function Name: _ZN2lg25{kernel}E", "    ScratchSize [bytes/lane]: 32",
        "    SGPRs Spill: 3", "    VGPRs Spill: 7"))
    assert len(build.spills(remarks)) == refused
