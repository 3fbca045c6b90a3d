"""Register and LDS use of the compiled kernels, read from the code-object notes of libfa8.so (no GPU): a vector register spilled to scratch costs memory
traffic in every step of a loop, and the shared-rows kernel of the wide head dims sits close to the 256 registers of a lane."""
import os
import re
import struct
import subprocess

import pytest

import cutlass_flash_atten_fp8_amd as fa

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects bundled in a shared library (one bundle per source file)."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if "gfx950" in triple and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


def kernel_notes(tmp_path, key):
    """{mangled kernel name: the number that its code object notes under .key}"""
    kernels = {}
    for i, blob in enumerate(code_objects(fa.LIBFA8_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(blob)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        names = re.findall(r"^\s+\.name:\s+(_Z\S+)$", notes, re.M)
        values = re.findall(rf"\.{key}:\s+(\d+)", notes)
        assert len(names) == len(values)
        kernels.update(zip(names, map(int, values)))
    return kernels


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_no_kernel_spills_vector_registers(tmp_path):
    kernels = kernel_notes(tmp_path, "vgpr_spill_count")
    for part in ("fa8_fwd_kernel", "fa8_shared_rows_kernel", "fa8_split_fused_kernel", "fa8_split_logits_kernel", "fa8_split_values_kernel"):
        assert any(part in n for n in kernels), part
    assert {n: s for n, s in kernels.items() if s} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_registers_leave_room_for_the_workgroups_that_the_plan_counts_on(tmp_path):
    """Two tiles a workgroup, two wavefronts a tile, head dims 32 and 64, sums together: four workgroups a compute unit, 128 registers a lane (three took up
    to 1.15 of the time).  Head dim 32 in the unshared loop: five, 96."""
    kernels = kernel_notes(tmp_path, "vgpr_count")
    for pattern, count, most in ((r"shared_rows_kernelILi(32|64)ELb[01]ELb[01]ELi2ELi2ELi[12]ELb0E", 12, 128), (r"fwd_kernelILi32E", 16, 96)):
        found = {n: v for n, v in kernels.items() if re.search(pattern, n)}
        assert len(found) == count and {n: v for n, v in found.items() if v > most} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_split_keys_in_one_kernel_hold_no_lds_that_their_ranges_do_not_need(tmp_path):
    """Every workgroup holds its ring of two tiles a wavefront and 2 KB; LDS for the logits is asked for by length at the launch, so that a
    call with short ranges does not need compute units that are empty."""
    lds = {n: x for n, x in kernel_notes(tmp_path, "group_segment_fixed_size").items() if "fa8_split_fused_kernel" in n}
    assert len(lds) == 8 * 4
    for name, x in lds.items():
        d = int(re.search(r"kernelILi(\d+)E", name)[1])
        row = 32 if d <= 32 else 64 if d <= 64 else 128 if d <= 128 else 256
        assert x <= 2 * 4 * 64 * row + 2048, name


OBJDUMP = os.path.join(os.path.dirname(READELF), "llvm-objdump")


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs llvm-objdump")
def test_outputs_are_kept_for_the_kernel_that_reads_them(tmp_path):
    """No store is non-temporal: the reader of O would find it in HBM (a copy right after the call then loses more than the call gains)."""
    stores = 0
    for i, blob in enumerate(code_objects(fa.LIBFA8_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(blob)
        listing = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], stdout=subprocess.PIPE, text=True)
        for line in listing.stdout:
            if "global_store_" in line:
                stores += 1
                assert " nt" not in line.split("//")[0], line
        assert listing.wait() == 0
    assert stores > 0
