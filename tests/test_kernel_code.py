"""What the compiler made of the kernels, read from the built library's own gfx950 code objects: registers and
scratch memory.  A thread's elements live in registers only while every loop over them unrolls in time; one that
does not leaves them in scratch memory, silently, with the same results at a fraction of the speed."""
import os
import re
import struct
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel name with template arguments: {".vgpr_count": ..., ...}} of every code object in the library, with the
    path of that code object as "object"."""
    import pfa_native as P

    P.lib()
    blob = open(P.LIB_PATH, "rb").read()
    out = {}
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", blob, at + len(magic))
        entry = at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, entry)
            triple = blob[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if "gfx950" in triple and size:
                path = tmp_path_factory.mktemp("code") / "object"
                path.write_bytes(blob[at + offset:at + offset + size])
                notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(path)], check=True,
                                       capture_output=True, text=True).stdout
                for block in re.split(r"\n  - (?=\.)", notes)[1:]:
                    fields = dict(re.findall(r"^ {0,4}(\.\w+): +(\S+)$", block, re.M))
                    if ".private_segment_fixed_size" in fields:
                        out[fields[".name"]] = {**fields, "object": str(path)}
        at = blob.find(magic, at + 1)
    names = subprocess.run(["c++filt"], input="\n".join(out), check=True,
                           capture_output=True, text=True).stdout.split("\n")
    plain = [re.sub(r"pfa::|\(anonymous namespace\)::|^void ", "", n).split("(")[0] for n in names]
    out = {p: f for p, f in zip(plain, out.values())}
    assert len(out) > 100
    return out


@pytest.mark.parametrize("kernel", ["ntt_fwd_rows<8, 9, 8, false>", "ntt_inv_rows<8, 9, 8>",
                                    "ntt_inv_rows_staged<8, 9, 8, false>", "ntt_fwd_cols<8, 9>", "ntt_inv_cols<8, 9>", "k_epi_rows<8, 9>",
                                    "k_inner_ws<8, 9>"])
def test_largest_ring_elements_in_registers(kernels, kernel):
    """N = 2^17: 32 elements a thread (64 sums in the inner product), the longest unrolled loops."""
    assert int(kernels[kernel][".private_segment_fixed_size"]) == 0


def _instructions(kernel):
    text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn",
                           "--disassemble-symbols=" + kernel[".name"], kernel["object"]], check=True,
                          capture_output=True, text=True).stdout
    return [line.split("//")[0].split() for line in text.split("\n") if line.startswith("\t")]


@pytest.mark.parametrize("ring", ["7, 7", "7, 8", "8, 8", "8, 9"])
def test_wide_conversions_keep_loads_in_flight(kernels, ring):
    """The 128-bit sums of more than seven inputs: residues are requested in groups of eight, not one by one with a wait
    for each (an eight-input conversion then waits for memory 16 times an input instead of twice)."""
    alone = run = 0
    for op in _instructions(kernels["k_bconv_cols<%s, 2>" % ring]):
        if op[0] == "global_load_dwordx2":
            run += 1
        elif op[0] == "s_waitcnt" and "vmcnt" in " ".join(op):
            alone += run == 1
            run = 0
    assert alone < 8


@pytest.mark.parametrize("kernel", ["ntt_fwd_rows<6, 7, 32, false>", "ntt_fwd_rows<7, 7, 32, false>",
                                    "ntt_fwd_rows<7, 8, 8, true>", "ntt_fwd_rows<8, 8, 8, true>"])
def test_forward_rows_occupancy(kernels, kernel):
    """The forward rows pass of large batches: four waves on each of a CU's SIMDs (512 registers a lane, 160 KiB of LDS a
    CU), integer primes or not."""
    k = kernels[kernel]
    waves = int(k[".max_flat_workgroup_size"]) // 64
    assert 16 // waves * int(k[".group_segment_fixed_size"]) <= 160 * 1024
    assert int(k[".vgpr_count"]) <= 128


@pytest.mark.parametrize("kernel", ["ntt_fwd_cols<6, 7>", "ntt_fwd_rows<6, 7, 32, false>",
                                    "ntt_fwd_rows<6, 7, 32, true>", "ntt_inv_rows<6, 7, 32>",
                                    "ntt_inv_rows_staged<6, 7, 32, true>", "ntt_inv_cols<6, 7>",
                                    "ntt_inv_cols<8, 8>"])
def test_persistent_loops_keep_the_grid_size(kernels, kernel):
    """The loop over tiles reads no launch argument between two tiles: its step, the grid's size, is in a register (the
    one-word scalar loads; the tables a tile reads have entries of two words and more)."""
    ops = [op[0] for op in _instructions(kernels[kernel])]
    assert "s_load_dword" not in ops[ops.index("s_barrier"):]


@pytest.mark.parametrize("ring", ["6, 7", "7, 7", "7, 8", "8, 8", "8, 9"])
@pytest.mark.parametrize("kind", [0, 1])
def test_conversions_in_registers(kernels, ring, kind):
    """Single inputs and sums of 30-bit limbs fit the registers of four waves a SIMD with nothing spilled: a spilled
    value, reloaded once an item, waits behind the stores of the item before."""
    k = kernels["k_bconv_cols<%s, %d>" % (ring, kind)]
    assert int(k[".private_segment_fixed_size"]) == 0
    assert int(k[".vgpr_count"]) <= 128
