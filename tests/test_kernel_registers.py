"""What the compiler made of kernels whose speed hangs on it: the register counts in the code objects of the built library."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from mojo_amd import _lib
from mojo_amd.build import HIPCC

LLVM = os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "llvm", "bin")
READELF, OBJCOPY = os.path.join(LLVM, "llvm-readelf"), os.path.join(LLVM, "llvm-objcopy")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled kernel name: (vector registers, spilled vector registers)}"""
    if not (os.path.exists(_lib.LIB_PATH) and os.path.exists(READELF) and os.path.exists(OBJCOPY) and shutil.which("c++filt")):
        pytest.skip("needs the built library, llvm-readelf, llvm-objcopy and c++filt")
    tmp = tmp_path_factory.mktemp("code")
    fat = tmp / "fat.bin"
    subprocess.run([OBJCOPY, "--dump-section", f".hip_fatbin={fat}", _lib.LIB_PATH, str(tmp / "rest")], check=True)
    data = fat.read_bytes()
    names, counts = [], []
    for at in (m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):  # one bundle per source file
        (entries,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" not in target or not size:
                continue
            obj = tmp / "kernel.o"
            obj.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
            for block in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
                names.append(re.search(r"\n    \.name:\s+(\S+)", block).group(1))
                counts.append(tuple(int(re.search(rf"\.{key}:\s+(\d+)", block).group(1)) for key in ("vgpr_count", "vgpr_spill_count")))
    plain = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout.split("\n")
    assert len(names) > 100
    return {re.sub(r"\(anonymous namespace\)::|qmm::|^void ", "", n).split("(")[0]: c for n, c in zip(plain, counts)}


@pytest.mark.parametrize("rows,lhs", [(1, "float"), (1, "unsigned short"), (2, "float")])
def test_act_order_look_up_keeps_its_table_reads_in_flight(kernels, rows, lhs):
    """Each weight waits for a chain of its own (group, table, product).  With 62 .. 75 registers the reads of eight weights overlap; a body that
    the compiler schedules one weight at a time takes 23 .. 27 and 14336 x 4096 with one bf16 row 19.1 us instead of 13.6."""
    found = [c for name, c in kernels.items() if re.match(rf"gemv_gptq_act_order_kernel<{rows}, true, .*{lhs}>$", name)]
    assert found and all(registers >= 56 and spilled == 0 for registers, spilled in found), found


def test_direct_and_shared_gemms_keep_their_sums_in_registers(kernels):
    """Their accumulators, operands and read-ahead are sized to the 256 registers of a wavefront.  Two plans (Q4_0 and Q6_K with fp32 rows) give up
    to seven registers to scratch outside the loop; an fp32 Q6_K body with a flush every four units spilled 30 and was 22 % slower."""
    found = {name: spilled for name, (_, spilled) in kernels.items() if re.match(r"gemm_(direct|shared)_kernel<", name)}
    assert len(found) > 60
    assert {name: spilled for name, spilled in found.items() if spilled > 8} == {}


def test_staged_gemm_keeps_its_sums_in_registers(kernels):
    """Up to 128 rows a wavefront fit 256 registers only because its loads hold none; a body that spilled 12 took twice the time."""
    found = {name: spilled for name, (_, spilled) in kernels.items() if name.startswith("gemm_staged_kernel<")}
    assert len(found) > 50
    assert {name: spilled for name, spilled in found.items() if spilled} == {}


def test_lhs_preparation_leaves_room_for_a_second_row(kernels):
    """Workgroups of 1024 threads: with more than 64 registers a compute unit holds one of them, 66 made thousands of long fp32 rows slower."""
    found = {name: c for name, c in kernels.items() if name.startswith("direct_prep_kernel<")}
    assert len(found) == 6
    assert {name: c for name, c in found.items() if c[0] > 64 or c[1]} == {}


def test_direct_gemm_of_gptq_runs_three_wavefronts_a_simd(kernels):
    """Two fragments of columns side by side, bf16 rows: up to 168 registers.  With 170 two wavefronts fit, and 10512 x 2304 with 349 rows took 44.8 us instead of 40.8."""
    (registers, spilled), = [c for name, c in kernels.items() if name == "gemm_direct_kernel<3, 8, 1, 2, 4, false>"]
    assert registers <= 168 and spilled == 0


def test_rms_normalisation_holds_values_not_addresses(kernels):
    """A value and its gamma for each of a thread's places in the row, and one offset: pointers for every load took 136, 236 and 400 registers for 16, 32 and 64 places."""
    found = {name: c for name, c in kernels.items() if name.startswith("rmsnorm_kernel<")}
    assert len(found) == 12
    for name, (registers, spilled) in found.items():
        held = int(re.search(r", (\d+), (?:true|false)>", name).group(1))
        assert registers <= 2 * held + 40 and spilled == 0, name


def test_grouped_q6_k_with_one_or_two_rows_is_not_packed_into_fewer_registers(kernels):
    """A launch has four wavefronts a SIMD; packed into the 80 registers of six, 4096 | 1024 | 1024 x 4096 with two bf16 rows took 8.4 us instead of 7.8."""
    found = [c for name, c in kernels.items() if re.match(r"gemv_kquant_small_mats_kernel<2, [12], unsigned short, 1>", name)]
    assert len(found) == 2 and all(84 <= registers <= 128 and spilled == 0 for registers, spilled in found), found
