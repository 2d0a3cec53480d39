"""What the library's own sources compile to, read from their AMD assembly; no GPU. The hand-written loads into LDS beside the
compiler's own: both take their LDS address from m0, so each must know of the other's. And phase 2's partial sums: lanes
exchange them through LDS behind the workgroup's barrier only."""
import re
import shutil
import subprocess

import pytest

from shrike_amd import capi
from tests.conftest import ROOT

FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "--cuda-device-only", "-S", "-w"]
KERNEL = """
#include "prefill_common.h"
using namespace shrike;
__global__ void k(const uint32_t *p, uint32_t *out) {
    __shared__ uint32_t a[64], b[256];
    auto into_a = [&](const uint32_t *q) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(q + threadIdx.x),
                                         (__attribute__((address_space(3))) void *)a, 4, 0, 0);
    };
    into_a(p);
    LOAD;
    into_a(p + 512);
    wait_loads_and_sync<0>();
    out[threadIdx.x] = a[threadIdx.x] + b[threadIdx.x];
}
"""
LDS_B = "uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)b))"


@pytest.mark.parametrize("load", [f"lds_load16({LDS_B}, p + 64 + 4 * threadIdx.x)", f"lds_load16({LDS_B}, p, 256 + 16 * threadIdx.x)"])
def test_the_compiler_knows_what_m0_holds_after_a_hand_written_load(tmp_path, load):
    source = tmp_path / "k.hip"
    source.write_text(KERNEL.replace("LOAD", load))
    subprocess.run(["/opt/rocm/bin/hipcc", *FLAGS, f"-I{ROOT}/shrike_amd/csrc", str(source), "-o", str(tmp_path / "k.s")], check=True)
    m0 = None
    addresses = []  # of the loads, in program order
    for line in (tmp_path / "k.s").read_text().splitlines():
        if written := re.search(r"s_mov\w* m0, (.+)", line):
            m0 = written.group(1)
        elif "global_load_lds" in line:
            addresses.append(m0)
    assert len(addresses) == 3
    assert addresses[0] == addresses[2] != addresses[1], f"the loads' LDS addresses: {addresses}"


@pytest.mark.parametrize("instance", ["4, 1, 2, true, 8, false, SHRIKE_META_F16, 16", "8, 1, 4, false, 8, false, SHRIKE_META_BF16, 32",  # rows that share a wave load
                                      "4, 1, 1, true, 8, false, SHRIKE_META_F16, 2", "8, 1, 4, false, 16, false, SHRIKE_META_BF16, 64",
                                      "8, 3, 4, true, 4, false, SHRIKE_META_BF16, 64", "4, 1, 4, false, 16, true, SHRIKE_META_F16, 64"])
def test_phase_2_reads_no_partial_sum_ahead_of_its_barrier(tmp_path, instance):
    """A lane's word of LDS is another lane's only behind the barrier: nothing else orders the two for the compiler."""
    with open(f"{ROOT}/shrike_amd/csrc/decode_phase2.hip") as f:
        text = f.read()
    source = tmp_path / "k.hip"
    source.write_text(text[:text.index("template <int BITS, int NCH>\n__global__ __launch_bounds__(256) void k_gemv")] +
                      f"template __global__ void k_phase2<{instance}>(Phase2Args);\n}}\n")
    subprocess.run(["/opt/rocm/bin/hipcc", *FLAGS, f"-I{ROOT}/shrike_amd/csrc", str(source), "-o", str(tmp_path / "k.s")], check=True)
    code = (tmp_path / "k.s").read_text().split("s_barrier")
    assert len(code) == 2 and re.search(r"\bds_write", code[0]) and re.search(r"\bds_read", code[1])
    assert not re.search(r"\bds_read", code[0]), "a partial sum is read ahead of the barrier"


def test_no_load_into_lds_reads_a_base_that_a_vector_instruction_has_just_written(tmp_path):
    """The library's own device code. A memory instruction that reads a scalar register needs five wait states behind a vector
    instruction that writes it (v_readlane of a spilled base), and the compiler keeps none ahead of assembly by hand. So the base of every
    such load is the scalar unit's own move, right ahead of it, and what stands between a write of m0 and the load is that or a wait state."""
    library = shutil.copy(capi.LIB_PATH, tmp_path)
    subprocess.run(["/opt/rocm/llvm/bin/llvm-objdump", "--offloading", library], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    loads = {"base": 0, "off": 0}
    for image in tmp_path.glob("*gfx950"):
        before = ""
        for line in subprocess.run(["/opt/rocm/llvm/bin/llvm-objdump", "-d", "--no-show-raw-insn", image], check=True, capture_output=True, text=True).stdout.splitlines():
            if "global_load_lds_dwordx" in line:
                base = re.search(r"(s\[\d+:\d+\])(?: nt)?\s", line)
                loads["base" if base else "off"] += 1
                assert f"s_mov_b64 {base[1]}, s[" in before if base else "s_nop" in before, f"{before.strip()} / {line.strip()}"
            before = line
    assert min(loads.values()) > 0
