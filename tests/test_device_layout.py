"""What the kernels assume of their LDS layout and of the order of LDS accesses, checked without a GPU by
compiling small probes of the kernels' headers (periodsearch_amd/csrc)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "periodsearch_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

pytestmark = pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")


def compile_probe(tmp_path, body, *flags):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.out"
    src.write_text('#include <hip/hip_runtime.h>\n#include <cmath>\n#include <cstddef>\n'
                   f'#include "{ROOT}/include/periodsearch_amd.h"\n#include "{CSRC}/ps_fit2.h"\n' + body)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++20", "-w", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", *flags, str(src), "-o", str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


def test_buffers_of_x_start_on_16_bytes(tmp_path):
    """orbit_loop stores and orbit_correct loads 16 bytes a lane at rows + {0, 64 pitches} + {0, kXBytes}."""
    compile_probe(tmp_path, """
constexpr size_t rows = offsetof(psk::Shared2<psk::kMaxFac>, u);
static_assert(rows % 16 == 0);
static_assert((rows + 64 * psk::kJP * sizeof(double)) % 16 == 0 && psk::kXBytes % 16 == 0);
static_assert(offsetof(psk::Shared2<psk::kMaxFac>, tab) % 16 == 0);
static_assert(2 * sizeof(psk::Shared2<psk::kMaxFac>) <= 160 * 1024);
""", "--cuda-host-only", "-fsyntax-only")


def fences_around_lds(ir, kernel):
    """The LDS accesses of a kernel's IR in order: 'w', 'r' and 'F' for a wavefront fence."""
    body = ir[ir.index(f"@{kernel}("):]
    body = body[:body.index("\n}")]
    seq = []
    for line in body.split("\n"):
        if 'fence syncscope("wavefront' in line:
            seq.append("F")
        elif re.search(r"\bstore <4 x i32>", line) and "addrspace(3)" in line:
            seq.append("w")
        elif re.search(r"\bload <8 x bfloat>", line) and "addrspace(3)" in line:
            seq.append("r")
    return "".join(seq)


def test_x_is_fenced_between_lanes(tmp_path):
    """A lane reads the X of other lanes of its wave: a fence lies between the stores and the loads, and between
    the loads and the next piece's stores."""
    out = compile_probe(tmp_path, """
extern "C" __global__ void probe(const psk::orb_u4 *corr, int norb, int cnt, double *res) {
    __shared__ __attribute__((aligned(16))) char x[psk::kXBytes];
    psk::OrbAcc<3, false> A;
    A.clear();
    psk::orbit_correct<3, false>(corr, norb, 0, cnt, x, A);
    for (int j = 0; j < 16; ++j) res[16 * threadIdx.x + j] = A.c[j];
}
""", "--cuda-device-only", "-O1", "-S", "-emit-llvm")
    seq = fences_around_lds(out.read_text(), "probe")
    assert re.fullmatch(r"w+Fr+F", seq), seq
