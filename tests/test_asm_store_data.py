"""Wait states behind wide stores, in the compiled code.

gfx950 needs two wait states between a store of more than 8 bytes and a VALU
write of the registers that hold its data.  The compiler keeps them where the
store's offset field is a constant, and keeps none where it is an SGPR: such a
store may read the next value in place of its own.  No 16-byte store of the
kernels may therefore be followed by such a write, and the buffer store that
they share leaves no offset in an SGPR."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "inq_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
WAIT = 2


def _vgprs(tok):
    out = set()
    for m in re.finditer(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", tok):
        out |= set(range(int(m.group(1)), int(m.group(2)) + 1)) if m.group(1) else {int(m.group(3))}
    return out


def overwritten(asm):
    """[store | write] of every wide store whose data a VALU instruction writes fewer than WAIT wait states later"""
    found, stores, pos = [], [], 0
    for raw in asm.split("\n"):
        line = raw.split(";")[0].strip()
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        ops = rest.split(",")
        if op.startswith("v_"):
            dst = _vgprs(ops[0]) | (_vgprs(ops[1]) if "swap" in op else set())
            found += [f"{s} | {line}" for p, data, s in stores if pos - p - 1 < WAIT and data & dst]
        if re.match(r"(buffer|global|flat|scratch)_store_dwordx[34]", op):
            stores = stores[-3:] + [(pos, _vgprs(ops[0 if op.startswith("buffer") else 1]), line)]
        pos += int(ops[0], 0) + 1 if op == "s_nop" else 1
    return found


def _assembly(src, out):
    subprocess.check_call([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                           "-packed-fp32-ops", "-fno-gpu-rdc", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                           "--cuda-device-only", "-S", "-x", "hip", str(src), "-o", str(out)], stderr=subprocess.DEVNULL)
    return out.read_text()


def test_check_finds_the_overwrite():
    store = "\tbuffer_store_dwordx4 v[0:3], v9, s[8:11], s4 offen\n"
    assert overwritten(store + "\tv_mul_f64 v[2:3], v[4:5], v[6:7]")
    assert overwritten(store + "\ts_mov_b32 s4, s5\n\tv_mov_b32 v0, v7")
    assert overwritten(store + "\tv_permlane32_swap_b32 v8, v3")
    assert not overwritten(store + "\ts_nop 1\n\tv_mov_b32 v0, v7")
    assert not overwritten(store + "\tv_mov_b32 v4, v0")
    assert not overwritten("\tbuffer_store_dwordx2 v[0:1], v9, s[8:11], s4 offen\n\tv_mov_b32 v0, v7")


PROBE = """
#include "plane_common.hpp"
using namespace inqx;
// a line's values stored at offsets that are constants and at offsets known at run time
extern "C" __global__ void probe(const double *a, cplx<double> *out, unsigned n, unsigned pl) {
  const auto r = make_rsrc(out, n);
  cplx<double> v[8];
  for (int k = 0; k < 8; ++k) v[k] = cplx<double>{a[k * 64 + threadIdx.x], a[k * 64 + 32 + threadIdx.x]};
#pragma unroll
  for (int k = 0; k < 8; ++k) bstore(r, threadIdx.x * 16u, 55u * 16u * k, cscale(v[k], a[k]));
#pragma unroll
  for (int k = 0; k < 8; ++k) bstore(r, threadIdx.x * 16u, pl * k, cscale(v[k], a[k + 8]));
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no HIP compiler")
def test_wide_buffer_store_has_no_scalar_offset(tmp_path):
    (tmp_path / "probe.hip").write_text(PROBE)
    asm = _assembly(tmp_path / "probe.hip", tmp_path / "probe.s")
    stores = re.findall(r"buffer_store_dwordx4 .*", asm)
    assert len(stores) == 16
    assert not [s for s in stores if re.search(r"\], s\d+ offen", s)]
    assert not overwritten(asm)


@pytest.mark.skipif(os.environ.get("INQX_ASM_CHECK") != "1", reason="compiles every source (minutes); set INQX_ASM_CHECK=1")
@pytest.mark.parametrize("src", ["ham_kernels", "plane_rect", "exx_kernels", "density", "small_grid", "linalg", "eigh",
                                 "eigensolver", "potential", "singularity", "layout"])
def test_library_kernels(src, tmp_path):
    asm = _assembly(os.path.join(CSRC, src + ".hip"), tmp_path / (src + ".s"))
    assert "s_endpgm" in asm
    assert not overwritten(asm)[:3]
