"""Registers and spills of built kernels, read from the code objects' metadata.

Some kernels are fast only while the compiler keeps them in registers at the occupancy they are
written for, and a change of shared arithmetic can push them over without any wrong result.  The
limits here are the architecture's (512 VGPRs per SIMD and lane: 168 for three waves, 128 for
four), not measured values.
"""
import os
import shutil
import struct
import subprocess

import pytest

import cholla_amd as chl
from cholla_amd import build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(blob):
    """The gfx950 code objects of every offload bundle in a library."""
    at = blob.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        (count,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in triple and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, pos)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Demangled kernel name (without its arguments) -> VGPRs, spilled VGPRs and LDS."""
    if not os.path.exists(chl.LIB_PATH) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    entries = []  # one per kernel; .agpr_count is the first key of each
    with open(chl.LIB_PATH, "rb") as f:
        blob = f.read()
    d = tmp_path_factory.mktemp("co")
    for i, co in enumerate(code_objects(blob)):
        path = d / f"{i}.co"
        path.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        path.unlink()
        for line in notes.splitlines():
            key, _, value = line.strip().lstrip("- ").partition(":")
            if key == ".agpr_count":
                entries.append({})
            if key in (".vgpr_count", ".vgpr_spill_count", ".group_segment_fixed_size"):
                entries[-1][key[1:]] = int(value)
            elif key == ".name" and value.strip().startswith("_Z"):
                entries[-1]["name"] = value.strip()
    names = [e.pop("name") for e in entries]
    out = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout
    short = (n.replace("void ", "").replace("chl::", "").split("(")[0] for n in out.splitlines())
    return dict(zip(short, entries))


def matching(kernels, prefix):
    hits = {n: k for n, k in kernels.items() if n.startswith(prefix)}
    assert hits, prefix
    return hits


@pytest.mark.parametrize("prefix", ["Vl1dStage1Kernel<", "Vl1dStage2Kernel<", "Vl2dPcmFluxKernel<",
                                    "ReconGridKernel<", "RiemannGridKernel<"])
def test_line_kernels_do_not_spill(kernels, prefix):
    """The unfused 1D stages, the 2D PCM fluxes and the interface and flux kernels over a grid,
    every solver and reconstruction."""
    spills = {n: k["vgpr_spill_count"] for n, k in matching(kernels, prefix).items() if k["vgpr_spill_count"]}
    assert not spills


@pytest.mark.parametrize("form", ["PolicyExact", "PolicyFast"])
def test_mhd_ppmc_x_faces_hold_three_waves(kernels, form):
    """The FP64 x-face launch of the MHD step with PPMC: three waves per SIMD, nothing spilled."""
    k = matching(kernels, f"mhd::MhdFlux2TileKernel<{form}, 2>").popitem()[1]
    assert k["vgpr_spill_count"] == 0 and k["vgpr_count"] <= 168


def test_mhd_mixed_stage_1_holds_four_waves(kernels):
    """The mixed stage-1 march of the MHD step is compiled for four waves per SIMD, with its dt
    reduction in registers too."""
    k = matching(kernels, "mhd::MhdFlux1MarchKernel<PolicyMixed").popitem()[1]
    assert k["vgpr_spill_count"] == 0 and k["vgpr_count"] <= 128


def test_mhd_ct_chunks_count_the_workgroups_a_cu_holds(kernels, tmp_path):
    """The planes per workgroup of the CT updates on a 128^3 box (64 columns of tiles): one round
    of the workgroups that the kernel's LDS admits, 8 chunks of 16 for the FP64 forms' two per CU
    and 11 of 12 for the mixed form's three."""
    per_cu = {}
    for form in ("PolicyExact", "PolicyFast", "PolicyMixed"):
        lds = {k["group_segment_fixed_size"] for k in matching(kernels, f"mhd::MhdCtUpdateKernel<{form}").values()}
        per_cu[form] = 160 * 1024 // max(lds)
    assert per_cu == {"PolicyExact": 2, "PolicyFast": 2, "PolicyMixed": 3}
    src = tmp_path / "chunk.hip"
    src.write_text('#include "mhd_launch.hpp"\n#include <cstdio>\n'
                   "int main() { std::printf(\"%d %d %d\", chl::MhdCtChunk<chl::PolicyExact>(64, 128),"
                   " chl::MhdCtChunk<chl::PolicyFast>(64, 128), chl::MhdCtChunk<chl::PolicyMixed>(64, 128)); }\n")
    exe = tmp_path / "chunk"
    subprocess.run([build.hipcc(), *build.COMMON, "-O0", "--cuda-host-only", f"-I{build.CSRC}", str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout == "16 16 12"
