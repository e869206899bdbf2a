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
    """Demangled kernel name (without its arguments) -> VGPRs and spilled VGPRs."""
    if not os.path.exists(chl.LIB_PATH) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    names, found = [], []
    with open(chl.LIB_PATH, "rb") as f:
        blob = f.read()
    d = tmp_path_factory.mktemp("co")
    for i, co in enumerate(code_objects(blob)):
        path = d / f"{i}.co"
        path.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        path.unlink()
        entry = None
        for line in notes.splitlines():
            key, _, value = line.strip().lstrip("- ").partition(":")
            if key == ".name" and value.strip().startswith("_Z"):
                names.append(value.strip())
                entry = {}
                found.append(entry)
            elif entry is not None and key in (".vgpr_count", ".vgpr_spill_count"):
                entry[key[1:]] = int(value)
    out = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout
    short = (n.replace("void ", "").replace("chl::", "").split("(")[0] for n in out.splitlines())
    return dict(zip(short, found))


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
