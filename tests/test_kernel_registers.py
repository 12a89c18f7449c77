"""The registers of the split-reduction streaming GEMMs, from the notes of the
built gfx950 code object: at most 168 VGPRs, so that three waves of a SIMD (three
blocks of a CU) hold them. With 172 to 198 they held two, and launches of 512 to
768 blocks took two rounds instead of one."""

import os
import re
import shutil
import struct
import subprocess

import pytest

from maxim_amd import plan as P

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: (VGPRs, spilled VGPRs)}"""
    path = os.path.join(P.LIB_DIR, "maxim_kernels.hsaco")
    if not (os.path.exists(READELF) and os.path.exists(path)):
        pytest.skip("no llvm-readelf or no built code object")
    # the gfx950 entry of the offload bundle: a count, then (offset, size, name)
    blob = open(path, "rb").read()
    assert blob.startswith(b"__CLANG_OFFLOAD_BUNDLE__")
    at, elf = 32, tmp_path_factory.mktemp("co") / "gfx950.elf"
    for _ in range(struct.unpack_from("<Q", blob, 24)[0]):
        off, size, n = struct.unpack_from("<3Q", blob, at)
        if b"gfx950" in blob[at + 24:at + 24 + n]:
            elf.write_bytes(blob[off:off + size])
        at += 24 + n
    notes = subprocess.run([READELF, "--notes", str(elf)], capture_output=True, text=True, check=True).stdout
    out = {}
    for k in notes.split("- .agpr_count:")[1:]:
        f = dict(re.findall(r"\.(name|vgpr_count|vgpr_spill_count):\s+(\S+)", re.sub(r"\n {6,}.*", "", k)))
        out[f["name"]] = (int(f["vgpr_count"]), int(f["vgpr_spill_count"]))
    return out


def test_split_reductions_leave_three_waves_a_simd(kernels):
    ks = kernels
    # 32 outputs a wave, one operand: not _mul, nor a LayerNorm folded in from
    # a statistics pass, nor the run-time epilogue with one of its output
    split = [k for k in ks if re.match(r"mx_pw_(ch|chb|rw)2_k4", k) and not re.search(r"_mul|_ln(_|$)|_f_lo$", k)]
    assert len(split) >= 20
    over = {k: ks[k] for k in split if ks[k][0] > 168}
    assert not over, over


def test_no_streaming_gemm_spills(kernels):
    assert not {k: v for k, v in kernels.items() if k.startswith("mx_pw_") and v[1]}
