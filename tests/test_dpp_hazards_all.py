"""Wait states before every DPP instruction of every device bundle of the
library: each mesh length is an object of its own, so libcpwgpu.so holds one
gfx950 code object per length (tests/test_dpp_hazards.py reads the first)."""

import os
import subprocess

import pytest

from tests.test_dpp_hazards import LIB, LINE, LLVM, dpp_hazards

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _bundles(tmp):
    fb = os.path.join(tmp, "fb.bin")
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fb}", LIB, os.path.join(tmp, "x.so")],
                   check=True)
    with open(fb, "rb") as f:
        data = f.read()
    at = [0]
    while (nxt := data.find(MAGIC, at[-1] + 1)) >= 0:
        at.append(nxt)
    assert data.startswith(MAGIC)
    return [data[a:b] for a, b in zip(at, [*at[1:], len(data)])]


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(f"{LLVM}/llvm-objdump"),
                    reason="libcpwgpu.so not built or LLVM tools absent")
def test_dpp_wait_states_of_every_bundle(tmp_path):
    from cpw2000_amd.build import mesh_lengths

    bundles = _bundles(str(tmp_path))
    assert len(bundles) == len(mesh_lengths()) + 1  # one per length, and the rest
    fmacs = 0
    for i, b in enumerate(bundles):
        one, co = tmp_path / f"{i}.bin", tmp_path / f"{i}.o"
        one.write_bytes(b)
        subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={one}", f"--output={co}"], check=True)
        out = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--mcpu=gfx950", str(co)], check=True,
                             capture_output=True, text=True).stdout
        code = [(int(m.group(2), 16), m.group(1)) for m in map(LINE.match, out.split("\n")) if m]
        assert code
        bad, n_dpp, n_fmac = dpp_hazards(code)
        fmacs += n_fmac
        assert not bad, f"bundle {i}: {len(bad)} of {n_dpp} DPP instructions lack wait states: " + "; ".join(bad[:5])
    assert fmacs > 0
