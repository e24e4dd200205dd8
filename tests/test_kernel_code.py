"""The compiled gfx950 code of the attention kernels (the objects of this repository's build)."""
import pathlib
import re
import shutil
import subprocess

import pytest

BUILD = pathlib.Path(__file__).resolve().parent.parent / "infengine_amd" / "_build"
LLVM = pathlib.Path("/opt/rocm/llvm/bin")
TARGET = "hipv4-amdgcn-amd-amdhsa--gfx950"


def kernels(obj: pathlib.Path, tmp: pathlib.Path) -> dict[str, str]:
    """kernel symbol -> its disassembly"""
    subprocess.run([LLVM / "llvm-objcopy", "--dump-section", f".hip_fatbin={tmp / 'fat'}", obj, tmp / "o"],
                   check=True)
    subprocess.run([LLVM / "clang-offload-bundler", "--type=o", "--unbundle", f"--input={tmp / 'fat'}",
                    f"--targets={TARGET}", f"--output={tmp / 'code'}"], check=True)
    text = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", tmp / "code"], check=True,
                          capture_output=True, text=True).stdout
    parts = re.split(r"^[0-9a-f]+ <(\S+)>:$", text, flags=re.M)
    return dict(zip(parts[1::2], parts[2::2]))


@pytest.mark.parametrize("source", ["k_attn_prefill", "k_attn_decode"])
def test_buffer_descriptors_stay_scalar(source, tmp_path):
    """The K and V tiles' buffer descriptors are in scalar registers.  One that the compiler takes
    through a vector register (a clamp of a uniform size between two bounds did it) turns every
    load of the tile into a readfirstlane loop, up to 99 of them a kernel: paged prefill of 1024
    rows at position 5000 then takes 137 us in place of 123."""
    obj = BUILD / f"{source}.o"
    if not obj.exists() or not shutil.which(LLVM / "llvm-objdump"):
        pytest.skip("no object of the build, or no disassembler")
    code = {k: v for k, v in kernels(obj, tmp_path).items() if "buffer_load" in v}
    assert len(code) >= 4
    counts = {k: len(re.findall(r"\bv_readfirstlane_b32\b", v)) for k, v in code.items()}
    assert max(counts.values()) <= 8, counts
