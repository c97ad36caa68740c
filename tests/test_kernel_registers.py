"""The decode GEMV's kernels of whole 256-value units compile without the partial units' arithmetic (the code object of the
last build, its kernels' own metadata)."""

import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
OBJ = ROOT / "artlite_amd" / "csrc" / "_build" / "gemv.o"
LLVM = Path("/opt/rocm/lib/llvm/bin")


@pytest.mark.skipif(not OBJ.exists() or not (LLVM / "llvm-readelf").exists(), reason="no build here, or no LLVM tools")
def test_whole_unit_kernels(tmp_path: Path) -> None:
    """Q4_0 (format 2): the partial units' counts of units took gate / up from 16 spilled SGPRs to 19 and the down from 84
    SGPRs to 98."""
    fat, co = tmp_path / "gemv.fat", tmp_path / "gemv.co"
    subprocess.run(["objcopy", "--dump-section", f".hip_fatbin={fat}", str(OBJ), str(tmp_path / "o")], check=True)
    subprocess.run([LLVM / "clang-offload-bundler", "-type=o", "-unbundle", f"-input={fat}", f"-output={co}",
                    "-targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([LLVM / "llvm-readelf", "--notes", co], capture_output=True, text=True, check=True).stdout
    regs = {}
    for kernel in notes.split("  - .agpr_count")[1:]:
        name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
        regs[name] = {k: int(re.search(rf"\.{k}:\s+(\d+)", kernel).group(1))
                      for k in ("sgpr_count", "sgpr_spill_count", "vgpr_spill_count")}

    def whole(swiglu: int) -> dict:
        return next(r for n, r in regs.items() if re.search(rf"k_gemvILi2ELb{swiglu}ELi2E(Li0E|Lb0E)?EEv", n))

    assert whole(1)["sgpr_spill_count"] <= 16 and whole(0)["sgpr_count"] <= 84
    assert not any(r["vgpr_spill_count"] for r in regs.values())
