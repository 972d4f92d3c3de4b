"""Host side of the kernel launches (csrc/it_launch.h), built and run on the CPU with the runtime's calls stood in for."""
import re
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "inferred-thoughts_amd" / "csrc"


def test_dynamic_lds_is_asked_for_once_per_kernel_and_device(tmp_path):
    exe = tmp_path / "host_launch_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(ROOT / "tests" / "native" / "host_launch_check.cpp"), "-o", str(exe)], check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def test_no_launcher_asks_by_itself():
    """Per call it is a trip through the runtime in front of every launch; kept in a plain static it holds for one device only."""
    callers = [f.name for f in sorted(CSRC.iterdir()) if f.suffix in (".hip", ".cpp", ".h") and re.search(r"\bhipFuncSetAttribute\s*\(", f.read_text())]
    assert callers == ["it_launch.h"], callers
