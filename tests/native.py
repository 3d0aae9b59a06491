"""Compiles a C++ program against the library's internal headers and libccoil_hip.so and runs it on the host (no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "c-coil_amd")


def run(tmp_path, source, timeout=120):
    """The lines that the program prints."""
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(source)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-std=c++17", "-x", "hip", "--offload-host-only",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"), str(src), "-o", str(exe),
                    "-L" + PKG, "-lccoil_hip", "-Wl,-rpath," + PKG], check=True, capture_output=True, text=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=timeout).stdout.splitlines()
