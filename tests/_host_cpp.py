"""Runs host code of csrc/ headers that need no GPU (not collected by pytest)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pack3d_amd", "csrc")


def run_host_cpp(tmp_path, headers, body):
    """The lines that ``body`` prints, compiled as the main function of a host
    program that includes the given headers of csrc/."""
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    includes = "".join(f'#include "{h}"\n' for h in headers)
    src.write_text(f"{includes}#include <cstdio>\nint main() {{\n{body}\nreturn 0;\n}}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()
