"""Small C++ programs compiled by g++ inside tests of the host-side headers."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "movement-sim_amd", "csrc")


def run(tmp_path, source, includes=(), args=()):
    """Compiles `source` (with csrc and include/ on the path, after `includes`) and returns what it prints."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    inc = [f"-I{d}" for d in (*includes, CSRC, os.path.join(ROOT, "include"))]
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", *inc, str(src), "-o", str(exe)], check=True,
                   timeout=110)
    return subprocess.run([str(exe), *map(str, args)], check=True, stdout=subprocess.PIPE, text=True, timeout=60).stdout
