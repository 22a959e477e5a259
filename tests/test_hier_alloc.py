"""Allocations of a multigrid build (no GPU): the library against stand-ins for its HIP calls."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.join(HERE, "..")


def _build_run(name, tmp_path):
    from opflow_amd import build
    if not os.path.exists(build.LIB):
        build.build()
    exe = str(tmp_path / name)
    lib = os.path.dirname(build.LIB)
    # -rdynamic: the library's calls bind to the program's stand-ins
    subprocess.run([build.HIPCC, "-x", "c++", "-O1", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + build.CSRC, "-Wno-unused-value", "-Wno-unused-result",
                    os.path.join(HERE, "cpp_host", name + ".cpp"), "-o", exe, "-L" + lib, "-lopflow_hip",
                    "-Wl,-rpath," + lib, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "passed" in r.stdout


def test_build_after_a_failed_one(tmp_path):
    _build_run("hier_alloc_check", tmp_path)


def test_footprint_covers_what_a_hierarchy_takes(tmp_path):
    _build_run("footprint_check", tmp_path)
