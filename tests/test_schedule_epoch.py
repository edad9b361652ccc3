"""Settings that a captured V-cycle depends on count the mesh's schedule epoch up, so that the next replay captures again
(host only: a replay of a stale graph, whose work-unit table is freed, is never run to find out)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_settings_count_the_epoch_up(tmp_path):
    import hyteg_amd
    lib_dir = os.path.dirname(hyteg_amd._lib.LIB_PATH)
    exe = str(tmp_path / "hymi_epoch_check")
    cmd = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
           "-I", os.path.join(ROOT, "hyteg_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "hymi_epoch_check.cpp"), "-o", exe,
           "-L", lib_dir, "-lhymi", f"-Wl,-rpath,{lib_dir}", "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
