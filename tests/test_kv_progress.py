"""When wait_kv_written's per-layer events stand for the pass that runs (KvProgress in
relay_amd/csrc/host/host_common.h): a host-only program with threads, on the CPU."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_waits_end_with_their_layer_or_their_pass(tmp_path):
    exe = str(tmp_path / "kv_progress_check")
    host = os.path.join(REPO, "relay_amd", "csrc", "host")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include", f"-I{host}",
                    f"-I{os.path.join(REPO, 'include')}", os.path.join(REPO, "tests", "kv_progress_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
