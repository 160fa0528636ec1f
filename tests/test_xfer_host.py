"""The threaded copies of large results (pcx_xfer.hip) on the CPU, over a host
stand-in of the runtime calls they make."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_copies_on_the_host(tmp_path):
    exe = str(tmp_path / "xfer_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(HERE, "xfer"), "-o", exe,
                           os.path.join(HERE, "xfer", "xfer_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
