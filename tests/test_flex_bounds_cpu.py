"""The LDS a block of the flexible kernels asks for covers every load of its
ordered sums, which run a batch ahead of their lists: checked on the host by a
program that repeats the loads on small systems of every shape."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_ordered_sums_load_inside_the_block(tmp_path):
    exe = str(tmp_path / "flex_bounds_check")
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950",
                           "--offload-host-only", "-x", "hip", "-std=c++17", "-O1", "-o", exe,
                           os.path.join(HERE, "flex_bounds_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "outside 0" in r.stdout, r.stdout + r.stderr
