"""The deepest fp32 policies that collect_lane_kernel has LDS for, from the
dispatch's own rule compiled for the host (tests/native/lane_limits.hip), so
that a change of the layout shows which policies it moves to the tiles and the
GPU tests at the limits keep testing them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

DEEPEST = {  # env, shares of the hidden units: blocks
    ("cartpole", 1): 4, ("cartpole", 2): 8,
    ("cartpole_continuous", 1): 8, ("cartpole_continuous", 2): 8,
    ("voxelnav16", 1): 2, ("voxelnav16", 2): 7,
    ("voxelnav", 1): 2, ("voxelnav", 2): 8,
}


def test_deepest_policies_of_the_lane_collects(tmp_path):
    obj, exe = str(tmp_path / "lane_limits.o"), str(tmp_path / "lane_limits")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-Wno-unused-function",
                    "-I", os.path.join(ROOT, "include"), "-c", os.path.join(ROOT, "tests", "native", "lane_limits.hip"),
                    "-o", obj], check=True)
    subprocess.run([HIPCC, obj, "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120, check=True).stdout
    got = {(env, int(shares)): int(blocks) for env, shares, blocks in (line.split() for line in out.splitlines())}
    assert got == DEEPEST
