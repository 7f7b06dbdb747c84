"""Queue order of a launch's camera paths (pupiloptixlab_amd/csrc/pt_slots.h,
used by the raygen kernel), checked on the host by tests/slot_sim.cpp: every
(frame, pixel) of a launch is traced by exactly one queue slot, over films of
full and partial 8x8 tiles (1 to 2M pixels) and 1 to 64 frames."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_slots_cover_a_launch(tmp_path):
    exe = str(tmp_path / "slot_sim")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "pupiloptixlab_amd", "csrc"),
                    os.path.join(ROOT, "tests", "slot_sim.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
