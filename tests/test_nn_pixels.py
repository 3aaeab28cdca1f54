"""The weight gradient's pixel positions, on the host: they stay those of their
linear index and no shifted pixel lies outside the batch."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_positions_stay_inside_the_batch(tmp_path):
    exe = tmp_path / "wgrad_pixels"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{ROOT / 'gpuvmem_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "wgrad_pixels_main.cpp"), "-o", str(exe)],
                   check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
