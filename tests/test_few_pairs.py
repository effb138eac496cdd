"""The few-token products' sharing out of a chunk's tokens among threads: plain arithmetic, checked without a GPU."""
import subprocess
from pathlib import Path


def test_threads_stay_inside_a_chunk_and_cover_it(tmp_path):
    root = Path(__file__).resolve().parent.parent
    exe = tmp_path / "few_pairs"
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{root / 'cera_amd' / 'csrc'}", str(root / "tests" / "native" / "few_pairs.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "6 instances\n", r.stdout
