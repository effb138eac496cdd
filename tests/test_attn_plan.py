"""How attention's keys are cut into parts: plain arithmetic, checked without a GPU."""
import subprocess
from pathlib import Path


def _run(tmp_path, name):
    root = Path(__file__).resolve().parent.parent
    exe = tmp_path / name
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{root / 'cera_amd' / 'csrc'}", str(root / "tests" / "native" / f"{name}.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_more_parts_only_where_there_is_room(tmp_path):
    _run(tmp_path, "attn_plan_room")


def test_more_parts_fill_the_chip_once(tmp_path):
    _run(tmp_path, "attn_plan_rules")
