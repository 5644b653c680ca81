"""The entry and pair arenas' sizes at their limits, on the CPU
(tests/cpp/arena_limits.cpp), and that no kernel computes a place in the pair
arrays from the arena's start in 32 bits."""
import pathlib
import re
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]
CSRC = ROOT / "softrast_amd" / "csrc"


def test_arena_limits(tmp_path):
    exe = tmp_path / "arena_limits"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(ROOT / "tests/cpp/arena_limits.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, text=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
    assert res.stdout.strip() == "failed: 0"


def test_pair_arrays_have_their_own_base():
    text = "".join(p.read_text() for p in sorted(CSRC.glob("*.h")))
    assert not re.search(r"\bF\.pairs\b", text)
    for name in ("pair_rec", "pair_key", "pair_slot"):
        uses = re.findall(rf"F\.{name}\[([^\]]*)\]", text)
        assert uses and set(uses) == {"p"}, (name, uses)
