"""Turn the recorded RCPPS fixture (rcpps_table.txt) into C initialiser lists.

Writes oracle/rcpps_table.inc (used by the CPU oracle) and
softrast_amd/csrc/rcpps_table.inc (what rcp_check.hip holds the library's
formula against, word for word). Both hold the same 2048 words: bits of rcp(1 + i/2048) as observed on an Intel host
(see gen_rcpps_table.c). tests/test_oracle_kat.py checks both against the fixture.
"""
import pathlib

ROOT = pathlib.Path(__file__).resolve().parents[2]


def main():
    words = [w.strip() for w in (ROOT / "tests/golden/rcpps_table.txt").read_text().split()]
    assert len(words) == 2048
    body = ",\n".join(", ".join("0x" + w + "u" for w in words[i:i + 8]) for i in range(0, 2048, 8))
    text = ("/* Generated by tests/golden/make_rcpps_inc.py from tests/golden/rcpps_table.txt.\n"
            " * RCPPS bits of 1 + i/2048 for i = 0..2047 (top 11 mantissa bits). */\n" + body + "\n")
    for dst in ("oracle/rcpps_table.inc", "softrast_amd/csrc/rcpps_table.inc"):
        (ROOT / dst).write_text(text)


if __name__ == "__main__":
    main()
