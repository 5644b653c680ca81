"""Turn the recorded RSQRTPS fixture (rsqrtps_table.txt) into C initialiser lists.

Writes oracle/rsqrtps_table.inc (used by the CPU oracle) and
softrast_amd/csrc/rsqrtps_table.inc (what rcp_check.hip holds the library's
formula against, word for word). Both hold the same 4096 words: bits of rsqrt(1 + i/2048) for i = 0..2047, then of
rsqrt(2 + i/1024), as observed on an Intel host (see gen_rsqrtps_table.c).
tests/test_oracle_kat.py checks both against the fixture.
"""
import pathlib

ROOT = pathlib.Path(__file__).resolve().parents[2]


def main():
    words = [w.strip() for w in (ROOT / "tests/golden/rsqrtps_table.txt").read_text().split()]
    assert len(words) == 4096
    body = ",\n".join(", ".join("0x" + w + "u" for w in words[i:i + 8]) for i in range(0, 4096, 8))
    text = ("/* Generated by tests/golden/make_rsqrtps_inc.py from tests/golden/rsqrtps_table.txt.\n"
            " * RSQRTPS bits of [1, 2) then [2, 4) by the top 11 mantissa bits. */\n" + body + "\n")
    for dst in ("oracle/rsqrtps_table.inc", "softrast_amd/csrc/rsqrtps_table.inc"):
        (ROOT / dst).write_text(text)


if __name__ == "__main__":
    main()
