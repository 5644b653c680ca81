"""The device's RCPPS and RSQRTPS, computed with the hardware's reciprocals,
against the recorded tables: every cell, exponent and sign (rcp_check.hip)."""
import pathlib
import subprocess

import pytest

pytestmark = pytest.mark.gpu


def test_rcpps_rsqrtps_every_cell():
    exe = pathlib.Path(__file__).resolve().parents[1] / "softrast_amd" / "rcp_check"
    if not exe.exists():
        from softrast_amd import build
        build.build_rcp_check()
    print("[rcp] every cell", flush=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "differing results: 0" in r.stdout
