"""What the build makes together, with a compiler that only notes its calls."""
import pathlib


def test_library_and_its_device_check_are_built_together(tmp_path, monkeypatch):
    """rcp_check runs device functions of the library; tests/test_gpu_rcp.py
    runs it as it finds it, so no library is built without it."""
    from softrast_amd import build
    calls = []

    def run(cmd):
        calls.append(cmd)
        pathlib.Path(cmd[cmd.index("-o") + 1]).write_text("built")

    monkeypatch.setattr(build, "PKG", tmp_path)
    monkeypatch.setattr(build, "_run", run)
    (tmp_path / "rcp_check").write_text("stale")
    (tmp_path / "libsrgpu.so").write_text("stale")
    build.build_gpu()
    sources = [pathlib.Path(c[-1]).name for c in calls]
    assert sorted(sources) == ["rcp_check.hip", "srgpu.hip"]
    assert (tmp_path / "libsrgpu.so").read_text() == (tmp_path / "rcp_check").read_text() == "built"
