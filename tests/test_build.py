"""Host: what build.py builds with and without torch, and when the incremental build keeps the extension.  No compiler
runs: the commands are recorded and their outputs are made empty."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture
def build(monkeypatch, tmp_path):
    spec = importlib.util.spec_from_file_location("mxopt_build_under_test", os.path.join(ROOT, "mlx-node_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    mod.made = []

    def run(cmd, *_):
        out = cmd[cmd.index("-o") + 1]
        open(out, "w").close()
        mod.made.append(os.path.basename(out))

    monkeypatch.setattr(mod, "_run", run)
    monkeypatch.setattr(mod.subprocess, "check_call", run)
    for name in ("LIB", "ARRAYS", "DEMO", "NAPI"):
        monkeypatch.setattr(mod, name, str(tmp_path / os.path.basename(getattr(mod, name))))
    monkeypatch.setattr(mod, "OBJ_DIR", str(tmp_path / "obj"))
    return mod


def test_without_torch_everything_but_the_python_extension_is_built(build, monkeypatch, capsys):
    find = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, "find_spec", lambda name, *a: None if name == "torch" else find(name, *a))
    assert build.build() == build.LIB and os.path.exists(build.LIB)
    assert "cabi_demo" in build.made and not os.path.exists(build.ARRAYS)
    assert "torch is not installed" in capsys.readouterr().err


def test_a_failing_extension_leaves_the_library_and_the_demo_built(build, monkeypatch):
    def fails(*_):
        raise RuntimeError("g++ failed")

    monkeypatch.setattr(build, "build_arrays", fails)
    with pytest.raises(RuntimeError, match="g\\+\\+ failed"):
        build.build()
    assert os.path.exists(build.LIB) and os.path.exists(build.DEMO)


def test_incremental_build_renews_the_extension_for_another_torch(build, monkeypatch, tmp_path):
    build.build()
    assert "_arrays.so.tmp" in build.made
    build.made.clear()
    build.build(incremental=True)
    assert "_arrays.so.tmp" not in build.made
    other = tmp_path / "torch"
    other.mkdir()
    (other / "version.py").write_text("__version__ = '0.0'\n")
    monkeypatch.setattr(build, "_torch_dir", lambda: str(other))
    build.build(incremental=True)
    assert "_arrays.so.tmp" in build.made
    build.made.clear()
    build.build(incremental=True)
    assert "_arrays.so.tmp" not in build.made
