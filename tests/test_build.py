"""The build script: the dispatcher library, which needs torch's headers, is a step whose failure leaves the others."""
import importlib.util
import os

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-attention-kernels_amd")


@pytest.fixture
def builder(tmp_path, monkeypatch):
    """build.py with outputs in a scratch folder and commands that only create what they are asked to write."""
    spec = importlib.util.spec_from_file_location("build_script", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    for name in ("LIB_OUT", "PROBE_OUT", "TORCH_OUT"):
        monkeypatch.setattr(build, name, str(tmp_path / name))
    monkeypatch.setattr(build, "BUILD_DIR", str(tmp_path / "obj"))

    def run(cmd):
        if any("torch" in c for c in cmd) and build.fail == "compile":
            raise RuntimeError("no torch headers")
        open(cmd[cmd.index("-o") + 1], "w").close()

    build.fail = None
    monkeypatch.setattr(build, "_run", run)
    return build


def test_builds_all(builder):
    assert builder.build() == builder.LIB_OUT
    assert all(os.path.exists(f) for f in (builder.LIB_OUT, builder.PROBE_OUT, builder.TORCH_OUT))


@pytest.mark.parametrize("fail", ["compile", "import"])
def test_hip_libraries_without_the_dispatcher_library(builder, fail, monkeypatch, capsys):
    open(builder.TORCH_OUT, "w").close()  # a stale one
    builder.fail = fail
    if fail == "import":
        monkeypatch.setitem(__import__("sys").modules, "torch", None)
    assert builder.build() == builder.LIB_OUT
    assert os.path.exists(builder.LIB_OUT) and os.path.exists(builder.PROBE_OUT)
    assert not os.path.exists(builder.TORCH_OUT)
    assert "NOT built" in capsys.readouterr().err
