"""When the build makes its libraries again (no compiler and no GPU needed)."""
import importlib.util
import os

from conftest import ROOT


def test_another_torch_or_another_recipe_makes_the_binding_stale(tmp_path, monkeypatch):
    spec = importlib.util.spec_from_file_location("ftc_build", os.path.join(ROOT, "fast-transformers_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    source, out = tmp_path / "binding.cpp", tmp_path / "binding.so"
    for name, value in (("OBJ_DIR", str(tmp_path)), ("HOST_OUT", str(out))):
        monkeypatch.setattr(build, name, value)
    cmd = ["true", str(source), "-o", str(out)]
    source.write_text("")
    assert build.stale(str(out), cmd, [str(source)])
    out.write_text("")
    assert build.stale(str(out), cmd, [str(source)])       # nothing says how it was built
    build.link(str(out), cmd, False)
    assert not build.stale(str(out), cmd, [str(source)])
    assert build.stale(str(out), cmd + ["-O3"], [str(source)])
    import torch
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    assert build.stale(str(out), cmd, [str(source)])
    build.link(str(out), cmd, False)
    assert not build.stale(str(out), cmd, [str(source)])
    os.utime(out, (1, 1))
    assert build.stale(str(out), cmd, [str(source)])
