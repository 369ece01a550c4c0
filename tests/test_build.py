"""When the build makes its libraries again, and what a build for measurements compiles to (no GPU
needed)."""
import importlib.util
import os
import subprocess

from conftest import ROOT


def load_build():
    spec = importlib.util.spec_from_file_location("ftc_build", os.path.join(ROOT, "fast-transformers_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    return build


def test_time_stamps_are_not_written_over_key_lengths(tmp_path):
    """A build with -DFTC_TIMELINE passes the buffer for time stamps where the fused attention form has the
    caller's key lengths: that form takes no stamps."""
    build, out = load_build(), tmp_path / "out.s"
    counts = {}
    for source in ("ftc_tp_norm.hip", "ftc_tp.hip"):
        subprocess.run([build.find_hipcc(), os.path.join(build.CSRC, source), "-S", "-o", str(out),
                        "--offload-device-only", "-DFTC_TIMELINE"] + build.HIPCC_FLAGS + ["-O1"], check=True)
        counts[source] = out.read_text().count("s_memrealtime")
    assert counts["ftc_tp_norm.hip"] == 0 and counts["ftc_tp.hip"] > 0


def test_another_torch_or_another_recipe_makes_the_binding_stale(tmp_path, monkeypatch):
    build = load_build()
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
