"""The build without what only the Python ops' helpers need."""
import builtins
import subprocess

import pytest

from litert_amd import build


@pytest.fixture
def commands(monkeypatch, tmp_path):
    """Commands instead of compilers; a test's `fails` names what may not work."""
    ran = []
    monkeypatch.setattr(build, "LIB", str(tmp_path))

    def run(cmd):
        ran.append(" ".join(cmd))
    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "build_fc", lambda: ran.append("fc") or "fc")
    return ran


def _not_built(ran):
    assert "fc" in ran
    assert any("liblitert_amd_delegate" in c for c in ran) and any("liblitert_amd_bench_probes" in c for c in ran)


@pytest.mark.parametrize("missing", ["torch is not installed", "torch does not load"])
def test_everything_else_is_built_without_torch(commands, monkeypatch, missing):
    real = builtins.__import__

    def without_torch(name, *args, **kw):
        if name == "torch":
            raise (ModuleNotFoundError if "installed" in missing else OSError)(missing)
        return real(name, *args, **kw)
    monkeypatch.setattr(builtins, "__import__", without_torch)
    outs = build.build_all()
    assert not any("litert_amd_tensors" in o for o in outs) and all(outs)
    _not_built(commands)


def test_everything_else_is_built_where_the_helper_does_not_compile(commands, monkeypatch, tmp_path):
    ran = commands
    stale = tmp_path / build.torch_tensors_name(pytest.importorskip("torch").__version__)
    stale.write_text("of an earlier build")

    def run(cmd):
        ran.append(" ".join(cmd))
        if any("torch_tensors.cc" in c for c in cmd):
            raise subprocess.CalledProcessError(1, cmd)
    monkeypatch.setattr(build, "_run", run)
    outs = build.build_all()
    assert not any("litert_amd_tensors" in o for o in outs)
    assert not stale.exists()  # it would be loaded in place of the fallback
    _not_built(ran)
