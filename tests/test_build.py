"""The build script: the C library needs hipcc only, the host module is extra."""
import sys
from pathlib import Path

import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "mixture-of-convolutions_amd"))
import build_lib  # noqa: E402


@pytest.fixture
def tree(tmp_path, monkeypatch):
    """A package of one small kernel, with a host module of an earlier build."""
    if not Path(build_lib.HIPCC).exists():
        pytest.skip("no hipcc")
    for name, path in (("CSRC", "csrc"), ("BUILD", "csrc/_build"), ("LIB", "moc/libmoc_hip.so"),
                       ("HOST", "moc/_moc_host.so")):
        monkeypatch.setattr(build_lib, name, tmp_path / path)
    (tmp_path / "csrc").mkdir()
    (tmp_path / "moc").mkdir()
    (tmp_path / "csrc" / "one.hip").write_text('extern "C" int one(void) { return 1; }\n')
    (tmp_path / "csrc" / "moc_host.cpp").write_text("#error not this one\n")
    build_lib.HOST.write_text("stale")
    return build_lib


def test_library_without_a_host_compiler(tree, monkeypatch, capsys):
    monkeypatch.setattr(tree, "CXX", "no-such-compiler", raising=False)
    monkeypatch.setenv("CXX", "no-such-compiler")
    assert tree.build(out=tree.LIB) == tree.LIB and tree.LIB.exists()
    assert not tree.HOST.exists()
    assert "no-such-compiler" in capsys.readouterr().err


def test_library_is_linked_before_the_host_module_fails(tree):
    with pytest.raises(RuntimeError, match="not this one"):
        tree.build(out=tree.LIB)
    assert tree.LIB.exists() and not tree.HOST.exists()
