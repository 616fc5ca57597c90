"""The torch front end's extension (dooms_amd._native) where it is absent or was built for something else. No GPU needed."""
import ctypes
import sys

import pytest

from dooms_amd import _lib
from dooms_amd import attention as A
from dooms_amd import build as B


@pytest.fixture
def unbound(monkeypatch):
    monkeypatch.setattr(A, "_bound", None)
    monkeypatch.setattr(A, "_ext", None)


def test_absent_extension_leaves_the_general_path(monkeypatch, unbound):
    import dooms_amd
    monkeypatch.delattr(dooms_amd, "_native", raising=False)
    monkeypatch.delitem(sys.modules, "dooms_amd._native", raising=False)
    monkeypatch.setattr(sys, "meta_path", [_Hide(f) for f in sys.meta_path])
    with pytest.warns(RuntimeWarning, match="dooms_amd.build"):
        ext = A._native()
    for name in ("prefill", "decode", "decode_rope", "prefill_rope", "linear", "self_attention"):
        assert getattr(ext, name)(1, 2) is None
    assert A._native() is ext  # and says so once


class _Hide:
    """A finder that does not find the extension."""

    def __init__(self, finder):
        self.finder = finder

    def find_spec(self, name, *args):
        return None if name == "dooms_amd._native" else self.finder.find_spec(name, *args)


def test_extension_of_another_version_is_refused(unbound):
    from dooms_amd import _native as ext
    sizes = [ctypes.sizeof(t) for t in (_lib.MxAttnDesc, _lib.MxAttnRope, _lib.MxLinearDesc, _lib.MxSelfAttnDesc)]
    version = _lib.lib().mx_attn_abi_version()
    for v, s in [(version + 1, sizes)] + [(version, sizes[:i] + [sizes[i] + 8] + sizes[i + 1:]) for i in range(4)]:
        with pytest.raises(ImportError, match="dooms_amd.build"):
            ext.bind(v, tuple(s), *[0] * 9)
    assert A._native() is ext


def test_build_makes_the_extension_too(monkeypatch, tmp_path):
    ran = []
    monkeypatch.setattr(B, "_run", lambda cmd: (ran.append(cmd), (0, ""))[1])
    monkeypatch.setattr(B.os, "replace", lambda *a: None)
    monkeypatch.setattr(B.os, "makedirs", lambda *a, **k: None)
    B.build()
    assert any(c[0] == "g++" and B.EXT + ".tmp" in c for c in ran)
    ran.clear()
    B.build(out=str(tmp_path / "variant.so"))
    assert not any(c[0] == "g++" for c in ran)
