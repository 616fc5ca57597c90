"""The torch front end's extension (dooms_amd._native) against the general path of dooms_amd.attention: the same bits for
every form of argument that it takes, and the same exceptions for what it leaves to the general path."""
import numpy as np
import pytest
import torch

from dooms_amd import MxAttnError
from dooms_amd import attention as A

pytestmark = pytest.mark.gpu


class _General:
    """Stands in for the extension: every call goes the general path."""

    def __getattr__(self, name):
        return lambda *a: None


class _Counted:
    """The extension, with the number of calls that it answered."""

    def __init__(self, ext):
        self.ext, self.taken = ext, 0

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.ext, name)(*a)
            self.taken += r is not None
            return r
        return call


def both(monkeypatch, fn, taken=1):
    """fn() through the extension and through the general path: equal results (None, tensors, tuples or lists)."""
    ext = _Counted(A._native())
    res = []
    for n in (ext, _General()):
        monkeypatch.setattr(A, "_native", lambda n=n: n)
        r = fn()
        torch.cuda.synchronize()
        res.append([None if t is None else t.clone() for t in (r if isinstance(r, (tuple, list)) else [r])])
        kind = type(r)
    monkeypatch.undo()
    assert ext.taken == taken
    assert len(res[0]) == len(res[1]) and kind in (tuple, list, torch.Tensor)
    for a, b in zip(*res):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and a.device == b.device and torch.equal(a, b)


def t(device, *shape, dtype=torch.float16, seed=0):
    x = np.random.default_rng(seed + sum(shape)).standard_normal(shape, dtype=np.float32)
    return torch.from_numpy(x).to(device).to(dtype)


H = dict(n_head=8, n_head_kv=2, head_dim=64)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_decode(device, monkeypatch, dtype):
    ws = A.new_workspace(1 << 22, device)
    ks, vs = [t(device, n, 160)[:, :128] for n in (300, 77)], [t(device, n, 160, seed=1)[:, :128] for n in (300, 77)]
    q = t(device, 2, 520, dtype=dtype)[:, :512]
    out = torch.zeros(2, 512, dtype=dtype, device=device)
    lse = torch.zeros(2, 8, device=device)
    for kw in (dict(), dict(scale=0.3), dict(scale=1), dict(out=out), dict(want_lse=True), dict(lse=lse), dict(causal=True)):
        both(monkeypatch, lambda: A.decode(q, ks, vs, [300, 77], workspace=ws, **H, **kw))
    both(monkeypatch, lambda: A.decode(q, tuple(ks), tuple(vs), (300, 77), workspace=ws, **H))
    q3 = t(device, 3, 512, dtype=dtype)
    both(monkeypatch, lambda: A.decode(q3, ks[:1], vs[:1], [300], n_q=3, causal=True, workspace=ws, **H))
    # forms that stay on the general path
    both(monkeypatch, lambda: A.decode(q, ks, vs, np.array([300, 77]).tolist(), **H), taken=0)  # its own workspace
    both(monkeypatch, lambda: A.decode(q, ks, vs, [300, 77], workspace=ws, tuning=dict(decode_splits=2), **H), taken=0)
    both(monkeypatch, lambda: A.decode(q, ks, vs, [np.int32(300), 77], workspace=ws, **H), taken=0)


def test_decode_rope(device, monkeypatch):
    ws = A.new_workspace(1 << 22, device)
    ks, vs = [t(device, 300, 128), t(device, 40, 128)], [t(device, 300, 128, seed=1), t(device, 40, 128, seed=1)]
    qkv = t(device, 2, 768, dtype=torch.float32)
    for mode, kw in ((0, {}), (1, dict(rope_base=1e6, want_lse=True)), (2, dict(scale=0.2))):
        both(monkeypatch, lambda: A.decode_rope(qkv, ks, vs, [300, 40], rope_mode=mode, workspace=ws, **H, **kw) + (ks[0], vs[1]))


@pytest.mark.parametrize("ws_bytes", [None, 1 << 25])
def test_prefill(device, monkeypatch, ws_bytes):
    ws = None if ws_bytes is None else A.new_workspace(ws_bytes, device)
    k, v = t(device, 260, 128), t(device, 260, 128, seed=1)
    q, qkv = t(device, 60, 512), t(device, 60, 768, dtype=torch.float32)
    for kw in (dict(p0=200), dict(p0=100, n_kv=200, want_lse=True), dict(causal=False, n_kv=260, scale=0.5),
               dict(p0=200, out=torch.zeros(60, 512, dtype=torch.float16, device=device))):
        both(monkeypatch, lambda: A.prefill(q, k, v, workspace=ws, **H, **kw))
    for kw in (dict(p0=200, rope_mode=1), dict(p0=100, rope_mode=0, rope_base=500000, want_lse=True)):
        both(monkeypatch, lambda: A.prefill_rope(qkv, k.clone(), v.clone(), workspace=ws, **H, **kw))
    both(monkeypatch, lambda: A.prefill(q, k, v, p0=200, workspace="auto", **H), taken=0)


@pytest.mark.parametrize("M", [1, 5, 40])
def test_linear(device, monkeypatch, M):
    x, w = t(device, M, 256, dtype=torch.float32), [t(device, 64, 256, seed=i) for i in range(2)]
    g, b = t(device, 256, dtype=torch.float32), t(device, 64, dtype=torch.float32)
    for kw in (dict(), dict(gamma=g), dict(bias=b), dict(out_f16=True), dict(gamma=g, eps=1e-3, bias=b)):
        both(monkeypatch, lambda: A.linear(x, w[0], **kw))
    both(monkeypatch, lambda: A.linear(x, w, bias=[b, None]))
    both(monkeypatch, lambda: A.linear(x, tuple(w)))
    both(monkeypatch, lambda: A.linear(x, w[0], out=torch.ones(M, 64, device=device), accumulate=True))
    both(monkeypatch, lambda: A.linear(x, w, out=[torch.ones(M, 72, device=device)[:, :64] for _ in w], accumulate=True))
    assert isinstance(A.linear(x, w), list)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [64, 6])
def test_self_attention(device, monkeypatch, dtype, head_dim):
    qkv = t(device, 2, 50, 3 * 4 * head_dim, dtype=dtype)
    both(monkeypatch, lambda: A.self_attention(qkv, heads=4))
    both(monkeypatch, lambda: A.self_attention(qkv, heads=4, scale=0.1, out=torch.zeros(2, 50, 4 * head_dim, dtype=dtype, device=device)))


def test_refused(device, monkeypatch):
    ws = A.new_workspace(1 << 20, device)
    k, q = t(device, 300, 128), t(device, 1, 512)
    x, w = t(device, 12, 256, dtype=torch.float32), t(device, 64, 256)
    calls = [
        lambda: A.decode(q, [k], [k, k], [50], workspace=ws, **H),
        lambda: A.decode(q.double(), [k], [k], [50], workspace=ws, **H),
        lambda: A.decode(q, [k], [k.T], [50], workspace=ws, **H),
        lambda: A.decode(q, [k], [k], [300], workspace=ws[:256], **H),                        # too small
        lambda: A.decode(q, [k], [k], [0], workspace=ws, **H),
        lambda: A.decode(q.cpu(), [k], [k], [50], workspace=ws, **H),
        lambda: A.decode(q, [k], [k], [50], workspace=ws, n_head=8, n_head_kv=3, head_dim=64),
        lambda: A.decode_rope(q.float(), [k], [k], [50], rope_mode=5, workspace=ws, **H),
        lambda: A.prefill(q, k, t(device, 300, 136), p0=3, **H),
        lambda: A.prefill(q, k, k, p0=-1, **H),
        lambda: A.linear(x, [w, w[:32]]),
        lambda: A.linear(x, w[:, :100]),
        lambda: A.linear(x, w, out=torch.zeros(12, 66, device=device)),
        lambda: A.self_attention(q, heads=4),
        lambda: A.self_attention(t(device, 1, 4, 30), heads=7),
    ]
    for i, fn in enumerate(calls):
        said = []
        for general in (False, True):
            if general:
                monkeypatch.setattr(A, "_native", lambda: _General())
            with pytest.raises((ValueError, MxAttnError, RuntimeError)) as e:
                fn()
            monkeypatch.undo()
            said.append((e.type, str(e.value)))
        assert said[0] == said[1], i
