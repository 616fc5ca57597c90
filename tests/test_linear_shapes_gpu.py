"""Every tile shape of the projections' GEMM (M > 8) on its own, through the diagnostic variant of the library, which runs a
product on a given shape and number of parts of K (mx_linear picks among them by cost, so that which products reach a
shape moves with the fit): one step, two, an odd number and more than the buffers hold, K an odd multiple of 32, rows and
columns at and beside the tiles' edges, f32 and f16 outputs, bias, accumulation, the RMS norm and several matrices.

Tolerance as in test_linear_gpu: per element with S = sum_k |a_k w_k| over the half operands, 1e-5 S + 1e-6 (f32 sums in
any order), 2^-10 S with the norm (an operand may round to the neighbouring half), and half an ulp of an f16 output."""
import ctypes

import pytest
import torch

from dooms_amd import _lib
from dooms_amd import build as B

pytestmark = pytest.mark.gpu

SHAPES = [(16, 64, 128), (32, 64, 128), (64, 64, 64), (128, 64, 128), (128, 128, 64), (128, 128, 64), (256, 192, 64),
          (256, 256, 64), (64, 64, 64)]  # (rows, columns, K step), in the library's order; checked below
OPTIONS = [dict(), dict(bias=True, accumulate=True), dict(out_f16=True, bias=True, accumulate=True), dict(norm=True, accumulate=True),
           dict(norm=True, bias=True, count=3), dict(out_f16=True, count=2)]


@pytest.fixture(scope="module")
def lib():
    L = ctypes.CDLL(B.LIB_TRACE)
    L.mx_linear_trace_run.argtypes = _lib.lib().mx_linear.argtypes + [ctypes.c_int32, ctypes.c_int32]
    L.mx_linear_trace_run.restype = ctypes.c_int32
    L.mx_linear_trace_shape.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int32)]
    L.mx_linear_trace_plan.argtypes = [ctypes.POINTER(_lib.MxLinearDesc), ctypes.c_int32, ctypes.POINTER(ctypes.c_int32)]
    L.mx_linear_trace_plan.restype = None
    L.mx_attn_last_error.restype = ctypes.c_char_p
    return L


def shape_of(lib, i, K):
    s = (ctypes.c_int32 * 5)()
    assert lib.mx_linear_trace_shape(i, K, s) == len(SHAPES)
    return list(s)


def run(lib, device, shape, parts, M, N, K, bias=False, accumulate=False, out_f16=False, norm=False, count=1):
    g = torch.Generator(device=device)
    g.manual_seed(1000 * M + 10 * N + K + parts)
    rnd = lambda *s: torch.randn(*s, generator=g, device=device)
    unit = 8 if out_f16 else 4
    stride = (N + unit - 1) // unit * unit + unit
    odt = torch.float16 if out_f16 else torch.float32
    x = 2 * rnd(M, K)
    w = [(rnd(N, K) / K ** 0.5).half() for _ in range(count)]
    y = [rnd(M + 2, stride).to(odt) for _ in range(count)]
    y0 = [t.clone() for t in y]
    b = [rnd(N) for _ in range(count)] if bias else None
    gamma = 0.2 + 1.8 * torch.rand(K, generator=g, device=device) if norm else None
    staged = (M * ((K + 63) // 64 * 64) * 2 + 255) // 256 * 256
    bm, bn, _, most, _ = shape_of(lib, shape, K)
    tiles = count * (-(-N // bn)) * (-(-M // bm))
    assert parts <= most
    ws = torch.full((staged + (tiles * (256 + parts * bm * bn * 4) if parts > 1 else 0),), 0xAB, dtype=torch.uint8, device=device)
    d = _lib.MxLinearDesc(M=M, N=N, K=K, flags=(_lib.LINEAR_RMS_NORM if norm else 0) | (_lib.LINEAR_ACCUMULATE if accumulate else 0) |
                          (_lib.LINEAR_BIAS if bias else 0) | (_lib.LINEAR_OUT_F16 if out_f16 else 0), x_stride=K, y_stride=stride,
                          eps=1e-5, reserved=0)
    arr = lambda ts: (ctypes.c_void_p * count)(*[t.data_ptr() for t in ts])
    what = f"shape {shape} parts {parts}: {M} x {N} x {K}"
    print(what, flush=True)
    rc = lib.mx_linear_trace_run(ctypes.byref(d), count, arr(w), x.data_ptr(), arr(y), gamma.data_ptr() if norm else None,
                                 arr(b) if bias else None, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream, shape, parts)
    assert rc == 0, lib.mx_attn_last_error()
    a = x.double()
    if norm:
        a = a * gamma.double() / (a.square().mean(1, keepdim=True) + 1e-5).sqrt()
    a = a if norm else x.half().double()
    for i in range(count):
        wd = w[i].double()
        ref = a @ wd.T
        if bias:
            ref = ref + b[i].double()
        if accumulate:
            ref = ref + y0[i][:M, :N].double()
        tol = (2.0 ** -10 if norm else 1e-5) * (a.abs() @ wd.abs().T) + 1e-6
        if out_f16:
            tol = tol + ref.abs() * 2.0 ** -11 + 2.0 ** -25
        bad = (y[i][:M, :N].double() - ref).abs() > tol
        assert not bool(bad.any()), f"{what}: {int(bad.sum())} of {bad.numel()}, first {bad.nonzero()[0].tolist()}"
        assert torch.equal(y[i][M:], y0[i][M:]) and torch.equal(y[i][:, N:], y0[i][:, N:]), what  # nothing outside the output


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("steps", [0.5, 1, 1.5, 2, 3, 5.5, 7, 13])
def test_shape(lib, device, shape, steps):
    bm, bn, bk = SHAPES[shape]
    assert shape_of(lib, shape, 1 << 10)[:3] == [bm, bn, bk]
    K = int(steps * bk)
    most = shape_of(lib, shape, K)[3]
    if most == 0:  # half a step of the 128-column shapes is no multiple of their step
        assert bk == 128 and K % 128
        return
    n = 0
    for M in sorted({9, max(9, bm - 1), max(9, bm), bm + 1, 2 * bm + 3}):
        for N in (1, bn - 1, bn + 2, 2 * bn):
            for parts in sorted({1, min(2, most), min(3, most), most}):
                run(lib, device, shape, parts, M, N, K, **OPTIONS[n % len(OPTIONS)])
                n += 1


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_shape_fills_the_chip(lib, device, shape):
    """More tiles than CUs, so that workgroups of every XCD and several rounds run, K whole and in parts."""
    bm, bn, bk = SHAPES[shape]
    M, N = 5 * bm + 1, 60 * bn - 3
    K = 4 * bk
    for parts in {1, min(3, shape_of(lib, shape, K)[3])}:
        run(lib, device, shape, parts, M, N, K, bias=True, accumulate=True)


def test_refused(lib, device):
    t = torch.zeros(64, 128, device=device)
    d = _lib.MxLinearDesc(M=16, N=64, K=96, flags=0, x_stride=128, y_stride=64, eps=0.0, reserved=0)
    p = (ctypes.c_void_p * 1)(t.data_ptr())
    call = lambda ws, shape, parts: lib.mx_linear_trace_run(ctypes.byref(d), 1, p, t.data_ptr(), p, None, None, t.data_ptr(), ws, None, shape, parts)
    for shape, parts in ((0, 1), (-1, 1), (9, 1), (2, 0), (2, 3), (7, 2)):  # a shape or a number of parts that K = 96 has not
        assert call(1 << 14, shape, parts) == _lib.INVALID_ARGUMENT
    assert call(16 * 128 * 2, 2, 2) == _lib.RESOURCE_EXHAUSTED  # room for the staged rows only


# What the plan takes for the products that test_linear_gpu names by their tiles: a fit that moves them has to move those.
@pytest.mark.parametrize("M,N,K,count,rows,columns", [
    (1300, 8300, 2080, 1, 256, 256), (1900, 5700, 1056, 1, 256, 192), (1900, 5704, 1056, 1, 256, 192), (1500, 1280, 1280, 8, 256, 256),
    (1300, 8300, 2048, 1, 256, 256), (1900, 5700, 1024, 1, 256, 192), (2048, 6144, 4096, 1, 256, 192)])
def test_planned_shape(lib, device, M, N, K, count, rows, columns):
    d = _lib.MxLinearDesc(M=M, N=N, K=K, flags=0, x_stride=K, y_stride=N, eps=0.0, reserved=0)
    plan = (ctypes.c_int32 * 2)()
    lib.mx_linear_trace_plan(ctypes.byref(d), count, plan)
    assert SHAPES[plan[0]][:2] == (rows, columns)
