"""Both gradients of a projection in one launch (castle_projection_grads: csrc/castle_gemm.hip, csrc/castle_gemm32.hip)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ROUND = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # of a result to its type


class Amax(ctypes.Structure):
    _fields_ = [("partials", ctypes.c_void_p), ("status", ctypes.c_void_p), ("column", ctypes.c_int32), ("columns", ctypes.c_int32)]


def entry():
    from lookahead_keys_attention_amd import _native as N

    lib, i, i64, vp = N.lib(), ctypes.c_int, ctypes.c_int64, ctypes.c_void_p
    lib.castle_projection_grads_workspace_bytes.restype = i64
    lib.castle_projection_grads.argtypes = [vp, i64, vp, i64, vp, i64, vp, vp, i, i, i, i, i, vp, vp, vp, vp, i64, vp]
    return N, lib


def run(dy, x, w, aux=None, amax=None):
    N, lib = entry()
    R, n, k, code, slope = dy.shape[0], dy.shape[1], x.shape[1], N.DTYPE_CODES[dy.dtype], 0 if aux is None else 2
    need = lib.castle_projection_grads_workspace_bytes(R, n, k, code, slope, int(amax is not None))
    if need < 0:
        return None
    plan = [ctypes.c_int() for _ in range(4)]
    N.check(lib.castle_projection_grads_plan(R, n, k, code, slope, int(amax is not None), *map(ctypes.byref, plan)), "castle_projection_grads_plan")
    dw, dx = (torch.full(s, float("nan"), device=DEV, dtype=dy.dtype) for s in ((n, k), (R, k)))
    ws = torch.empty(max(need, 16), device=DEV, dtype=torch.uint8)
    N.check(lib.castle_projection_grads(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), dw.data_ptr(), dx.data_ptr(), R, n, k, code, slope,
                                        None if aux is None else aux.data_ptr(), None if amax is None else ctypes.byref(amax), None, ws.data_ptr(), need,
                                        N.stream_ptr(dy.device)), "castle_projection_grads")
    return dw, dx, tuple(p.value for p in plan)


def close(got, a, b, dtype):   # a b in 64 bits: the result is rounded once, a sum of n products by n 2^-24 of their sizes at most
    ref, size = a @ b, a.abs() @ b.abs()
    return torch.all((got.double() - ref).abs() <= ROUND[dtype] * ref.abs() + (a.shape[1] + 4) * 2.0 ** -24 * size)


# one row, remainders of tiles in every direction, contractions in ranges on either side, one and two groups of waves; what two launches do better is left to them
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("R,n,k", [(1, 8, 8), (33, 72, 40), (67, 1024, 256), (199, 384, 384), (257, 3072, 512), (1001, 264, 136), (3000, 1536, 256), (3000, 256, 256), (8001, 128, 64)])
def test_both_gradients(dtype, R, n, k):
    g = torch.Generator(device=DEV).manual_seed(R)
    dy, x, w = (torch.randn(a, b + 8, generator=g, device=DEV).to(dtype)[:, :b] for a, b in ((R, n), (R, k), (n, k)))
    got = run(dy, x, w)
    assert got is not None
    dw, dx, _ = got
    assert close(dw, dy.double().t(), x.double(), dtype) and close(dx, dy.double(), w.double(), dtype)


def test_every_kind_of_workgroup():
    _, lib = entry()
    kinds = set()
    for code in (0, 1):
        for R in (32, 100, 256, 700, 3000):
            for n in (64, 256, 1536, 3072):
                for k in (64, 256, 512):
                    plan = [ctypes.c_int() for _ in range(4)]
                    if lib.castle_projection_grads_plan(R, n, k, code, 0, 0, *map(ctypes.byref, plan)) == 0:
                        tile, waves, w, x = (p.value for p in plan)
                        kinds |= {(code, tile, waves), (code, "dw", w > 1), (code, "dx", x > 1)}
    assert kinds == {(0, 32, 4), (0, 32, 8), (0, 64, 4), (1, 64, 4), (1, 64, 8)} | {(c, s, b) for c in (0, 1) for s in ("dw", "dx") for b in (False, True)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R,n,k", [(100, 256, 512), (1003, 512, 256)])
def test_slope_and_maxima(dtype, R, n, k):
    g = torch.Generator(device=DEV).manual_seed(R + n)
    dy, x, w, u = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((R, n), (R, k), (n, k), (R, k)))
    part, status = torch.full((256,), float("nan"), device=DEV), torch.ones(1, dtype=torch.int32, device=DEV)
    got = run(dy, x, w, amax=Amax(part.data_ptr(), status.data_ptr(), 64, 128))
    assert got is not None and part.max() == got[1][:, 64:192].float().abs().max() and part.min() >= 0 and status.item() == 0
    got = run(dy, x, w, aux=u)
    assert got is not None
    v = u.double().requires_grad_()
    torch.nn.functional.gelu(v).sum().backward()
    plain = dy.double() @ w.double()
    # the product is rounded before and after it is multiplied by a slope of up to 1.13 that is good to 2e-6 (absolute)
    size = (dy.double().abs() @ w.double().abs()) * 1.13
    assert torch.all((got[1].double() - plain * v.grad).abs() <= 2.02 * ROUND[dtype] * (plain * v.grad).abs() + 2e-6 * plain.abs() + (n + 4) * 2.0 ** -24 * size)
    assert close(got[0], dy.double().t(), x.double(), dtype)


class Sum(ctypes.Structure):
    _fields_ = [("part", ctypes.c_void_p), ("n", ctypes.c_int64), ("out", ctypes.c_void_p), ("parts", ctypes.c_int32), ("columns", ctypes.c_int32)]


# (parts, n, columns) of each sum: both kinds, one part and many, less than a workgroup and its edges
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sums", [[(1, 8, 0)], [(5, 2048, 0), (300, 257, 1)], [(3, 2056, 0), (1, 16, 1), (16, 4096, 0), (17, 1000, 1)]])
def test_several_sums_in_one_launch(dtype, sums):
    N, lib = entry()
    g = torch.Generator(device=DEV).manual_seed(len(sums))
    parts = [torch.randn(p, n, generator=g, device=DEV) for p, n, _ in sums]
    outs = [torch.full((n,), float("nan"), device=DEV, dtype=dtype) for _, n, _ in sums]
    jobs = (Sum * len(sums))(*[Sum(a.data_ptr(), n, o.data_ptr(), p, c) for a, o, (p, n, c) in zip(parts, outs, sums)])
    lib.castle_sums.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    N.check(lib.castle_sums(ctypes.addressof(jobs), len(sums), N.DTYPE_CODES[dtype], N.stream_ptr(torch.device(DEV))), "castle_sums")
    for a, o in zip(parts, outs):
        ref = a.double().sum(0)
        assert torch.all((o.double() - ref).abs() <= ROUND[dtype] * ref.abs() + a.shape[0] * 2.0 ** -24 * a.double().abs().sum(0))
