"""The ragged GEMM kernels of linear_gemm.hip: linear and projection products that the direct-load
kernels refuse (any K, pitch, extent and element-aligned pointer; sequences of any length in a
head-split weight gradient), against float64 products of the same rounded inputs.

Every operand sits one element off a 16-byte boundary inside a NaN-filled buffer, so a read past
an edge that reached a sum would show, and the bands around the outputs must stay as they were.
Tolerance: sums of K products in fp32, relative to the largest value, 1e-5; 16-bit outputs round
once, half a unit in the last place of a value up to that largest: 2^-8 bf16, 2^-11 fp16.
"""
import math

import pytest
import torch

from cudatransformer_amd import _capi

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"f32": 1e-5, "bf16": 2.0 ** -8 + 1e-5, "f16": 2.0 ** -11 + 1e-5}
PAD = 520


class Guarded:
    """A tensor of `shape` one element past a 16-byte boundary, NaN around it."""

    def __init__(self, shape, dt, g=None, std=1.0):
        n = math.prod(shape)
        self.buf = torch.full((n + 2 * PAD + 1,), float("nan"), dtype=dt, device="cuda")
        self.t = self.buf[PAD + 1:PAD + 1 + n].view(shape)
        self.t.copy_(torch.zeros(shape) if g is None else std * torch.randn(shape, generator=g, device="cuda"))

    def intact(self):
        n = self.t.numel()
        return bool(torch.isnan(self.buf[:PAD + 1]).all() and torch.isnan(self.buf[PAD + 1 + n:]).all())


def close(got, want, name, what):
    err = (got.double() - want).abs().max() / want.abs().max().clamp_min(1e-30)
    assert err <= TOL[name], (what, float(err))


# Edges of the 64 and 128 tiles, of the 16 / 64-deep stages and of the chunks; enough rows and K
# for the split-K plans ((130, 70, 2051): dW splits, (200, 2051, 70): dX splits); one 128-tile grid.
SHAPES = [(1, 1, 1), (3, 5, 7), (63, 65, 15), (64, 64, 17), (129, 127, 65), (130, 70, 2051), (200, 2051, 70),
          (2051, 70, 200), (1800, 1801, 129)]


@pytest.mark.parametrize("mnk", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_ragged_linear(name, mnk):
    m, n, k = mnk
    dt = DT[name]
    print(f"ragged linear {name} M={m} N={n} K={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w, b = Guarded((m, k), dt, g), Guarded((n, k), dt, g, 1 / math.sqrt(k)), Guarded((n,), dt, g)
    dy, dw, db, y, dx = Guarded((m, n), dt, g), Guarded((n, k), dt), Guarded((n,), dt), Guarded((m, n), dt), Guarded((m, k), dt)
    lib, code = _capi.load(), _capi._DTYPE_CODE[dt]
    ws = torch.empty(max(lib.ctattn_linear_bwd_workspace_bytes(code, m, n, k), 16), dtype=torch.uint8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    p = lambda h: h.t.data_ptr()  # noqa: E731
    assert lib.ctattn_linear_fwd(code, p(x), p(w), p(b), p(y), m, n, k, st) == 0
    assert lib.ctattn_linear_bwd(code, p(x), p(w), p(dy), p(dx), p(dw), p(db), ws.data_ptr(), ws.numel(), m, n, k, st) == 0
    first = [t.t.clone() for t in (y, dx, dw, db)]
    for t in (dw, db):
        t.t.zero_()
    assert lib.ctattn_linear_bwd(code, p(x), p(w), p(dy), p(dx), p(dw), p(db), ws.data_ptr(), ws.numel(), m, n, k, st) == 0
    torch.cuda.synchronize()
    x64, w64, dy64 = x.t.double(), w.t.double(), dy.t.double()
    close(y.t, x64 @ w64.T + b.t.double(), name, "y")
    close(dx.t, dy64 @ w64, name, "dx")
    close(dw.t, dy64.T @ x64, name, "dw")
    close(db.t, dy64.sum(0), name, "db")
    assert all(t.intact() for t in (x, w, b, dy, dw, db, y, dx))
    assert all(torch.equal(a, t.t) for a, t in zip(first, (y, dx, dw, db)))  # fixed order
    # Without room for the K splits (the least the entry point asks for) the product runs unsplit.
    assert lib.ctattn_linear_bwd(code, p(x), p(w), p(dy), p(dx), None, None, None, 0, m, n, k, st) == 0
    torch.cuda.synchronize()
    close(dx.t, dy64 @ w64, name, "dx without workspace")


@pytest.mark.parametrize("dims", [(2, 1, 40, 3, 8), (3, 37, 64, 2, 40), (2, 333, 136, 3, 48), (4, 65, 512, 8, 64)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_ragged_projections(name, dims):
    """Sequences that straddle the K stages of the weight gradients, heads that straddle those of
    the forward and dX (d = 40, 48)."""
    b, t, e, h, d = dims
    dt, hd = DT[name], h * d
    print(f"ragged projections {name} {dims}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(t)

    def rnd(*shape, std=1.0):
        return (std * torch.randn(shape, generator=g, device="cuda")).to(dt)

    def rows(v):
        return v.double().permute(0, 2, 1, 3).reshape(b * t, hd)

    x, ws = rnd(b, t, e), [rnd(hd, e, std=1 / math.sqrt(e)) for _ in range(3)]
    q = _capi.qkv_proj_fwd(x, *ws, None, None, None, h, d)
    x64 = x.double().reshape(b * t, e)
    grads = [rnd(b, h, t, d) for _ in range(3)]
    dw, db = tuple(torch.zeros_like(w) for w in ws), tuple(torch.zeros(hd, dtype=dt, device="cuda") for _ in ws)
    dx = _capi.qkv_proj_bwd(x, *grads, *ws, dw=dw, db=db)
    c, wo, dy = rnd(b, h, t, d), rnd(e, hd, std=1 / math.sqrt(hd)), rnd(b, t, e)
    dwo, dbo = torch.zeros_like(wo), torch.zeros(e, dtype=dt, device="cuda")
    y = _capi.out_proj_fwd(c, wo, None)
    dc = _capi.out_proj_bwd(c, dy, wo, dwo, dbo)
    torch.cuda.synchronize()
    dy64 = dy.double().reshape(b * t, e)
    for i in range(3):
        close(rows(q[i]), x64 @ ws[i].double().T, name, "qkv")
        close(dw[i], rows(grads[i]).T @ x64, name, "dw")
        close(db[i], rows(grads[i]).sum(0), name, "db")
    close(dx.reshape(b * t, e), sum(rows(gr) @ w.double() for gr, w in zip(grads, ws)), name, "dx")
    close(y.reshape(b * t, e), rows(c) @ wo.double().T, name, "y")
    close(rows(dc), dy64 @ wo.double(), name, "dc")
    close(dwo, dy64.T @ rows(c), name, "dwo")
    close(dbo, dy64.sum(0), name, "dbo")


# Stages taken whole and the last one not: every tile inside the matrix, one row or column past it, K
# at a stage, one more and one less.
@pytest.mark.parametrize("mnk", [(256, 128, 128), (129, 256, 127), (256, 257, 193), (1280, 1281, 64), (300, 128, 1087)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_ragged_linear_whole_stages(name, mnk):
    test_ragged_linear(name, mnk)


# Head-split stages inside one batch or head and across two: T and d at, past and below the stages.
@pytest.mark.parametrize("dims", [(3, 64, 260, 4, 64), (2, 130, 196, 3, 80), (3, 127, 256, 2, 128), (5, 96, 132, 4, 32)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_ragged_projections_whole_stages(name, dims):
    test_ragged_projections(name, dims)


@pytest.mark.parametrize("name", sorted(DT))
def test_dx_alone_leaves_the_workspace_alone(name):
    """A backward for dX alone may overlap, on another stream, a call that works in the same workspace:
    it writes none of it, in shapes whose dX splits K into the workspace of a call that also asks for
    the weight gradient, and gives the same dX as with no workspace at all."""
    print(f"dx alone {name}", flush=True)
    lib, code, dt = _capi.load(), _capi._DTYPE_CODE[DT[name]], DT[name]
    g = torch.Generator(device="cuda").manual_seed(5)

    def rnd(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(dt)

    st = torch.cuda.current_stream().cuda_stream
    ws = torch.full((64 << 20,), 0xA5, dtype=torch.uint8, device="cuda")

    def check(call, out):
        assert call(None, 0) == 0, _capi.last_error()
        torch.cuda.synchronize()
        plain = out.clone()
        out.zero_()
        assert call(ws.data_ptr(), ws.numel()) == 0, _capi.last_error()
        torch.cuda.synchronize()
        assert torch.equal(plain, out)
        assert bool((ws == 0xA5).all())

    m, n, k = 100, 5003, 256  # 8 tiles of 64 x 64, 79 or 157 stages of K
    dy, w, pre, dx = rnd(m, n), rnd(n, k), rnd(m, k), rnd(m, k)
    check(lambda p, b: lib.ctattn_linear_bwd(code, None, w.data_ptr(), dy.data_ptr(), dx.data_ptr(), None, None, p, b,
                                             m, n, k, st), dx)
    check(lambda p, b: lib.ctattn_linear_act_bwd(code, _capi.ACT_GELU, None, w.data_ptr(), dy.data_ptr(),
                                                 pre.data_ptr(), dx.data_ptr(), None, None, p, b, m, n, k, st), dx)
    b_, t, e, h, d = 1, 101, 1003, 8, 40
    x, gr, wq = rnd(b_, t, e), [rnd(b_, h, t, d) for _ in range(3)], [rnd(h * d, e) for _ in range(3)]
    dxp = torch.empty_like(x)
    args = [a.data_ptr() for a in (x, *gr, *wq)]
    check(lambda p, b: lib.ctattn_qkv_proj_bwd(code, *args, *[None] * 6, dxp.data_ptr(), p, b, b_, t, e, h, d, st), dxp)
    wo, dc = rnd(e, h * d), torch.empty_like(gr[0])
    check(lambda p, b: lib.ctattn_out_proj_bwd(code, None, x.data_ptr(), wo.data_ptr(), None, None, dc.data_ptr(), p, b,
                                               b_, t, e, h, d, st), dc)
