"""The 32 x 32-tile plans of linear_gemm.hip for small grids, at the edges of their rule: forward,
forward with its activation and dX against float64 products of the same rounded inputs, with NaN
around every operand and output; and both sides of the lines between the ragged kernels' tiles and
between them and the projection family.

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
PAD = 512

# One tile and less; tile edges; 256 / 272 and 384 / 400 tiles at a long contraction; 768 / 800
# tiles at contractions of 512 and just above (the same sets transposed serve dX).
SHAPES = [(1, 16, 32), (1, 32, 64), (31, 48, 96), (33, 80, 544), (65, 1040, 512), (512, 512, 544), (544, 512, 1024),
          (512, 768, 2048), (512, 800, 2048), (1024, 768, 512), (1024, 768, 544), (1024, 800, 512),
          (512, 2048, 512), (33, 512, 1040)]


def guarded(shape, dt, g=None, std=1.0):
    n = math.prod(shape)
    buf = torch.full((n + 2 * PAD,), float("nan"), dtype=dt, device="cuda")
    t = buf[PAD:PAD + n].view(shape)
    t.copy_(torch.zeros(shape) if g is None else std * torch.randn(shape, generator=g, device="cuda"))
    return buf, t


@pytest.mark.parametrize("mnk", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_small_grid_linear(name, mnk):
    m, n, k = mnk
    dt, code = DT[name], _capi._DTYPE_CODE[DT[name]]
    print(f"small grid {name} M={m} N={n} K={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    ops = [guarded((m, k), dt, g), guarded((n, k), dt, g, 1 / math.sqrt(k)), guarded((n,), dt, g),
           guarded((m, n), dt, g, 1 / math.sqrt(n))]
    outs = [guarded((m, n), dt), guarded((m, n), dt), guarded((m, n), dt), guarded((m, k), dt)]
    (x, w, b, dy), (y, pre, post, dx) = [t for _, t in ops], [t for _, t in outs]
    lib, st = _capi.load(), torch.cuda.current_stream().cuda_stream
    p = lambda t: t.data_ptr()  # noqa: E731
    assert lib.ctattn_linear_fwd(code, p(x), p(w), p(b), p(y), m, n, k, st) == 0
    assert lib.ctattn_linear_act_fwd(code, 0, p(x), p(w), p(b), p(pre), p(post), m, n, k, st) == 0
    assert lib.ctattn_linear_bwd(code, p(x), p(w), p(dy), p(dx), None, None, None, 0, m, n, k, st) == 0
    torch.cuda.synchronize()
    for got, want, what in ((y, x.double() @ w.double().T + b.double(), "y"), (dx, dy.double() @ w.double(), "dx")):
        err = (got.double() - want).abs().max() / want.abs().max().clamp_min(1e-30)
        assert err <= TOL[name], (what, float(err))
    assert torch.equal(pre, y) and torch.equal(post, y.relu())
    for buf, t in ops + outs:
        assert torch.isnan(buf[:PAD]).all() and torch.isnan(buf[PAD + t.numel():]).all()


def close(got, want, name):
    err = (got.double() - want).abs().max() / want.abs().max()
    assert err <= TOL[name], float(err)


def against_float64(name, m, n, k, grads):
    """Forward, dX (and with `grads` dW, db) of one linear layer on aligned tensors against float64, and
    the fused activation's results against the two calls' it stands for, bit for bit."""
    dt = DT[name]
    print(f"route {name} {m} {n} {k} grads={grads}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w, dy, b = ((std * torch.randn(shape, generator=g, device="cuda")).to(dt)
                   for shape, std in (((m, k), 1.0), ((n, k), k ** -0.5), ((m, n), 1.0), ((n,), 0.1)))
    dw, db = (torch.zeros_like(w), torch.zeros(n, dtype=dt, device="cuda")) if grads else (None, None)
    y = _capi.linear_fwd(x, w, b)
    dx = _capi.linear_bwd(x, w, dy, dw, db)
    pre, h = _capi.linear_act_fwd(x, w, b, _capi.ACT_GELU)
    dwa, dba = (torch.zeros_like(w), torch.zeros_like(db)) if grads else (None, None)
    dpre = _capi.linear_act_bwd(x, w, dy, x, _capi.ACT_GELU, dw=dwa, db=dba)
    torch.cuda.synchronize()
    x64, w64, dy64 = x.double(), w.double(), dy.double()
    close(y, x64 @ w64.T + b.double(), name)
    close(dx, dy64 @ w64, name)
    if grads:
        close(dw, dy64.T @ x64, name)
        close(db, dy64.sum(0), name)
    assert torch.equal(pre, y) and torch.equal(h, _capi.activation_fwd(y, _capi.ACT_GELU))
    assert torch.equal(dpre, _capi.activation_bwd(x, dx, _capi.ACT_GELU))


# fp32 sizes that are multiples of 4 and not of the K chunk: forwards of 32 rows and more (contraction 516 and
# 508), a dX of 256 tiles of 64 x 64 and of more, contractions of 2 and of more K splits.
@pytest.mark.parametrize("mnk", [(32, 100, 516), (36, 100, 516), (32, 100, 508), (4, 1000, 1000), (1024, 500, 1000),
                                 (1028, 500, 1000), (64, 132, 64), (64, 300, 64)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("grads", [False, True], ids=["dx", "all"])
def test_f32_products_off_the_chunk(mnk, grads):
    against_float64("f32", *mnk, grads)


# 210 and 225 tiles of 128 x 128 (rounds of CUs 82 and 88 % full).
@pytest.mark.parametrize("mnk", [(1700, 1900, 70), (1900, 1900, 70)], ids=lambda s: "x".join(map(str, s)))
def test_f32_ragged_tile_choice(mnk):
    against_float64("f32", *mnk, True)


# 384 tiles of 32 x 32 at a contraction of 1536 and past it.
@pytest.mark.parametrize("mnk", [(192, 2048, 1536), (192, 2048, 1568), (192, 1536, 2048)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", ["bf16", "f16"])
def test_small_grid_contractions(name, mnk):
    against_float64(name, *mnk, True)


# Up to and past 256 tiles of 64 x 64, stacked batches and not, the last launch of three with fewer.
@pytest.mark.parametrize("shape", [(1, 1, 1024, 1000, 1000), (1, 1, 1028, 1000, 1000), (4, 1, 28, 1000, 100),
                                   (4, 4, 28, 1000, 100), (4, 4, 512, 132, 1024), (2, 2, 1024, 68, 516)],
                         ids=lambda s: "x".join(map(str, s)))
def test_f32_matmul_off_the_chunk(shape):
    batch, batch_b, m, k, n = shape
    print(f"matmul f32 {shape}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(k)
    a = torch.randn((batch, m, k), generator=g, device="cuda")
    b = torch.randn((batch_b, k, n), generator=g, device="cuda")
    c = torch.empty((batch, m, n), device="cuda")
    assert _capi.load().ctattn_tensor_matmul(0, a.data_ptr(), b.data_ptr(), c.data_ptr(), batch, batch_b, m, k, n,
                                             torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    close(c, a.double() @ b.double(), "f32")
