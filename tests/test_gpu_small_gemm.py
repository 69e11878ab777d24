"""The 32 x 32-tile plans of linear_gemm.hip for small grids, at the edges of their rule: forward,
forward with its activation and dX against float64 products of the same rounded inputs, with NaN
around every operand and output.

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
