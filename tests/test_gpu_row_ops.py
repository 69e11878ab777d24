"""LayerNorm, softmax and the fused softmax-cross-entropy gradient at the edges of their row
kernels: waves per row, 16-byte granules per lane, rows off 16-byte boundaries (odd lengths, a
tensor one element into its storage), and the lengths past which the general kernels take over,
against float64.

Tolerance: fp32 sums of up to 66000 terms, 1e-5 relative; 16-bit outputs round once more, at most
2^-8 (bf16) or 2^-11 (fp16) of a value, so of the 2-norm too; dgamma / dbeta accumulate in storage
from 0 and round once.
"""
import pytest
import torch

from cudatransformer_amd import _capi

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"f32": 1e-5, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}


def rnd(shape, dt, seed, std=1.0, shift=0.0, offset=1):
    """Random values `offset` elements past a 16-byte boundary."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = 1
    for s in shape:
        n *= s
    buf = torch.empty(n + 16, dtype=dt, device="cuda")
    t = buf[offset:offset + n].view(shape)
    t.copy_(shift + std * torch.randn(shape, generator=g, device="cuda"))
    return t


def close(got, want, tol, what):
    err = (got.double() - want).norm() / want.norm().clamp_min(1e-30)
    assert err <= tol, (what, float(err))


@pytest.mark.parametrize("d", [1, 7, 64, 255, 256, 511, 512, 513, 1024, 1029, 2048, 2056, 4096, 4100, 8192, 8200])
@pytest.mark.parametrize("name", sorted(DT))
def test_layernorm_edges(name, d):
    dt, n = DT[name], 37  # one full 32-row chunk and a ragged one
    print(f"layernorm {name} D={d}", flush=True)
    for offset in (0, 1):
        x, dy = rnd((n, d), dt, 1, 2.0, 0.5, offset), rnd((n, d), dt, 2, offset=offset)
        g, b = rnd((d,), dt, 3, 0.1, 1.0, offset), rnd((d,), dt, 4, 0.1, 0.0, offset)
        y, mean, rstd = _capi.layernorm_fwd(x, g, b)
        dg, db = torch.zeros_like(g), torch.zeros_like(b)
        dx = _capi.layernorm_bwd(x, g, dy, mean, rstd, dg, db)
        torch.cuda.synchronize()
        x64, g64, b64, dy64 = x.double(), g.double(), b.double(), dy.double()
        mu = x64.mean(-1, keepdim=True)
        rs = torch.rsqrt(((x64 - mu) ** 2).mean(-1, keepdim=True) + 1e-5)
        xh = (x64 - mu) * rs
        dxh = dy64 * g64
        close(mean, mu[:, 0], 1e-5, "mean")
        close(rstd, rs[:, 0], 1e-5, "rstd")
        close(y, xh * g64 + b64, TOL[name], "y")
        # D = 1: dx vanishes; its scale is the terms that cancel.
        want = rs * (dxh - dxh.mean(-1, keepdim=True) - xh * (dxh * xh).mean(-1, keepdim=True))
        scale = (rs * dxh).norm()
        assert ((dx.double() - want).norm() / scale) <= TOL[name], "dx"
        if d > 1:
            close(dg, (dy64 * xh).sum(0), TOL[name], "dgamma")
        close(db, dy64.sum(0), TOL[name], "dbeta")


@pytest.mark.parametrize("d", [96, 101, 200])
def test_layernorm_bwd_large_constant_rows(d):
    """Rows of one value 2^120: the statistics are exact (variance 0), but -mean rstd overflows, which
    must stay out of the sums over the columns (lanes past the row's end hold zeros)."""
    print(f"layernorm large rows D={d}", flush=True)
    for name in ("f32", "bf16"):
        dt = DT[name]
        x = torch.full((5, d), 2.0 ** 120, device="cuda").to(dt)
        g, dy = rnd((d,), dt, 3, 0.1, 1.0), rnd((5, d), dt, 2)
        _, mean, rstd = _capi.layernorm_fwd(x, g, torch.zeros_like(g))
        dx = _capi.layernorm_bwd(x, g, dy, mean, rstd)
        torch.cuda.synchronize()
        assert bool((mean == 2.0 ** 120).all())
        dxh = dy.double() * g.double()
        close(dx, rstd.double()[:, None] * (dxh - dxh.mean(-1, keepdim=True)), TOL[name], "dx")


@pytest.mark.parametrize("nd", [(5, 65), (37, 300), (5, 600), (2100, 1100), (4100, 1100), (4100, 3000), (4100, 5000)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", ["f32", "bf16"])
def test_layernorm_bwd_given_large_statistics(name, nd):
    """The same with given statistics, for rows of one and of several waves, dx with the partial sums and by
    itself, and written onto x; a NaN in a row stays in that row's dx."""
    n, d = nd
    dt = DT[name]
    print(f"layernorm given statistics {name} {n} x {d}", flush=True)
    x = torch.full((n, d), 2.0 ** 120, device="cuda").to(dt)
    g, dy = rnd((d,), dt, 3, 0.1, 1.0), rnd((n, d), dt, 2)
    dy[1, d - 1] = float("nan")
    mean, rstd = torch.full((n,), 2.0 ** 120, device="cuda"), torch.full((n,), 2.0 ** 9, device="cuda")
    dg, db = torch.zeros_like(g), torch.zeros_like(g)
    dx = _capi.layernorm_bwd(x, g, dy, mean, rstd, dg, db)
    alone = _capi.layernorm_bwd(x, g, dy, mean, rstd)
    torch.cuda.synchronize()
    ok = [i for i in range(n) if i != 1]
    assert bool(dx[1].isnan().all()) and torch.equal(alone[ok], dx[ok])
    dxh = dy.double() * g.double()
    close(dx[ok], (2.0 ** 9 * (dxh - dxh.mean(-1, keepdim=True)))[ok], TOL[name], "dx")
    assert bool((dg[:-1] == 0).all()) and bool(dg[-1].isnan()) and bool(db[-1].isnan())
    close(db[:-1], dy.double().sum(0)[:-1], TOL[name], "dbeta")
    code, lib = _capi._DTYPE_CODE[dt], _capi.load()
    assert lib.ctattn_layernorm_bwd(code, x.data_ptr(), g.data_ptr(), dy.data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                                    x.data_ptr(), None, None, None, 0, n, d, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(x[ok], dx[ok])


@pytest.mark.parametrize("v", [1, 3, 65, 256, 257, 512, 1025, 2048, 4097, 8193, 16385, 32769, 65536, 65537])
@pytest.mark.parametrize("name", sorted(DT))
def test_softmax_and_gradient_edges(name, v):
    dt, n = DT[name], 6
    print(f"softmax {name} V={v}", flush=True)
    z = rnd((n, v), dt, 5, 3.0)
    if v > 3:
        z[1, 2:] = float("-inf")  # masked classes
        z[2] = torch.finfo(dt).min  # a row at the type's lowest value
    t = torch.randint(0, v, (n,), device="cuda", dtype=torch.int32)
    t[3], t[4] = -1, v
    p = _capi.softmax_fwd(z, 0.7)
    dz = _capi.softmax_cross_entropy_bwd(p, t, 0.7)
    torch.cuda.synchronize()
    want = torch.softmax(z.double() / 0.7, -1)
    # fp16: probabilities below its subnormals' half step round to 0.
    floor = 2.0 ** -25 if name == "f16" else 0.0
    assert ((p.double() - want).abs() <= TOL[name] * want + floor + 1e-5 * (name == "f32") * want).all()
    onehot = torch.zeros_like(want)
    ok = (t >= 0) & (t < v)
    onehot[ok.nonzero()[:, 0], t[ok].long()] = 1.0
    ref = (p.double() - onehot) * ok[:, None] / (n * 0.7)
    assert ((dz.double() - ref).abs() <= TOL[name] * ref.abs() + floor + 1e-7).all()


@pytest.mark.parametrize("temperature", [3e38, 1e39, float("inf")])
@pytest.mark.parametrize("v", [5, 129, 3001])
def test_softmax_temperatures_past_fp32(v, temperature):
    """A temperature whose fp32 reciprocal is subnormal or 0: every class alike, at lengths off the granules."""
    print(f"softmax V={v} temperature={temperature}", flush=True)
    for name, dt in DT.items():
        p = _capi.softmax_fwd(rnd((3, v), dt, 7), temperature)
        assert ((p.double() * v - 1).abs() <= TOL[name] + (2.0 ** -25 * v if name == "f16" else 0)).all()


# The first length past each number of waves per row, and several past the row kernels.
@pytest.mark.parametrize("d", [1025, 2049, 4097, 8193, 9001, 16390])
@pytest.mark.parametrize("name", sorted(DT))
def test_layernorm_past_the_edges(name, d):
    test_layernorm_edges(name, d)


def test_softmax_exponential_ulps():
    """The softmax's exponential through rows (0, x) in fp32, in units in the last place of the result.
    Below -18 the probability of x is e^x itself: 1 ulp of the hardware's exp2 and 2 x 2^-26 of its
    argument's fraction (0.7 ulp), results in the subnormals rounded once more (half a step).  Above,
    the sum, its reciprocal and the product add 0.5, 1 and 0.5 ulp, and e^x enters twice: 6."""
    print("softmax exponential", flush=True)
    x = torch.cat([torch.linspace(-110, -18, 200001), torch.linspace(-18, 0, 200001)]).cuda()
    p = _capi.softmax_fwd(torch.stack([torch.zeros_like(x), x], 1))[:, 1]
    torch.cuda.synchronize()
    want = torch.softmax(torch.stack([torch.zeros_like(x), x], 1).double(), 1)[:, 1]
    ulp = torch.exp2(torch.floor(torch.log2(want)).clamp_min(-126) - 23)
    err = (p.double() - want).abs() / ulp
    print(f"largest {float(err[x < -18].max()):.2f} and {float(err[x >= -18].max()):.2f} ulp", flush=True)
    assert float(err[x < -18].max()) <= 2.2
    assert float(err.max()) <= 6
    assert bool((p[x < -104] == 0).all())  # e^x below half of 2^-149


@pytest.mark.parametrize("nd", [(8192, 65), (8193, 65), (16384, 128), (16385, 128), (16385, 129),
                                (8193, 250), (8193, 384), (8193, 448), (8193, 513), (8193, 896),
                                (2048, 1032), (2049, 1032), (4096, 1032), (4097, 1032), (4096, 2052), (4097, 2052),
                                (2049, 4100), (4097, 4100)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_layernorm_bwd_one_pass_or_two(name, nd):
    """Both sides of the lines in N and D between dx with the partial sums in one pass and dx by itself,
    against float64; each output alone and dx written onto dy: the same bits."""
    n, d = nd
    dt, code, lib = DT[name], _capi._DTYPE_CODE[DT[name]], _capi.load()
    print(f"layernorm backward {name} {n} x {d}", flush=True)
    x, dy = rnd((n, d), dt, 1, 2.0, 0.5), rnd((n, d), dt, 2)
    g = rnd((d,), dt, 3, 0.1, 1.0)
    _, mean, rstd = _capi.layernorm_fwd(x, g, torch.zeros_like(g))
    ws = torch.empty(lib.ctattn_layernorm_bwd_workspace_bytes(code, n, d), dtype=torch.uint8, device="cuda")

    def bwd(want_dx, want_g):
        dx, dg, db = torch.zeros_like(x), torch.zeros_like(g), torch.zeros_like(g)
        rc = lib.ctattn_layernorm_bwd(code, x.data_ptr(), g.data_ptr(), dy.data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                                      dx.data_ptr() if want_dx else None, dg.data_ptr() if want_g else None,
                                      db.data_ptr() if want_g else None, ws.data_ptr() if want_g else None,
                                      ws.numel() if want_g else 0, n, d, None)
        assert rc == 0, _capi.last_error()
        torch.cuda.synchronize()
        return dx, dg, db

    dx, dg, db = bwd(True, True)
    assert torch.equal(bwd(True, False)[0], dx)
    assert all(torch.equal(a, b) for a, b in zip(bwd(False, True)[1:], (dg, db)))
    dy2, dg2, db2 = dy.clone(), torch.zeros_like(g), torch.zeros_like(g)  # dx onto dy
    assert lib.ctattn_layernorm_bwd(code, x.data_ptr(), g.data_ptr(), dy2.data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                                    dy2.data_ptr(), dg2.data_ptr(), db2.data_ptr(), ws.data_ptr(), ws.numel(), n, d,
                                    None) == 0
    torch.cuda.synchronize()
    assert torch.equal(dy2, dx) and torch.equal(dg2, dg) and torch.equal(db2, db)
    x64, dy64, mu, rs = x.double(), dy.double(), mean.double()[:, None], rstd.double()[:, None]
    xh, dxh = (x64 - mu) * rs, dy64 * g.double()
    close(dx, rs * (dxh - dxh.mean(-1, keepdim=True) - xh * (dxh * xh).mean(-1, keepdim=True)), TOL[name], "dx")
    close(dg, (dy64 * xh).sum(0), TOL[name], "dgamma")
    close(db, dy64.sum(0), TOL[name], "dbeta")
