"""Head dims above 128 (a multiple of 8) on the MFMA kernels of attn_wide.hip, against the generic
kernels (POLICY_GENERIC) on the same inputs and forward state.

Both sides accumulate in fp32, and P and dS keep 24 significant bits (fp32, and bf16 as three
terms) or 22 (fp16 as two), so before the one rounding to storage they differ by an error
e < 1e-5 of the result's norm.  At fp32 that is the tolerance.  At 16 bits with unit roundoff u a
value changes by one step (2u) only when e crosses a rounding boundary, a share e / 2u of the
values: a norm of sqrt(e / 2u) 2u = sqrt(2 u e), 2e-4 for bf16 (u = 2^-9) and 1e-4 for fp16
(u = 2^-11); twice that is allowed.
"""
import pytest
import torch

import cudatransformer_amd as ct

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"f32": 1e-5, "bf16": 4e-4, "f16": 2e-4}


def inputs(shape, name, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [(std * torch.randn(shape, generator=g, device="cuda")).to(DT[name]) for _ in range(4)]


def both(x, causal):
    """(MFMA, generic) outputs, the backward of both from the generic forward's O and LSE."""
    q, k, v, do = x
    out = []
    prev = ct.set_policy(ct.POLICY_GENERIC)
    try:
        og, lg = ct.flash_attn_fwd(q, k, v, causal)
        gen = dict(zip(("o", "lse", "dq", "dk", "dv"), (og, lg, *ct.flash_attn_bwd(q, k, v, og, do, lg, causal))))
    finally:
        ct.set_policy(prev)
    o, lse = ct.flash_attn_fwd(q, k, v, causal)
    out = dict(zip(("o", "lse", "dq", "dk", "dv"), (o, lse, *ct.flash_attn_bwd(q, k, v, og, do, lg, causal))))
    torch.cuda.synchronize()
    return out, gen


def check(got, want, name):
    floor = want["dv"].double().norm()  # dQ and dK of a row with one key vanish
    for key in want:
        w, g = want[key].double(), got[key].double()
        tol = 1e-5 if key == "lse" else TOL[name]
        err = (g - w).norm() / torch.maximum(w.norm(), floor if key in ("dq", "dk") else w.norm())
        assert err <= tol, (key, float(err))


@pytest.mark.parametrize("shape", [(1, 2, 8, 256), (2, 1, 31, 160), (1, 2, 33, 192), (1, 3, 64, 256), (1, 1, 97, 136),
                                   (2, 2, 200, 200), (1, 3, 161, 160), (2, 1, 129, 192), (1, 2, 333, 256)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("name", sorted(DT))
def test_wide_matches_generic(name, causal, shape):
    print(f"wide heads {name} causal={causal} {shape}", flush=True)
    x = inputs(shape, name, seed=sum(shape))
    got, want = both(x, causal)
    check(got, want, name)
    again, _ = both(x, causal)
    assert all(torch.equal(got[k], again[k]) for k in got)  # no atomics


@pytest.mark.parametrize("std", [2e-4, 30.0])
def test_wide_f16_range(std):
    """dS far below and above 1: the fp16 split keeps its precision over fp16's inputs."""
    print(f"wide heads f16 gradient scale {std}", flush=True)
    x = inputs((1, 2, 130, 256), "f16", seed=7)
    x[3] = (x[3].float() * std).half()
    got, want = both(x, True)
    # dV and dK of a small dO are fp16 subnormals on both sides: compare what is above them.
    for key in ("dq", "dk", "dv"):
        w, g = want[key].double(), got[key].double()
        err = ((g - w).abs() - 2.0 ** -24).clamp_min(0).norm() / w.norm()
        assert err <= TOL["f16"], (key, float(err))


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("name", sorted(DT))
def test_wide_nonfinite_inputs(name, causal):
    """An infinity and a NaN reach exactly the outputs they reach in the generic kernels: under a
    causal mask not the rows before theirs, though those share a tile with it."""
    print(f"wide heads non-finite {name} causal={causal}", flush=True)
    x = inputs((1, 2, 110, 256), name, seed=3)
    x[2][0, 0, 40, 5] = float("inf")
    x[1][0, 1, 50, 7] = float("nan")
    x[3][0, 0, 20, 9] = float("inf")
    got, want = both(x, causal)
    for key in want:
        g, w = got[key].double(), want[key].double()
        assert torch.equal(torch.isnan(g), torch.isnan(w)), key
        assert torch.equal(torch.isinf(g), torch.isinf(w)), key
        ok = torch.isfinite(w)
        err = (g[ok] - w[ok]).norm() / w[ok].norm().clamp_min(1e-30)
        assert err <= max(TOL[name], 1e-5), (key, float(err))


def reference(x, causal, dtype):
    """O, LSE in float64, and dQ, dK, dV in float64 from O rounded to `dtype` and LSE to fp32."""
    q, k, v, do = (t.double() for t in x)
    T, scale = q.shape[2], q.shape[3] ** -0.5
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    lse = torch.logsumexp(s, -1)
    o = torch.matmul(torch.exp(s - lse[..., None]), v)
    o_in, lse_in = o.to(dtype), lse.float()
    p = torch.exp(s - lse_in.double()[..., None])
    delta = (do * o_in.double()).sum(-1, keepdim=True)
    ds = p * (torch.matmul(do, v.transpose(-1, -2).contiguous()) - delta)
    grads = (torch.matmul(ds, k) * scale, torch.matmul(ds.transpose(-1, -2).contiguous(), q) * scale,
             torch.matmul(p.transpose(-1, -2).contiguous(), do))
    return o, lse, o_in, lse_in, dict(zip(("dq", "dk", "dv"), grads))


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("name", ["bf16", "f16"])
def test_wide_rounds_as_often_right_as_generic(name, causal):
    """The error before the rounding to 16 bits, from the share of outputs that are not the
    float64 result rounded once (proportional to it): no larger than the generic kernels', which
    keep P and dS in fp32.  262144 outputs and shares from 0.04 % make 100 expected, 10 % of
    standard deviation: a third more is allowed.  (P and dS of 16 significant bits give five
    times the generic share in bf16.)"""
    print(f"wide heads rounding {name} causal={causal}", flush=True)
    x = inputs((1, 2, 512, 256), name, seed=11)
    o, _, o_in, lse_in, grads = reference(x, causal, DT[name])
    q, k, v, do = x

    def shares():
        got = {"o": ct.flash_attn_fwd(q, k, v, causal)[0]}
        got.update(zip(("dq", "dk", "dv"), ct.flash_attn_bwd(q, k, v, o_in, do, lse_in, causal)))
        want = {"o": o, **grads}
        return {key: float((got[key] != want[key].to(DT[name])).double().mean()) for key in want}

    wide = shares()
    prev = ct.set_policy(ct.POLICY_GENERIC)
    try:
        generic = shares()
    finally:
        ct.set_policy(prev)
    for key in wide:
        assert wide[key] <= 4 / 3 * generic[key], (key, wide[key], generic[key])


UNIT = {"f32": 0.0, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}  # most that one rounding to storage changes a value


def rel(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("a", [1.1, 1.4, 2.6])  # mean row LSE about -14, -26, -103
@pytest.mark.parametrize("shape", [(1, 2, 33, 160), (1, 2, 33, 256), (1, 2, 97, 160), (1, 2, 97, 256)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(DT))
def test_wide_rows_past_the_end_do_not_reach_dk(name, shape, a):
    """Queries that oppose an offset the keys share (row LSE far below 0) at a T that leaves the
    last 32-key tile partly empty: the empty keys' scores are 0, so exp(0 - LSE) there is up to
    e^103, and must not move the scale of the fp16 dS of the keys beside them.  dK against
    float64, keys of the partial tile by themselves: a unit roundoff u and the fp32 error of
    scores of up to 2000 (1e-4)."""
    print(f"wide heads negative LSE {name} {shape} {a}", flush=True)
    x = inputs(shape, name, seed=13)
    x[0] = (x[0].float() - a).to(DT[name])
    x[1] = (x[1].float() + a).to(DT[name])
    _, lse, o_in, lse_in, grads = reference(x, False, DT[name])
    assert float(lse.max()) < 0
    q, k, v, do = x
    got = dict(zip(("dq", "dk", "dv"), ct.flash_attn_bwd(q, k, v, o_in, do, lse_in, False)))
    tol = UNIT[name] + 1e-4
    tail = shape[2] // 32 * 32
    assert rel(got["dk"][:, :, tail:], grads["dk"][:, :, tail:]) <= tol
    for key in grads:
        assert rel(got[key], grads[key]) <= tol, key


def check64(x, causal, name):
    """All outputs against float64: one rounding to storage and the fp32 error of scores of up to
    1000 (1e-4)."""
    o, lse, o_in, lse_in, grads = reference(x, causal, DT[name])
    q, k, v, do = x
    got_o, got_lse = ct.flash_attn_fwd(q, k, v, causal)
    got = dict(zip(("dq", "dk", "dv"), ct.flash_attn_bwd(q, k, v, o_in, do, lse_in, causal)))
    assert rel(got_lse, lse) <= 1e-5
    for key, want in {"o": o, **grads}.items():
        assert rel({"o": got_o, **got}[key], want) <= UNIT[name] + 1e-4, key


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("name", sorted(DT))
def test_wide_running_max_grows(name, causal):
    """Scores that rise by 6 with every 32 keys (9 in log2 units): the running max passes its
    first block's by more than 2^8 again and again."""
    print(f"wide heads growing scores {name} causal={causal}", flush=True)
    x = inputs((1, 2, 333, 256), name, seed=17)
    x[0] = (x[0].float() + 1).to(DT[name])
    x[1] = (x[1].float() + torch.linspace(0, 4, 333, device="cuda")[:, None]).to(DT[name])
    check64(x, causal, name)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("name", sorted(DT))
def test_wide_gradients_grow_along_the_sequence(name, causal):
    """dO and V grow by 2^14 and 2^12 along the sequence, so the running scale of the fp16 dS has to
    come down several times in the dK and dQ passes."""
    print(f"wide heads growing gradients {name} causal={causal}", flush=True)
    x = inputs((1, 2, 333, 256), name, seed=19)
    x[2] = (x[2].float() * torch.logspace(-8, 4, 333, 2.0, device="cuda")[:, None]).to(DT[name])
    x[3] = (x[3].float() * torch.logspace(-12, 2, 333, 2.0, device="cuda")[:, None]).to(DT[name])
    check64(x, causal, name)


@pytest.mark.parametrize("name", sorted(DT))
def test_wide_gradients_on_their_inputs(name):
    """dK and dV written onto K and V: the generic kernels' results, which such calls run on."""
    print(f"wide heads gradients on inputs {name}", flush=True)
    q, k, v, do = inputs((2, 2, 150, 160), name, seed=23)
    o, lse = ct.flash_attn_fwd(q, k, v, True)
    prev = ct.set_policy(ct.POLICY_GENERIC)
    try:
        want = ct.flash_attn_bwd(q, k, v, o, do, lse, True)
    finally:
        ct.set_policy(prev)
    k2, v2 = k.clone(), v.clone()
    got = ct.flash_attn_bwd(q, k2, v2, o, do, lse, True, dk=k2, dv=v2)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
