"""The 32-row forward kernel of attn_fwd_mfma.hip (small fp32 grids, key blocks shared out over the
waves of a workgroup) and the edges of its rule, against float64 attention, with NaN around every
operand and output.

Tolerance: a score is a sum of d products of size |q| |k| / sqrt(d); d roundings of 2^-24 of the
growing sum, adding as a random walk, leave 8 |q| 2^-24 sqrt(d) at d = 128, |q| the spread of the
queries.  A probability's relative error is the score's, so o moves by as much of |v| < 5: 2e-5 |q|.
The log-sum-exp moves by the score's error and the rounding of its own size: 1e-5 |q|.
"""
import math

import pytest
import torch

from cudatransformer_amd import _capi

pytestmark = pytest.mark.gpu
PAD = 512


def guarded(shape, g=None, std=1.0):
    n = math.prod(shape)
    buf = torch.full((n + 2 * PAD,), float("nan"), device="cuda")
    t = buf[PAD:PAD + n].view(shape)
    t.copy_(torch.zeros(shape) if g is None else std * torch.randn(shape, generator=g, device="cuda"))
    return buf, t


# (B, H, T): single blocks and remainders, one block per wave and one more (8 waves; 4 at d = 128),
# the grid sizes around one, two, three and four workgroups per CU with T at the rule's edges.
SHAPES = [(1, 1, 32), (1, 1, 33), (2, 3, 63), (1, 2, 97), (1, 6, 128), (1, 2, 129), (1, 6, 255), (1, 6, 257),
          (1, 1, 1111), (1, 16, 512), (1, 17, 511), (1, 32, 512), (3, 11, 500), (1, 24, 1024), (2, 16, 1000)]


@pytest.mark.parametrize("bht", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128, 56])
def test_small_grid_forward(d, causal, bht):
    b, h, t = bht
    print(f"small grid forward d={d} causal={causal} B={b} H={h} T={t}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(b + h + t + d)
    qs = 8.0 if t % 2 else 1.0  # wide scores: the waves' maxima lie far apart
    ops = [guarded((b, h, t, d), g, qs), guarded((b, h, t, d), g), guarded((b, h, t, d), g)]
    outs = [guarded((b, h, t, d)), guarded((b, h, t))]
    (q, k, v), (o, lse) = [x for _, x in ops], [x for _, x in outs]
    _capi.flash_attn_fwd(q, k, v, causal, out=o, lse=lse)
    o2, lse2 = _capi.flash_attn_fwd(q, k, v, causal)
    torch.cuda.synchronize()
    s = q.double() @ k.double().transpose(-1, -2).contiguous() / math.sqrt(d)
    if causal:
        s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    assert (o.double() - torch.softmax(s, -1) @ v.double()).abs().max() <= 2e-5 * qs
    assert (lse.double() - torch.logsumexp(s, -1)).abs().max() <= 1e-5 * qs
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    for buf, x in ops + outs:
        assert torch.isnan(buf[:PAD]).all() and torch.isnan(buf[PAD + x.numel():]).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_small_grid_forward_infinite_keys(d, causal):
    """Key blocks whose every score is -inf add nothing, also where they are the first block of a wave."""
    b, h, t = 1, 2, 400
    print(f"small grid forward, infinite keys d={d} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(d)
    q, k, v = [torch.randn((b, h, t, d), generator=g, device="cuda") for _ in range(3)]
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, :, 32:96, 0] = float("-inf")
    k[:, :, 352:, 0] = float("-inf")
    o, lse = _capi.flash_attn_fwd(q, k, v, causal)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) / math.sqrt(d)
    if causal:
        s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    assert (o.double() - torch.softmax(s, -1) @ v.double()).abs().max() <= 2e-5
    assert (lse.double() - torch.logsumexp(s, -1)).abs().max() <= 1e-5
