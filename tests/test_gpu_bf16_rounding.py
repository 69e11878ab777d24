"""fp32 -> bf16 storage rounds to nearest even at every edge: the cast's values against torch's on the
CPU, bit for bit (NaN stays NaN), over every upper half of a float with the lower halves around 0, the
tie and the carry."""
import pytest
import torch

from cudatransformer_amd import _capi

pytestmark = pytest.mark.gpu


def test_fp32_to_bf16_rounding():
    hi = torch.arange(1 << 16, dtype=torch.int64)[:, None] << 16
    lo = torch.tensor([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF])[None]
    bits = (hi | lo).reshape(-1)
    x = (bits - ((bits >> 31) << 32)).to(torch.int32).view(torch.float32)
    xd = x.cuda()
    y = torch.empty(x.shape, dtype=torch.bfloat16, device="cuda")
    rc = _capi.load().ctattn_tensor_cast(_capi._DTYPE_CODE[torch.float32], xd.data_ptr(),
                                         _capi._DTYPE_CODE[torch.bfloat16], y.data_ptr(), x.numel(),
                                         torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    got, want = y.cpu(), x.to(torch.bfloat16)
    nan = torch.isnan(x)
    assert torch.isnan(got[nan]).all()
    assert torch.equal(got[~nan].view(torch.int16), want[~nan].view(torch.int16))
