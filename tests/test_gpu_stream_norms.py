"""GPU parity of the streaming LayerNorm / RMSNorm kernels (rows beyond the
registers): batches of four vectors per lane, with a whole last batch, a partial
one and a partial vector's lane count, unaligned rows, and rows far from 0,
against torch in 64 bits.
"""
import pytest
import torch

from dslperfgap_amd.viperbench.layer_norm.hip_impl import layer_norm
from dslperfgap_amd.viperbench.rms_norm.hip_impl import rms_norm

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# outputs up to about 6: fp32 sums of up to 140000 terms in pairs and batches, or
# half an ulp of the output type and of the weights' products
TOL = {torch.float32: 2e-5, torch.float16: 4e-3, torch.bfloat16: 3e-2}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cols", [65544, 70001, 98304, 131072, 131080, 139272])
def test_streaming_norms(cols, dtype):
    g = torch.Generator().manual_seed(451)
    x = 2 * torch.randn(3, cols, generator=g) + 0.5
    x[1] += 100.0
    x[2] *= 0.01
    x = x.to(dtype)
    w = (1 + 0.1 * torch.randn(cols, generator=g)).to(dtype)
    b = (0.1 * torch.randn(cols, generator=g)).to(dtype)
    xd, w64, x64 = x.to(DEV), w.double(), x.double()
    d = x64 - x64.mean(1, keepdim=True)
    ln = d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-5) * w64
    rms = x64 / torch.sqrt((x64 * x64).mean(1, keepdim=True) + 1e-5) * w64
    tol = TOL[dtype]
    for got, want in ((layer_norm(xd, w.to(DEV), b.to(DEV)), ln + b.double()),
                      (layer_norm(xd, w.to(DEV).float(), None), ln),
                      (rms_norm(xd, (cols,), w.to(DEV)), rms)):
        assert got.dtype == dtype
        assert torch.allclose(got.cpu().double(), want, atol=tol, rtol=tol)
