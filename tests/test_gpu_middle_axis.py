"""GPU parity of softmax / log_softmax over a middle axis (column tiles): every
launch shape of the kernel -- 4, 8 and 16 rows per lane in 256 lanes, 8 and 16
in 1024, the streaming one, each at 8 lanes per line; 16, 4, 2 and 1 lanes per
line as well; vectors moved back at a slab's edge -- and short axes with one lane
per column (4, 8 and 16 values per lane), against the oracle.
"""
import pytest
import torch

from dslperfgap_amd import _lib
from dslperfgap_amd.viperbench.log_softmax.hip_impl import log_softmax
from oracle import pytorch_impl as ref

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
CODE = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}
# fp32: sums of exps of up to 10000 rows in 32 bits and 1-ulp exp and log, at
# values up to about 30; 16-bit: half an ulp of the output
TOL = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}

SHAPES = [(3, n, i) for n in (1, 2, 4, 5, 33, 64, 65) for i in (2, 5, 8, 13, 64, 130)] + [
    (200, 3, 136), (200, 40, 136), (2, 513, 33), (30, 500, 64), (1, 1025, 40), (100, 1024, 16),
    (3, 2049, 9), (200, 2048, 8), (1, 9000, 20), (200, 2300, 9),
    # 8 and 16 lanes per line: 8 and 16 rows per lane in 256 lanes, then 8 and 16
    # rows in 1024, streaming; the smallest that the rule sends to each
    (260, 33, 257), (260, 33, 520), (260, 17, 520), (200, 129, 17), (100, 65, 65),
    (200, 513, 17), (200, 1025, 17), (200, 2049, 17), (200, 9000, 3), (1, 2049, 2), (1, 2049, 3)]
# one lane per column at every count of values per lane, and beyond it (narrow slabs
# of more than 6 or 8, the others of more than 10 or 16); a large launch in tiles
SHAPES += [(3, n, i) for n in (3, 6, 7, 8, 9, 10, 11, 16, 17) for i in (2, 3, 7, 13, 65)] + [
    (400, 8, 1024), (70000, 10, 12)]


def _input(shape, dtype):
    x = 3 * torch.randn(shape, generator=torch.Generator().manual_seed(411))
    x[0, shape[1] // 2, 0] = 25.0
    x[-1, :, 1] = -1e4  # far from 0
    x = x.to(dtype)
    if shape[2] > 4 and shape[1] > 1:
        x[0, 1, 2] = float("nan")
        x[0, 0, 3] = float("inf")
        x[-1, 1:, 4] = float("-inf")
        x[-1, :, 3] = float("-inf")
        x[-1, :, 2] = torch.finfo(dtype).min
    return x


@pytest.mark.parametrize("dtype,out", [(torch.float32, None), (torch.float16, None),
                                       (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_middle_axis_softmax(shape, dtype, out):
    x = _input(shape, dtype)
    xd = x.to(DEV)
    tol = TOL[out or dtype]
    got, want = log_softmax(xd, 1, out).cpu(), ref.log_softmax(x, 1, out)
    if shape[1] > 4096 and want.dtype == torch.float32:
        # the oracle adds up a column's exps one after the other in 32 bits: over
        # 9000 of them it is up to 1.39 of this tolerance off the result in 64 bits
        # (200 x 9000 x 3, these inputs)
        want = torch.log_softmax(x.double(), 1).float()
    assert got.dtype == want.dtype and got.shape == want.shape
    assert torch.allclose(got.float(), want.float(), atol=tol, rtol=tol, equal_nan=True)
    # softmax over a middle axis is reached through the C ABI only
    y = torch.empty(shape, dtype=out or dtype, device=DEV)
    _lib.call("vbh_softmax_dim_fwd", xd.data_ptr(), y.data_ptr(), *shape, CODE[dtype],
              CODE[out or dtype], 0, torch.cuda.current_stream().cuda_stream)
    want = torch.softmax(x.double(), 1)
    assert torch.allclose(y.cpu().double(), want, atol=tol, rtol=tol, equal_nan=True)
