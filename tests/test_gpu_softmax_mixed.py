"""GPU parity of the softmax row kernels' vector shapes: 16-bit rows written as
fp32 (4 elements per lane access: row widths around multiples of 4 and 8, one
vector, one wave, several waves, the streaming kernel, split rows; 8 elements in
large launches of short rows), fp32 softmax
rows of 64 values per lane (near and far from 0), and streaming rows of every
type with special values, against torch in 64 bits: over rows this long the
oracle's own 32-bit sums are up to 1.7e-5 off (an output of -0.5582618 in 64 bits
among 131072 columns: the oracle -0.5582452, the kernel -0.5582619).
"""
import pytest
import torch

from dslperfgap_amd.viperbench.log_softmax.hip_impl import log_softmax
from dslperfgap_amd.viperbench.logsumexp.hip_impl import logsumexp
from dslperfgap_amd.viperbench.softmax.hip_impl import softmax

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# fp32: 32-bit sums of up to 140000 exps with 1-ulp exp and log; 16-bit: half an
# ulp of the output, at values up to about 30
TOL = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}


def _rows(rows, cols, dtype):
    x = (3 * torch.randn(rows, cols, generator=torch.Generator().manual_seed(431))).to(dtype)
    big = torch.finfo(dtype).max
    x[0, cols // 2] = 25.0
    if rows > 8:
        x[1, -1] = float("nan")
        x[2, 0] = float("inf")
        x[3, :] = float("-inf")
        x[4, : cols // 2] = float("-inf")
        x[5, :] = -big
        x[6, cols // 3] = big
        x[7, :] = x[7, :] + 30000.0
    return x


def _close(got, want, dtype, what):
    assert got.dtype == dtype and got.shape == want.shape, what
    tol = TOL[dtype]
    w = want.to(dtype).double()
    assert torch.allclose(got.cpu().double(), w, atol=tol, rtol=tol, equal_nan=True), what


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(33, c) for c in (1, 7, 16, 17, 20, 132, 255, 256, 260, 1001,
                                                         4096, 4098, 16389, 50257)]
                         + [(200, 65540), (140, 131072), (4, 50257), (3, 131075)]
                         # split, on both sides of 7 * 2^18 and 2^23 elements
                         + [(14, 131072), (13, 131072), (64, 131072), (65, 131072), (40, 120987)]
                         # 2, 4 vectors per lane
                         + [(33, c) for c in (516, 569, 1024, 1028, 2560, 5824)]
                         # large launches of short rows: 8 elements per access at
                         # 24 to 56 and 37 to 67 columns, 4 beside them
                         + [(2**22 // c + 1, c) for c in (23, 24, 32, 36, 37, 40, 41, 44, 47, 48,
                                                          52, 55, 56, 63, 64, 65, 67, 69)])
def test_16_bit_rows_to_fp32(rows, cols, dtype):
    x = _rows(rows, cols, dtype)
    _close(log_softmax(x.to(DEV), -1, torch.float32), torch.log_softmax(x.double(), -1),
           torch.float32, f"{rows}x{cols}")


@pytest.mark.parametrize("rows,cols", [(40, 40000), (20, 50257), (12, 65536)])
def test_wide_fp32_softmax_rows(rows, cols):
    x = _rows(rows, cols, torch.float32)
    x[7, :] = x[7, :] + 1e9  # beyond the one-FMA form
    _close(softmax(x.to(DEV)), torch.softmax(x.double(), -1), torch.float32, f"{rows}x{cols}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(300, 65544), (520, 70001)])
def test_streaming_rows(rows, cols, dtype):
    x = _rows(rows, cols, dtype)
    xd, x64 = x.to(DEV), x.double()
    _close(softmax(xd), torch.softmax(x64, -1), dtype, "softmax")
    _close(log_softmax(xd), torch.log_softmax(x64, -1), dtype, "log_softmax")
    _close(logsumexp(xd), torch.logsumexp(x64, -1), dtype, "logsumexp")
