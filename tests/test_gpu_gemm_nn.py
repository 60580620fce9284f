"""GPU: soupk_gemm_nn (testt_amd/csrc/gemm_nn.hip), out = fp16_rn(a @ b) with the contraction cut
into parts, against the float64 product of the same fp16 operands.  An fp32 sum rounded once lies
within 1 fp16 ulp plus the summation error, bounded by 64 * 2^-24 * sum|terms| for these depths
(tests/test_gpu_splitk.py's bound)."""

import pytest
import torch

from testt_amd import blas
from tests.test_gpu_splitk import within_bound

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


# every row tile and its edges (16 .. 64, 96 .. 192, 256; one row over), K and N with and without
# remainders of the 64-deep steps and 256-wide tiles, one part and many
@pytest.mark.parametrize("M,K,N", [(1, 8, 8), (16, 128, 256), (17, 200, 264), (48, 4096, 1536),
                                   (64, 1000, 512), (65, 72, 248), (96, 5000, 1536), (128, 64, 256),
                                   (129, 640, 1000), (192, 704, 256), (193, 4104, 1536),
                                   (256, 2048, 256), (300, 64, 264), (420, 3000, 1536),
                                   (1100, 1032, 512)])
def test_gemm_nn(M, K, N):
    print(f"gemm_nn M={M} K={K} N={N}", flush=True)
    g = torch.Generator().manual_seed(M + K + N)
    a = (0.05 * torch.randn(M, K + 8, generator=g)).to(torch.float16).to(DEV)
    b = (0.05 * torch.randn(K, N + 16, generator=g)).to(torch.float16).to(DEV)
    buf = torch.full((M + 2, N + 8), float("nan"), dtype=torch.float16, device=DEV)
    # operands and result inside wider rows: the columns past K and N and the rows around hold
    # values that must not reach the result, and the result's surroundings stay as they are
    av, bv, out = a[:, :K], b[:, :N], buf[1:M + 1, :N]
    a[:, K:] = float("inf")
    b[:, N:] = float("nan")
    assert blas.gemm_nn_fits(av, bv, out)
    blas.gemm_nn(av, bv, out)
    within_bound(out, av, bv)
    keep = torch.isnan(buf)
    keep[1:M + 1, :N] = True
    assert bool(keep.all())
    again = torch.empty((M, N), dtype=torch.float16, device=DEV)
    blas.gemm_nn(av, bv, again)
    assert torch.equal(again.view(torch.int16), out.contiguous().view(torch.int16))


@pytest.mark.parametrize("M,count", [(1, 0), (64, 33), (65, 1), (200, 200), (700, 420), (700, -1),
                                     (300, 5000)])
def test_gemm_nn_device_rows(M, count):
    """The first `count` rows (clamped to [0, M]) computed, the others not written."""
    K, N = 2056, 264
    g = torch.Generator().manual_seed(M + count)
    a = (0.05 * torch.randn(M, K, generator=g)).to(torch.float16).to(DEV)
    b = (0.05 * torch.randn(K, N, generator=g)).to(torch.float16).to(DEV)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device=DEV)
    n = min(max(count, 0), M)
    a[n:] = float("inf")
    blas.gemm_nn(a, b, out, torch.tensor([count], dtype=torch.int32, device=DEV))
    assert bool(torch.isnan(out[n:]).all())
    if n:
        within_bound(out[:n], a[:n], b)


def test_gemm_nn_refuses():
    a = torch.zeros(4, 16, dtype=torch.float16, device=DEV)
    b = torch.zeros(16, 8, dtype=torch.float16, device=DEV)
    o = torch.zeros(4, 8, dtype=torch.float16, device=DEV)
    assert blas.gemm_nn_fits(a, b, o)
    assert not blas.gemm_nn_fits(a[:, :12], b[:12], o)           # K not a multiple of 8
    assert not blas.gemm_nn_fits(a, b.t().contiguous().t(), o)   # b not row-major
    assert not blas.gemm_nn_fits(a[:, 1:9], b[:8], o)            # rows not 16-byte aligned
    assert not blas.gemm_nn_fits(a.float(), b, o)
