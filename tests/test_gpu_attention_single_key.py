"""GPU: a query that sees a single key gets that key's value, bit for bit, however large its score:
its probability is 2^0, because the exponent is taken of the rounded score less that same rounded
score.  (The unrounded score less the rounded one leaves half an ulp of the score in the exponent:
at the scores of this test, about 6e4 in base 2, a probability off by up to 1.4e-3.)  Rows of the
64- and of the 128-query kernels, padded and packed; the single key is a row's first, or the only
one that its flags leave."""

import ctypes
import math

import pytest
import torch

from testt_amd import _ext, attention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
D, NH, NKV = 128, 12, 2
SCALE = 1.0 / math.sqrt(D)


def _wide(varlen, rows, length):
    out = ctypes.c_int32(-1)
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    _ext.call("soupk_attention_wide", varlen, 0, rows, length, NH, cus, ctypes.addressof(out))
    return out.value == 1


def _rows(g, *shape):
    """q and k near 60 in size and equal in sign: every score is large and positive."""
    return (60 + torch.randn(*shape, D, generator=g)).to(torch.float16).to(DEV)


def _heads(v):
    """[rows, NKV, D] values as the output of every query head, [rows, NH * D]."""
    return v.repeat_interleave(NH // NKV, 1).reshape(v.shape[0], NH * D)


@pytest.mark.parametrize("B,T", [(1, 1), (3, 70), (40, 256)])
def test_padded(B, T):
    assert _wide(0, B, T) == (T == 256)
    g = torch.Generator().manual_seed(B)
    q, k = _rows(g, B, NH, T), _rows(g, B, NKV, T)
    v = torch.randn(B, NKV, T, D, generator=g).to(torch.float16).to(DEV)
    out, _ = attention.attention_fwd(q, k, v, None, SCALE)
    assert torch.equal(out.view(B, T, -1)[:, 0], _heads(v[:, :, 0]))
    at = T // 2                                # the one visible key of every row
    flags = torch.zeros(B, T, dtype=torch.uint8, device=DEV)
    flags[:, at] = 1
    out, _ = attention.attention_fwd(q, k, v, flags, SCALE)
    out = out.view(B, T, -1)
    assert torch.equal(out[:, at:], _heads(v[:, :, at])[:, None].expand(B, T - at, -1))
    assert not bool(out[:, :at].any())


@pytest.mark.parametrize("lengths", [[1], [1, 70, 1, 3], [1, 300, 129] * 12])
def test_packed(lengths):
    M, B = sum(lengths), len(lengths)
    assert _wide(1, B, M) == (B == 36)
    g = torch.Generator().manual_seed(M)
    v = torch.randn(M, NKV * D, generator=g).to(torch.float16).to(DEV)
    qk = _rows(g, M, NH + NKV).view(M, -1)
    ends = torch.tensor([0] + lengths).cumsum(0)
    out, _ = attention.attention_varlen_fwd(torch.cat([qk, v], 1),
                                            ends.to(torch.int32).to(DEV), NH, NKV, SCALE)
    first = ends[:-1].to(DEV)
    assert torch.equal(out[first], _heads(v[first].view(B, NKV, D)))
