"""GPU: the 128-query attention forward (attn_fwd_wide_kernel, taken where its workgroups fill the
chip) against the 64-query kernel and float32.  A query's arithmetic is the same in both, so the
outputs and log-sum-exps must be the same bits: the wide launch of many rows against one launch per
row, which is small enough for the 64-query kernel.  Row lengths: whole 128-query blocks, one query
over, an odd 64-key block, shorter than one wavefront's 32 queries, empty (varlen)."""

import ctypes
import math

import pytest
import torch

from tests.test_gpu_attention import reference
from testt_amd import _ext, attention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
D, NH, NKV = 128, 12, 2
SCALE = 1.0 / math.sqrt(D)


def _wide(varlen, rows, length):
    """The forward's kernels for `rows` rows of T = length positions, or of length tokens in all."""
    out = ctypes.c_int32(-1)
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    _ext.call("soupk_attention_wide", varlen, 0, rows, length, NH, cus, ctypes.addressof(out))
    return out.value == 1


LENGTHS = [256, 129, 193, 31, 128, 65, 255, 1] * 4


def test_padded_wide_matches_row_launches_and_fp32():
    B, T = len(LENGTHS), 256
    assert _wide(0, B, T) and not _wide(0, 1, T)
    g = torch.Generator().manual_seed(3)
    q = torch.randn(B, NH, T, D, generator=g).to(torch.float16)
    k = torch.randn(B, NKV, T, D, generator=g).to(torch.float16)
    v = torch.randn(B, NKV, T, D, generator=g).to(torch.float16)
    q[0, 0, 5] *= 40.0            # a query whose reference value rises again and again
    valid = (torch.arange(T)[None] < torch.tensor(LENGTHS)[:, None]).to(torch.uint8)
    valid[3] = 0                  # a row without a visible key: output 0, lse +inf
    qd, kd, vd, fd = (t.to(DEV) for t in (q, k, v, valid))
    out, lse = attention.attention_fwd(qd, kd, vd, fd, SCALE)
    for flags in (fd, None):
        o, ls = attention.attention_fwd(qd, kd, vd, flags, SCALE)
        for b in range(B):
            f1 = None if flags is None else flags[b:b + 1].contiguous()
            o1, l1 = attention.attention_fwd(qd[b:b + 1], kd[b:b + 1], vd[b:b + 1], f1, SCALE)
            assert torch.equal(o1.view(torch.int16), o[b * T:(b + 1) * T].view(torch.int16)), b
            assert torch.equal(l1[0], ls[b]), b
    assert not bool(out[3 * T:4 * T].any()) and bool(torch.isinf(lse[3]).all())
    rows = [0, 1, 2, 7]
    r_out, r_lse = reference(q[rows], k[rows], v[rows], valid[rows], SCALE)
    got = out.view(B, T, -1)[rows].cpu().float().reshape(len(rows) * T, -1)
    assert float((got - r_out.reshape(len(rows) * T, -1)).abs().max()) < 2e-3
    rl = r_lse
    assert ((lse[rows].cpu() - rl).abs() <= 1e-4 * rl.abs() + 1e-5).all()


@pytest.mark.parametrize("lengths", [LENGTHS, [700, 0, 130, 1, 515, 64] * 3])
def test_varlen_wide_matches_row_launches(lengths):
    M, B = sum(lengths), len(lengths)
    assert _wide(1, B, M)
    g = torch.Generator().manual_seed(M)
    rows = torch.randn(M, (NH + 2 * NKV) * D, generator=g).to(torch.float16).to(DEV)
    cu = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32,
                      device=DEV)
    out, lse = attention.attention_varlen_fwd(rows, cu, NH, NKV, SCALE)
    dout = (0.1 * torch.randn(M, NH * D, generator=g)).to(torch.float16).to(DEV)
    dqkv = attention.attention_varlen_bwd(rows, cu, out, lse, dout, SCALE, NH, NKV)
    at = 0
    for n in lengths:
        if n:
            one = torch.tensor([0, n], dtype=torch.int32, device=DEV)
            assert not _wide(1, 1, n)
            o1, l1 = attention.attention_varlen_fwd(rows[at:at + n].contiguous(), one, NH, NKV,
                                                    SCALE)
            assert torch.equal(o1.view(torch.int16), out[at:at + n].view(torch.int16)), n
            assert torch.equal(l1, lse[:, at:at + n]), n
            d1 = attention.attention_varlen_bwd(rows[at:at + n].contiguous(), one, o1, l1,
                                                dout[at:at + n], SCALE, NH, NKV)
            assert torch.equal(d1.view(torch.int16), dqkv[at:at + n].view(torch.int16)), n
        at += n
