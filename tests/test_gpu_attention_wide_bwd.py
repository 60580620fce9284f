"""GPU: the 128-query attention kernels in the forms that training of long rows takes -- the padded
backward under key flags, and the varlen backward with RoPE's backward in it -- against launches of
one row each, which the 64-query kernels take (a query's and a key's arithmetic is the same in both:
equal bits), and against float32.  Float32 tolerances are those of tests/test_gpu_attention.py: P
and dS are rounded to fp16 for their products, outputs 2e-3 absolute, gradients 2e-3 of the largest
entry.  Row lengths: whole 128-query blocks, an odd 64-key block, one query over, shorter than a
wavefront's queries, one token, none."""

import ctypes
import math

import pytest
import torch

from tests.test_gpu_attention import reference
from testt_amd import _ext, attention, workloads

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
D, NH, NKV = 128, 12, 2
SCALE = 1.0 / math.sqrt(D)


def wide(varlen, backward, rows, length):
    out = ctypes.c_int32(-1)
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    _ext.call("soupk_attention_wide", varlen, backward, rows, length, NH, cus,
              ctypes.addressof(out))
    return out.value == 1


def bits(t):
    return t.contiguous().view(torch.int16)


def close(got, ref, name):
    top = max(float(ref.abs().max()), 1.0)
    assert torch.isfinite(got).all(), name
    assert float((got.cpu().float() - ref).abs().max()) <= 2e-3 * top, name


PADDED = [385, 384, 320, 0, 129, 64, 1, 31, 385]       # (the last row: holes in its flags)


@pytest.mark.parametrize("flags", [True, False])
def test_padded_wide_backward(flags):
    B, T = len(PADDED), 385
    assert wide(0, 1, B, T) and wide(0, 0, B, T) and not wide(0, 1, 1, T) and not wide(0, 0, 1, T)
    print(f"padded wide backward B={B} T={T} flags={flags}", flush=True)
    g = torch.Generator().manual_seed(17 + flags)
    q = torch.randn(B, NH, T, D, generator=g).to(torch.float16)
    k = torch.randn(B, NKV, T, D, generator=g).to(torch.float16)
    v = torch.randn(B, NKV, T, D, generator=g).to(torch.float16)
    dout = torch.randn(B * T, NH * D, generator=g).to(torch.float16)
    valid = None
    if flags:
        valid = (torch.arange(T)[None] < torch.tensor(PADDED)[:, None]).to(torch.uint8)
        valid[-1, 1::3] = 0
    qd, kd, vd, dd = (t.to(DEV) for t in (q, k, v, dout))
    fd = None if valid is None else valid.to(DEV)
    out, lse = attention.attention_fwd(qd, kd, vd, fd, SCALE)
    grads = attention.attention_bwd(qd, kd, vd, fd, out, lse, dd, SCALE)
    for b in range(B):
        one = [t[b:b + 1].contiguous() for t in (qd, kd, vd)]
        f1 = None if fd is None else fd[b:b + 1].contiguous()
        o1, l1 = attention.attention_fwd(*one, f1, SCALE)
        d1 = attention.attention_bwd(*one, f1, o1, l1, dd[b * T:(b + 1) * T].contiguous(), SCALE)
        assert torch.equal(bits(o1), bits(out[b * T:(b + 1) * T])), b
        for name, x, y in zip(("dq", "dk", "dv"), d1, grads):
            assert torch.equal(bits(x[0]), bits(y[b])), (name, b)
    rows = [0, 2, 3, 4, 8]
    qf, kf, vf = (t[rows].float().requires_grad_() for t in (q, k, v))
    ref, r_lse = reference(qf, kf, vf, None if valid is None else valid[rows], SCALE)
    ref.backward(dout.view(B, T, -1)[rows].float())
    assert float((out.view(B, T, -1)[rows].cpu().float() - ref.detach()).abs().max()) < 2e-3
    for name, got, r in zip(("dq", "dk", "dv"), grads, (qf, kf, vf)):
        close(got[rows], r.grad, name)
    if flags:                                  # (row 3 has no visible key)
        assert not any(bool(t[3].any()) for t in grads)


VARLEN = [700, 0, 130, 1, 515, 64, 129, 31] * 3


def _rows(lengths, seed):
    M = sum(lengths)
    g = torch.Generator().manual_seed(seed)
    rows = torch.randn(M, (NH + 2 * NKV) * D, generator=g).to(torch.float16)
    dout = torch.randn(M, NH * D, generator=g).to(torch.float16)
    cu = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32)
    return rows, dout, cu


def _reference_row(rows, dout, cos=None, sin=None):
    """float32 out and dq|dk|dv of one row's tokens, rotated back with the tables where given."""
    n = rows.shape[0]
    q, k, v = (t.float().view(1, n, -1, D).transpose(1, 2).contiguous().requires_grad_()
               for t in rows.split((NH * D, NKV * D, NKV * D), 1))
    out, _ = reference(q, k, v, None, SCALE)
    out.backward(dout.float()[None])
    grads = [t.grad[0].transpose(0, 1) for t in (q, k, v)]
    if cos is not None:
        c, s = cos[:n, None].float(), sin[:n, None].float()
        for i in (0, 1):
            g1, g2 = grads[i][..., :64], grads[i][..., 64:]
            grads[i] = torch.cat([g1 * c[..., :64] + g2 * s[..., 64:],
                                  g2 * c[..., 64:] - g1 * s[..., :64]], -1)
    return out.detach()[0], torch.cat([t.reshape(n, -1) for t in grads], 1)


@pytest.mark.parametrize("with_rope", [True, False])
def test_varlen_wide_backward(with_rope):
    lengths, T = VARLEN, 700
    B, M = len(lengths), sum(lengths)
    assert wide(1, 0, B, M) and wide(1, 1, B, M)
    print(f"varlen wide backward B={B} M={M} rope={with_rope}", flush=True)
    rows, dout, cu = (t.to(DEV) for t in _rows(lengths, 5 + with_rope))
    cos, sin = workloads.rope_tables(T, D, workloads.ROPE_THETA, device=DEV)
    pos = workloads.ragged_positions(lengths, T).to(DEV)
    lost = 40                                  # a token without a place gets no gradient for q, k
    pos[lost] = -1
    out, lse = attention.attention_varlen_fwd(rows, cu, NH, NKV, SCALE)
    dqkv = attention.attention_varlen_bwd(rows, cu, out, lse, dout, SCALE, NH, NKV,
                                          rope=(cos, sin, pos, B, T) if with_rope else None)
    at = 0
    for b, n in enumerate(lengths):
        if n == 0:
            continue
        part = slice(at, at + n)
        one = torch.tensor([0, n], dtype=torch.int32, device=DEV)
        assert not wide(1, 0, 1, n) and not wide(1, 1, 1, n)
        o1, l1 = attention.attention_varlen_fwd(rows[part].contiguous(), one, NH, NKV, SCALE)
        assert torch.equal(bits(o1), bits(out[part])) and torch.equal(l1, lse[:, part]), b
        d1 = attention.attention_varlen_bwd(
            rows[part].contiguous(), one, o1, l1, dout[part].contiguous(), SCALE, NH, NKV,
            rope=(cos, sin, pos[part].contiguous(), B, T) if with_rope else None)
        assert torch.equal(bits(d1), bits(dqkv[part])), b
        if b < 8:
            tables = (cos.cpu(), sin.cpu()) if with_rope else ()
            r_out, r_grad = _reference_row(rows[part].cpu(), dout[part].cpu(), *tables)
            assert float((out[part].cpu().float() - r_out).abs().max()) < 2e-3, b
            if with_rope and at <= lost < at + n:
                r_grad[lost - at, :(NH + NKV) * D] = 0
                r_grad[lost - at, (NH + NKV) * D:] = dqkv[lost, (NH + NKV) * D:].cpu().float()
            close(dqkv[part], r_grad, b)
        at += n
    if with_rope:
        assert not bool(dqkv[lost, :(NH + NKV) * D].any())
