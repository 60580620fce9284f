"""GPU: FusedHeadLoss without a host synchronisation (testt_amd/csrc/head_plan.hip) against the form
that reads its row plan back (head._RowPlan), which an fp32 denominator tensor still takes: the
same logits, statistics and scale, so entropy, token loss and hits are the same bits; the packed
gradient rows differ only in how the split products are summed (one fp16 ulp plus the summation
bound, here 2e-3 of the gradient's largest value), the loss by the order of an fp32 sum."""

import pytest
import torch

from testt_amd import head

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _inputs(rows, hidden, vocab, ignored, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(rows, hidden, generator=g).to(torch.float16).to(DEV)
    w = (torch.randn(vocab, hidden, generator=g) * 0.1).to(torch.float16).to(DEV)
    t = torch.randint(0, vocab, (rows,), generator=g)
    t[torch.rand(rows, generator=g) < ignored] = head.IGNORE_INDEX
    return h, w, t.to(DEV)


def _run(h, w, t, den):
    x = h.clone().requires_grad_(True)
    loss, ent, tok, hit = head.fused_head_loss(x, w, t, den)
    (loss * 1024.0).backward()
    return loss.detach(), ent, tok, hit, x.grad


# one row, one chunk, the chunk's edges, several chunks; nothing and everything ignored
@pytest.mark.parametrize("rows,chunk,ignored", [(1, 2048, 0.0), (64, 2048, 0.3), (300, 100, 0.5),
                                                (257, 256, 1.0), (1100, 1024, 0.0)])
@pytest.mark.parametrize("den", ["int", "int32", "python"])
def test_planned_matches_read_back(rows, chunk, ignored, den, monkeypatch):
    print(f"planned head rows={rows} chunk={chunk} ignored={ignored} den={den}", flush=True)
    monkeypatch.setattr(head, "CHUNK_ROWS", chunk)
    h, w, t = _inputs(rows, 64, 5000, ignored, rows)
    n = max(int((t != head.IGNORE_INDEX).sum()), 1)
    d = {"int": torch.tensor(n, device=DEV), "python": n,
         "int32": torch.tensor(n, dtype=torch.int32, device=DEV)}[den]
    assert head._device_plan(h, w, d) is not None
    f = torch.tensor(float(n), device=DEV)
    assert head._device_plan(h, w, f) is None
    got, want = _run(h, w, t, d), _run(h, w, t, f)
    assert abs(float(got[0]) - float(want[0])) <= 1e-6 * abs(float(want[0]))
    for a, b in zip(got[1:4], want[1:4]):
        assert a.dtype == b.dtype and torch.equal(a, b)
    assert got[4].dtype == want[4].dtype
    peak = float(want[4].abs().max())
    assert float((got[4].float() - want[4].float()).abs().max()) <= 2e-3 * peak
    assert not bool(got[4][t == head.IGNORE_INDEX].any())


@pytest.mark.parametrize("d", [-3, 0, 1, 2, 3, 5, 6, 11, 12, 22, 23, 1023, 1448, 1449, 1843, 2047,
                               2048, 10 ** 12])
def test_device_unit_and_scale(d):
    """soupk_head_plan's unit and scale from an integer denominator are the host's."""
    from testt_amd import _ext

    t = torch.zeros(1, dtype=torch.int64, device=DEV)
    slot, counts = (torch.empty(1, dtype=torch.int32, device=DEV) for _ in range(2))
    scal = torch.empty(2, dtype=torch.float32, device=DEV)
    den = torch.tensor(d, device=DEV)
    _ext.call("soupk_head_plan", t.data_ptr(), 1, 1, slot.data_ptr(), counts.data_ptr(),
              den.data_ptr(), 0.0, 0.0, scal.data_ptr(), _ext.stream_of(t))
    unit = head._grad_unit(d)
    want = torch.tensor([unit / max(float(d), 1e-6), unit], dtype=torch.float32)
    assert torch.equal(scal.cpu(), want)


def test_no_synchronisation_under_capture():
    """The whole head, forward and backward, records into a HIP graph; replays on new inputs equal
    the eager result."""
    h, w, t = _inputs(200, 64, 4096, 0.3, 7)
    x = h.clone().requires_grad_(True)
    den = (t != head.IGNORE_INDEX).sum()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            torch.autograd.grad(head.fused_head_loss(x, w, t, den)[0], x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = head.fused_head_loss(x, w, t, den)
        (dx,) = torch.autograd.grad(outs[0], x)
    for seed in range(4):
        h2, _, t2 = _inputs(200, 64, 4096, 0.1 + 0.2 * seed, 20 + seed)
        with torch.no_grad():
            x.copy_(h2)
            t.copy_(t2)
            den.copy_((t2 != head.IGNORE_INDEX).sum())
        graph.replay()
        torch.cuda.synchronize()
        y = h2.clone().requires_grad_(True)
        want = head.fused_head_loss(y, w, t2, den.clone())
        (dy,) = torch.autograd.grad(want[0], y)
        for a, b in zip(outs, want):
            assert torch.equal(a, b)
        assert torch.equal(dx, dy)


def test_planned_gradient_batched_and_differentiated():
    """Several loss gradients at once (is_grads_batched) and a gradient of the gradient: each equal
    to what the general form gives, as the same products of one fp16 row and one fp32 factor."""
    h, w, t = _inputs(40, 64, 5000, 0.4, 11)
    x = h.clone().requires_grad_(True)
    loss = head.fused_head_loss(x, w, t, torch.tensor(24, device=DEV))[0]
    one = torch.autograd.grad(loss, x, torch.tensor(2048.0, device=DEV), retain_graph=True)[0]
    many = torch.autograd.grad(loss, x, torch.tensor([1024.0, 2048.0], device=DEV),
                               is_grads_batched=True, retain_graph=True)[0]
    assert many.shape == (2, 40, 64) and torch.equal(many[1], one)
    s = torch.tensor(2048.0, device=DEV, requires_grad=True)
    dh = torch.autograd.grad(loss, x, s, create_graph=True)[0]
    assert torch.equal(dh, one)
    # d(sum dh)/ds = sum dh / s, fp16 rounding of each entry of dh apart
    ds = torch.autograd.grad(dh.float().sum(), s)[0]
    want = float(one.double().sum()) / 2048.0
    bound = 2.0 ** -10 * float(one.double().abs().sum()) / 2048.0
    assert abs(float(ds) - want) <= bound


def test_refusals_stay():
    """Targets of another shape, an autocast to another type and a denominator that is no number
    are refused as by the general form."""
    h, w, t = _inputs(8, 64, 5000, 0.0, 12)
    with pytest.raises(ValueError):
        head.fused_head_loss(h, w, t.view(2, 4), 8)
    with torch.autocast("cuda", dtype=torch.bfloat16), pytest.raises(TypeError):
        head.fused_head_loss(h, w, t, 8)
    with pytest.raises(ValueError):
        head.fused_head_loss(h, w, t, float("nan"))


def test_wrapped_tensors_raise():
    """A batched tensor has no storage to hand to a kernel: an error, as an exception."""
    from testt_amd import mlp

    gu = torch.zeros(3, 4, 64, dtype=torch.float16, device=DEV)
    with pytest.raises(RuntimeError):
        torch.func.vmap(mlp.gated_silu)(gu)
