"""CPU regression test: the index arithmetic of the fused LoRA + RoPE forward
(lora_fwd_kernel<true>, soupk_lora_rope_fwd in testt_amd/csrc/lora.hip) stays in bounds and
writes every output element exactly once.

The kernel takes 16 rows per workgroup (grid.x) and splits the heads (q, then v, then k) over
grid.y parts; wavefronts 2i and 2i + 1 of a part take its heads i, i + 2, ..., wavefront w the dims
32 (w%2) .. +31 and their rotation partners (+ 64), a lane 8 consecutive ones of each.  This test
replays, with numpy, the grid and the per-lane addresses of every load (qkv, B16 rows, cos / sin
entries) and store (the output rows) for the GPU tests' shapes, and checks that the B16 rows are
those of the columns a lane stores, the indices lie inside their buffers, and the stores cover the
[M, W] output exactly once.  The row backward's dy columns (32 per pair of tiles) are replayed in
the same way.  No GPU is needed."""

import numpy as np
import pytest

KR, KBATCH, KROWS = 16, 4, 16


def column_parts(M, n_tiles, target=256):
    """column_parts() of lora.hip (soupk_lora_rope_fwd then caps it at the head count)."""
    row_blocks = -(-M // KROWS)
    parts = target // row_blocks
    parts = min(parts, max(1, n_tiles // (4 * KBATCH)))
    return max(parts, 1)


def tile_part(n, part, parts):
    return (n * part) // parts


@pytest.mark.parametrize("M,NH,NKV,T", [(2048, 12, 2, 512), (888, 12, 2, 512), (1, 12, 2, 1),
                                        (17, 4, 2, 40), (130, 4, 4, 130), (53, 2, 1, 64)])
def test_lora_rope_fwd_indices(M, NH, NKV, T):
    D = 128
    NQ, NV, NK = NH * D, NKV * D, NKV * D
    W = NQ + NK + NV
    nlora = NQ // 16 + NV // 16
    nq_heads, nlora_heads = NQ // 128, nlora // 8
    heads = (nlora + NK // 16) // 8
    parts = min(column_parts(M, nlora), W // 128)
    grid_x = -(-M // KROWS)
    written = np.zeros((M, W), dtype=np.int32)
    lane = np.arange(64)
    ql, gr = lane & 15, lane >> 4
    slots = 4 * T

    def head_col(h):
        return 128 * h if h < nq_heads else (
            NQ + NK + 128 * (h - nq_heads) if h < nlora_heads else NQ + 128 * (h - nlora_heads))

    for by in range(parts):
        n_heads = tile_part(heads, by + 1, parts)
        assert n_heads <= heads
        for w in range(4):
            d0 = 32 * (w & 1) + 8 * gr
            # cos / sin entries of the lane's dims (t < T): d0 .. d0 + 7 and + 64
            assert (T - 1) * 128 + d0.max() + 64 + 7 < T * 128
            for h in range(tile_part(heads, by, parts) + (w >> 1), n_heads, 2):
                hb = min(h, nlora_heads - 1)
                col = head_col(h) + d0
                for half in (0, 1):
                    for u in (0, 1):
                        c = 64 * half + 32 * (w & 1) + 8 * (ql >> 2) + 4 * u + (ql & 3)
                        b_row = 128 * hb + c
                        assert 0 <= b_row.min() and b_row.max() * KR + 4 * 3 + 3 < (NQ + NV) * KR
                        # result i of the lane is operand row 4 gr + i: its column of the head
                        for i in range(4):
                            assert (c[4 * gr + i] == 64 * half + d0 + 4 * u + i).all()
                for bx in range(grid_x):
                    m = bx * KROWS + ql
                    ok = m < M
                    for i in range(8):
                        np.add.at(written, (m[ok], col[ok] + i), 1)
                        np.add.at(written, (m[ok], col[ok] + 64 + i), 1)
    assert (written == 1).all(), (int((written == 0).sum()), int((written > 1).sum()))
    # every workgroup's rows read the positions at clamped rows; 32-bit store offsets
    assert M * W * 2 < 2 ** 32 and slots < 2 ** 31


@pytest.mark.parametrize("M,H", [(2048, 1536), (888, 1536), (17, 512), (1, 128), (4100, 256)])
def test_lora_bwd_rows_columns(M, H):
    parts = column_parts(M, H // 16)
    lane = np.arange(64)
    ql, gr = lane & 15, lane >> 4
    written = np.zeros(H, dtype=np.int32)
    for by in range(parts):
        n32 = tile_part(H // 32, by + 1, parts)
        for w in range(4):
            for tile in range(tile_part(H // 32, by, parts) + w, n32, 4):
                for u in (0, 1):
                    c = 32 * tile + 4 * u + 8 * (ql >> 2) + (ql & 3)   # rows of A16T
                    assert 0 <= c.min() and c.max() < H
                    for i in range(4):
                        out = 32 * tile + 8 * gr + 4 * u + i
                        assert (c[4 * gr + i] == out).all()
                        np.add.at(written, out[ql == 0], 1)
    assert (written == 1).all()
