"""CPU: which of the head's forms and products a call takes, against what was measured on MI355X
(256 CUs): the form without a host synchronisation, or, where hipBLASLt is ahead by more than that
saves, the general form, whose products choose by their labelled rows."""

from types import SimpleNamespace

import pytest
import torch

from testt_amd import blas, head, nf4_gemm

CUS = 256
CPU = torch.device("cpu")


def operand(rows, cols):
    return SimpleNamespace(shape=(rows, cols), is_cuda=True, dtype=torch.float16, device=CPU,
                           is_contiguous=lambda: True, dim=lambda: 2, data_ptr=lambda: 0)


# (vocabulary, width, rows, labelled share, us without the wait, us in the general form)
FORMS = [(128256, 4096, 2048, 1.0, 3984, 3829), (128256, 4096, 4096, 1.0, 7995, 7487),
         (128256, 4096, 2048, 0.75, 3938, 3471), (128256, 3072, 2048, 1.0, 3512, 3130),
         (151936, 6144, 1024, 1.0, 4131, 3676), (32000, 8192, 3000, 1.0, 2884, 2802),
         (32000, 8192, 4096, 1.0, 3796, 3651),
         (32000, 4096, 2048, 1.0, 1051, 1155), (32000, 4096, 4096, 1.0, 2053, 2091),
         (32000, 8192, 1536, 1.0, 1456, 1551), (128256, 4096, 700, 1.0, 1643, 1776),
         (128256, 4096, 1024, 1.0, 2110, 2692), (151936, 1536, 2048, 1.0, 1951, 2240),
         (151936, 1536, 4096, 1.0, 3917, 4367), (151936, 5120, 2048, 1.0, 6318, 6551),
         (151936, 3584, 4096, 1.0, 8843, 9118), (128256, 2048, 4096, 1.0, 4375, 4643)]


# (The labelled share is known on the device alone: with 40% of 1536 rows labelled the form without
# the wait would take 2213 us at 128256 x 4096, the general form that the sizes ask for 2324.)
@pytest.mark.parametrize("vocab,width,rows,share,planned_us,general_us", FORMS)
def test_form(monkeypatch, vocab, width, rows, share, planned_us, general_us):
    monkeypatch.setitem(nf4_gemm._cu_count.cache, CPU, CUS)
    planned = head._device_plan(operand(rows, width), operand(vocab, width), 1.0) is not None
    assert planned == (planned_us < general_us)


# (rows, columns, us on gemm_nn, us on hipBLASLt), contraction 128256
PRODUCTS = [(2048, 3072, 1766, 1445), (1536, 4096, 1532, 1407), (2048, 4096, 2074, 1761),
            (1024, 6144, 1783, 1457), (2048, 6144, 3466, 2822), (768, 8192, 1562, 1441),
            (1024, 8192, 2081, 1762), (2048, 8192, 4029, 3409), (256, 896, 106, 433),
            (2048, 896, 540, 881), (1536, 1536, 635, 898), (2048, 1536, 821, 1083),
            (2048, 2048, 1076, 1433), (2048, 2560, 1356, 1665), (1536, 3072, 1343, 1565),
            (2048, 3584, 1940, 2295), (1024, 4096, 1063, 1493), (1792, 4096, 1915, 2231),
            (1536, 5120, 2022, 2580), (1792, 6144, 2867, 3935), (512, 8192, 1101, 1418)]


@pytest.mark.parametrize("rows,cols,own_us,library_us", PRODUCTS)
def test_product(rows, cols, own_us, library_us):
    assert blas.library_ahead(rows, cols, CUS) == (library_us < own_us)
