"""The batched contraction at the lines of its tile choice (small tiles: 3/2, 3, 4
and 5 a CU; 32 x 256: 5/2 and 3; 64 x 256: 2 and more), for rows read by scalars,
by 16-byte loads and in whole blocks of g, and one to four columns of 128.  Every
tile adds an element's products in the same order, so the rows of a batch equal
the same rows of a larger one bit for bit."""
import numpy as np
import pytest
import torch

from ragnar_amd import _capi as C
from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [C.RGN_PREC_F16X3, C.RGN_PREC_F16X1, C.RGN_PREC_BF16X6])
@pytest.mark.parametrize("ng,nb", [(63, 100), (65, 256), (66, 300), (68, 384), (128, 300), (67, 512)])
def test_lines_agree(precision, ng, nb):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    cols, wide = -(-nb // 128), -(-nb // 256)
    lines = [32 * k * cus // (2 * cols) for k in (3, 6, 8, 10)] + [32 * k * cus // (2 * wide) for k in (5, 6)]
    lines += [64 * 2 * cus // wide]
    many = max(lines) + 65
    grid = torch.logspace(0, 4, ng, device="cuda", dtype=torch.float64).float()
    plan = T.SyncPlan(T.default_table(), np.logspace(-2, 7, nb).astype(np.float32))
    gen = torch.Generator(device="cuda").manual_seed(ng + nb)
    p = -3.0 + 2.0 * torch.rand(many, generator=gen, device="cuda")
    f = (grid[None] ** p[:, None]).contiguous()
    rows = T.sync_fromdist_batched(plan, grid, f, True, precision)
    for nd in sorted({n + d for n in lines for d in (0, 1, 33)}):
        assert torch.equal(T.sync_fromdist_batched(plan, grid, f[:nd], True, precision), rows[:nd]), nd
