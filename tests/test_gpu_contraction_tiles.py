"""The batched contraction picks its tile (64 x 256, 32 x 256 or 32 x 128 rows by
photon bins) by the number of rows.  Every tile adds an element's products in the
same order, so a batch of few rows (the small tiles) equals the same rows inside
a batch of many (the large one) bit for bit; generated rows sum their FP64 norm
in eight parts instead of four, which may turn one float rounding (6e-8) of the
norm's reciprocal and of the product: 2e-7."""
import numpy as np
import pytest
import torch

from ragnar_amd import _capi as C
from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu

PRECISIONS = [C.RGN_PREC_F16X3, C.RGN_PREC_F16X1, C.RGN_PREC_BF16X6]
MANY = 40000  # over the small tiles' range from 129 bins


@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("ng,nb", [(63, 129), (64, 256), (70, 200), (300, 385), (128, 512)])
def test_tiles_agree(precision, ng, nb):
    grid = torch.logspace(0, 4, ng, device="cuda", dtype=torch.float64).float()
    plan = T.SyncPlan(T.default_table(), np.logspace(-2, 7, nb).astype(np.float32))
    gen = torch.Generator(device="cuda").manual_seed(ng + nb)
    p = -3.0 + 2.0 * torch.rand(MANY, generator=gen, device="cuda")
    xc = 10.0 ** (1.0 + 3.0 * torch.rand(MANY, generator=gen, device="cuda"))
    f = (grid[None] ** p[:, None] * torch.exp(-grid[None] / xc[:, None])).contiguous()
    rows = T.sync_fromdist_batched(plan, grid, f, True, precision)
    made = T.sync_fromdist_batched_plaw(plan, grid, p, xc, True, precision)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n128, n256 = -(-nb // 128), -(-nb // 256)
    edges = [32 * (3 * cus // 2 // n128), 32 * (5 * cus // n128), 32 * (3 * cus // n256), 32 * (cus // n128)]
    for nd in sorted({1, 31, 32, 33, 65, *edges, *(e + 1 for e in edges)}):
        if nd >= MANY:
            continue
        a = T.sync_fromdist_batched(plan, grid, f[:nd], True, precision)
        assert torch.equal(a, rows[:nd]), nd
        b, c = T.sync_fromdist_batched_plaw(plan, grid, p[:nd].contiguous(), xc[:nd].contiguous(), True, precision), made[:nd]
        assert torch.all((b - c).abs() <= 2e-7 * c.abs()), nd
