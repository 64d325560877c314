"""Where the automatic choice of the forward method changes over: on both sides
of the measured lines, far enough from them that the slower method costs a tenth
or more there (every index of the population, with and without E)."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,fields,direct,binned", [
    (40, False, 240000, 1100000), (87, False, 240000, 800000), (87, True, 400000, 1000000),
    (128, True, 560000, 1000000), (200, False, 400000, 900000), (256, True, 560000, 1130000),
    (320, False, 560000, 1000000), (512, False, 280000, 500000), (512, True, 280000, 560000)])
def test_forward_line(nb, fields, direct, binned):
    plan = T.SyncPlan(T.default_table(), np.logspace(-2, 7, nb).astype(np.float32))
    for n, expect in ((direct, "forward_kernel"), (binned, "binned_")):
        u = torch.full((3, n), 3.0, device="cuda")
        b = torch.ones(3, n, device="cuda")
        b[2] = 0.0
        names = [name for name, _ in T.spectrum_stages(plan, u, b, None, 0.1 * b if fields else None)]
        assert any(name.startswith(expect) for name in names), (n, names)  # a new scratch buffer is cleared first
