"""GPU: the norms a call plans from (one workgroup up to 40 KiB of matrix, the columns' sums
and a joint maximum above) are bit for bit the 1-norms clm_matrix_norm1_* reports, for the matrix
and for the powers formed before the plan; a column that is not finite is still seen."""
import numpy as np
import pytest
import torch

import calaman_g_amd as cg
from calaman_g_amd.expm import Context, gemm_cm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.float64, torch.complex64, torch.complex128])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 50, 51, 63, 64, 65, 71, 72, 101, 102, 127, 128, 129, 256,
                               257, 513])
def test_planned_norms_are_the_norms(dev, dt, n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    a = torch.randn((n, n), generator=gen, device=dev, dtype=dt)
    a = a * (20.0 / float(a.abs().sum(0).max()))
    _, plan = cg.expm(a, return_plan=True)
    assert plan["norm1"] == cg.matrix_norm1(a)
    acm, ctx = cg.to_cm(a), Context()
    left = acm
    for k, got in zip(range(2, plan["norm_powers"] + 1), plan["power_norm1"]):
        out = torch.empty_like(acm)
        assert gemm_cm(ctx, n, n, n, 1.0, left, n, acm, n, 0.0, out, n) == 0
        assert got == cg.matrix_norm1(out.t().contiguous())
        left = out


@pytest.mark.parametrize("n,col", [(7, 6), (128, 0), (128, 127), (129, 128), (300, 255)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_bad_column_is_refused_and_info_left_alone(dev, n, col, bad):
    a = torch.zeros((n, n), dtype=torch.float64, device=dev)
    a[n // 2, col] = bad
    work = torch.empty(cg.expm_buffer_size(n), dtype=torch.uint8, device=dev)
    info = torch.full((2,), 9, dtype=torch.int32, device=dev)
    acm = cg.to_cm(a)
    st, _ = cg.expm_cm(n, acm, n, torch.empty_like(acm), n, work, info)
    assert st == cg._lib.INVALID_VALUE
    assert info.tolist() == [9, 9]
