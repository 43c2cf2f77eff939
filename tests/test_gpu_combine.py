"""Combine on the GPU (mep_combine) vs the oracle, with absent cells and masked tokens.

Cells of entries that were not dispatched hold whatever the buffer held: here
NaN, which must never reach an output.  k = 8 runs the kernel that loads every
cell speculatively and skips absent ones with a select; k = 4 the general one,
which loads present cells only.
Bar: max |out - ref| <= tol * max |ref| (1e-5 fp32, 2e-2 bf16); invalid tokens
give exact zeros.
"""
import numpy as np
import pytest
import torch

from helpers import TOL_BF16, TOL_F32, banner, rel_err, to_np
from miniep_amd import ops
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("k", [8, 4])
@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 1024), (torch.float32, 1024), (torch.bfloat16, 1544),
                                     (torch.bfloat16, 4096), (torch.float32, 2048), (torch.float32, 1028)])
def test_combine_absent_cells_and_masks(k, dtype, H):
    """Rows of any length the 16-byte chunks allow (H % 8 bf16, H % 4 fp32),
    including rows longer than one workgroup and rows that straddle two."""
    banner(f"combine k={k} {dtype} H={H}")
    n = 301
    g = torch.Generator().manual_seed(11 + k)
    y = torch.randn(n * k, H, generator=g).to(dtype)
    gate = torch.softmax(torch.randn(n, k, generator=g), -1).to(dtype)
    present = torch.rand(n * k, generator=g) < 0.8
    row = torch.where(present, torch.arange(n * k), torch.full((n * k,), -1)).to(torch.int32)
    valid = torch.rand(n, generator=g) < 0.9
    y_dev = y.clone()
    y_dev[~present] = float("nan")                      # never written by any expert
    out = to_np(ops.combine(y_dev.to(DEV), gate.to(DEV), row.to(DEV), valid.to(DEV))).astype(np.float32)
    keep = present.numpy() & np.repeat(valid.numpy(), k)
    ref = O.combine(y.float().numpy(), gate.float().numpy(), keep, n, k)
    assert np.isfinite(out).all()
    assert (out[~valid.numpy()] == 0).all()
    assert rel_err(out, ref) <= (TOL_BF16 if dtype == torch.bfloat16 else TOL_F32)
    # run to run: bitwise identical
    out2 = to_np(ops.combine(y_dev.to(DEV), gate.to(DEV), row.to(DEV), valid.to(DEV))).astype(np.float32)
    assert np.array_equal(out, out2)


@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 1024), (torch.bfloat16, 1160), (torch.float32, 2052)])
def test_combine_rows_indexed(dtype, H):
    """mep_combine_rows: cell (t, s) is row row_of_entry[t*k+s] of y (the
    expert-parallel return path), summed in slot order."""
    banner(f"combine_rows {dtype} H={H}")
    n, k = 257, 8
    g = torch.Generator().manual_seed(5)
    present = torch.rand(n * k, generator=g) < 0.75
    m = int(present.sum())
    rows = torch.full((n * k,), -1, dtype=torch.int32)
    rows[present] = torch.randperm(m, generator=g).to(torch.int32)
    y = torch.randn(m, H, generator=g).to(dtype)
    gate = torch.softmax(torch.randn(n, k, generator=g), -1).to(dtype)
    out = to_np(ops.combine_rows(y.to(DEV), gate.to(DEV), rows.to(DEV))).astype(np.float32)
    cells = np.zeros((n * k, H), np.float32)
    cells[present.numpy()] = y.float().numpy()[rows.numpy()[present.numpy()]]
    ref = O.combine(cells, gate.float().numpy(), present.numpy(), n, k)
    assert rel_err(out, ref) <= (TOL_BF16 if dtype == torch.bfloat16 else TOL_F32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,H", [(1, 8), (7, 520), (129, 1024)])
def test_combine_rows_k8_masks_and_poison(dtype, n, H):
    """k = 8 through indices: masked tokens are 0 whatever their cells hold, a
    poisoned cell (-2) makes its token NaN, a token without cells is 0, and
    rows that nothing names (NaN here) do not reach an output.  Bar as above."""
    banner(f"combine_rows k=8 {dtype} n={n} H={H}")
    k = 8
    g = torch.Generator().manual_seed(n)
    y = torch.randn(n * k + 3, H, generator=g).to(dtype)
    y[n * k:] = float("nan")
    gate = torch.softmax(torch.randn(n, k, generator=g), -1).to(dtype)
    rows = torch.randperm(n * k, generator=g).to(torch.int32).reshape(n, k)
    rows[torch.rand(n, k, generator=g) < 0.3] = -1
    valid = torch.rand(n, generator=g) < 0.7
    rows[n // 2] = -1
    poisoned = torch.zeros(n, dtype=torch.bool)
    if n > 4:
        poisoned[1] = poisoned[4] = True
        valid[1], valid[4] = True, False
        rows[1, 3] = rows[4, 7] = -2
    out = ops.combine_rows(y.to(DEV), gate.to(DEV), rows.reshape(-1).to(DEV), valid.to(DEV)).float().cpu()
    nan = poisoned & valid
    assert bool(torch.isnan(out[nan]).all()) and bool(torch.isfinite(out[~nan]).all())
    present = (rows >= 0) & valid[:, None]
    cells = torch.where(present[..., None], y[rows.clamp(min=0).long()].float(), torch.zeros(()))
    ref = O.combine(cells.reshape(n * k, H).numpy(), gate.float().numpy(), present.reshape(-1).numpy(), n, k)
    assert not out[~valid].any() and not out[n // 2].nan_to_num().any()
    keep = ~nan.numpy()
    tol = TOL_BF16 if dtype == torch.bfloat16 else TOL_F32
    assert np.abs(out.numpy()[keep] - ref[keep]).max() <= tol * max(np.abs(ref[keep]).max(), 1e-30)
