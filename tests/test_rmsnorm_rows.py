"""RMSNorm of many rows, where a thread takes two chunks instead of one: against the oracle, and the rows that
both blocks can take alike."""

import numpy as np
import pytest
import torch

import w4a16
from oracle import oracle
from test_gpu_parity import from_dev, norm_inputs, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(385, 4096), (385, 4104), (600, 5120), (513, 8192), (385, 8200)])
def test_many_rows(cuda, rows, cols):
    """The FP64 sums differ in their order alone, 2^-53 of the scale, which the FP32 rounding of it swallows; the
    oracle's bar is 1 BF16 ULP, as for few rows."""
    print(f"rmsnorm rows={rows} cols={cols}", flush=True)
    x, w = norm_inputs(rows, cols, 1, seed=cols)
    xd, wd = to_dev(x, cuda), to_dev(w, cuda)
    out = w4a16.rmsnorm(xd, wd, 1, 1e-6)
    assert torch.equal(out[:200], w4a16.rmsnorm(xd[:200].contiguous(), wd, 1, 1e-6))
    got, want = from_dev(out).astype(np.int32), oracle.rmsnorm_bf16(x, w, 1, 1e-6).astype(np.int32)
    assert np.abs(got - want.reshape(got.shape)).max() <= 1  # neighbours of one sign are one apart
