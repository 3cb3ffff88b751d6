"""A row with an infinity or a NaN spoils its own outputs and no other row's: the multi-row kernels share staged
rows, padded row tiles and accumulators between rows."""

import pytest
import torch

import w4a16
from test_long_sums import random_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (50, 1032, 1536),    # slices of 16 rows
    (33, 2568, 3712),    # the row-tiled GEMM, one row tile
    (50, 12296, 2688),   # two
    (127, 19464, 640),   # four
    (40, 520, 35072),    # second-level sums
    (5, 4136, 8192),     # rows_stream_kernel
    (2, 4136, 17408),    # with second-level sums
    (11, 4136, 5248),    # the LDS-staged tile-pair form
])
def test_rows_stay_apart(cuda, m, n, k):
    print(f"gemm M={m} N={n} K={k}", flush=True)
    gen = torch.Generator().manual_seed(n + k)
    w = random_weight(gen, n, k, False)
    x = torch.randn(m, k, generator=gen).to(torch.bfloat16)
    clean = w4a16.gemm_int4_bf16(x.to(cuda), w)
    bad = x.clone()
    bad[0, k - 1] = float("inf")
    bad[m - 1, 130] = float("nan")
    out = w4a16.gemm_int4_bf16(bad.to(cuda), w)
    assert torch.equal(out[1:m - 1], clean[1:m - 1])
    assert bool(clean.isfinite().all()) and not bool(out[0].isfinite().any() or out[m - 1].isfinite().any())


def test_ffn_rows_stay_apart(cuda):
    """The chunk-major intermediate of 4 to 16 rows, and the pair."""
    hidden, inter = 4224, 8448
    gen = torch.Generator().manual_seed(1)
    gu, dn = random_weight(gen, 2 * inter, hidden, True), random_weight(gen, hidden, inter, False)
    for m in (4, 9, 16, 33):
        print(f"ffn M={m}", flush=True)
        x = (0.01 * torch.randn(m, hidden, generator=gen)).to(torch.bfloat16)
        clean = w4a16.mlp_int4(x.to(cuda), gu, dn)
        x[1, 5] = float("nan")
        out = w4a16.mlp_int4(x.to(cuda), gu, dn)
        rest = [r for r in range(m) if r != 1]
        assert torch.equal(out[rest], clean[rest]) and not bool(out[1].isfinite().any())
