"""The down projection of up to 16 rows with more tile pairs than CUs: rows_stream_kernel (a block a
CU over its tile pairs) where the rows fit LDS, the row-tiled GEMM beyond, at odd tile and group
counts, against the oracle."""

import numpy as np
import pytest
import torch

import w4a16
from conftest import assert_parity
from oracle import oracle
from test_gpu_parity import from_dev, make_ffn, make_weight, norm_inputs, to_dev, ws_act

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (2, 4136, 12544),   # the last block half filled, an odd tile count
    (3, 4136, 10496),
    (5, 4104, 5376),    # 257 tile pairs: most blocks own two
    (8, 16648, 5248),   # five tile pairs a block
    (8, 4136, 10496),   # 82 groups: the rows no longer fit, the GEMM takes it
    (16, 4136, 5248),
    (9, 4136, 8192),    # the longest K the LDS-staged tile-pair form holds at nine rows, and at thirteen
    (13, 4136, 5632),
    (10, 4136, 8192),
    (5, 4104, 7168),    # the few-row form, two blocks of it a CU
    (6, 4136, 5248),
])
def test_linear_parity(cuda, m, n, k):
    print(f"gemm M={m} N={n} K={k}", flush=True)
    p, s = make_weight(n, k, seed=n + k)
    x = oracle.synth_activation(m, k, seed=m + n)
    w = w4a16.TiledWeight.from_artifact(p, s, n, k, device=cuda)
    out = from_dev(w4a16.gemm_int4_bf16(to_dev(x, cuda), w))
    assert_parity(out, oracle.gemm_bf16(x, p, s, n, k), f"gemm M={m} N={n} K={k}")


@pytest.mark.parametrize("m", [4, 7, 9, 16])
def test_down_forms(cuda, m):
    """The chunk-major down projection of more tile pairs than CUs: the stage against the oracle
    on the call's own intermediate, then its FP32 and residual forms, which have to agree with the
    BF16 output bit for bit."""
    hidden, inter = 4224, 8448  # 33 and 66 groups, 264 tile pairs
    print(f"ffn M={m} H={hidden} I={inter}", flush=True)
    gup, gus, dp, ds = make_ffn(hidden, inter, layer=50)
    gu = w4a16.TiledWeight.from_artifact(gup, gus, 2 * inter, hidden, pair=True, device=cuda)
    dn = w4a16.TiledWeight.from_artifact(dp, ds, hidden, inter, device=cuda)
    xd = to_dev(oracle.synth_activation(m, hidden, seed=m), cuda)
    ws = torch.empty((m, inter), dtype=xd.dtype, device=cuda)
    out = w4a16.mlp_int4(xd, gu, dn, act_ws=ws)
    act = ws_act(from_dev(ws), m, inter)
    assert_parity(from_dev(out), oracle.gemm_bf16(act, dp, ds, hidden, inter), f"down M={m}")
    f32 = w4a16.mlp_int4(xd, gu, dn, partial_f32=True)
    assert torch.equal(f32.to(torch.bfloat16).view(torch.int16), out.view(torch.int16))
    res, nw = norm_inputs(m, hidden, 1, seed=10)
    sub = oracle.synth_activation(m, hidden, seed=11)
    summed, _ = oracle.residual_norm_bf16(res, sub, nw, 1, 1e-6)
    resd = to_dev(res, cuda)
    got = w4a16.mlp_int4_residual_norm(resd, to_dev(sub, cuda), to_dev(nw, cuda), 1, 1e-6, gu, dn)
    normed = w4a16.rmsnorm(to_dev(summed, cuda), to_dev(nw, cuda), 1, 1e-6)
    assert torch.equal(got, w4a16.mlp_int4(normed, gu, dn))
    assert np.array_equal(from_dev(resd), oracle.residual_add_bf16(summed, from_dev(got)))
