"""The row-tiled GEMM (rows_gemm_kernel), where launch_rows and calls of more than 16 rows send work to
it: each of its block shapes at the edges of their row tiles, tile pairs and K steps, against the oracle;
and the slices of 16 rows (gemv_rows16w_kernel) that some of the latter run as. The tolerances are the
suite's (assert_parity): 2 BF16 ULP and rel-L2 1e-3 of the double-accumulated product."""

import numpy as np
import pytest
import torch

import w4a16
from conftest import assert_parity
from oracle import oracle
from test_gpu_parity import from_dev, make_ffn, make_weight, norm_inputs, to_dev

pytestmark = pytest.mark.gpu

# (rows, N, K): one half-filled tile pair of one group; then every block shape (row tiles x tile
# pairs x groups a step) where the launcher's estimate picks it, with odd tile counts, rows that do
# not fill the row tiles and K that does not fill the steps; the slices of 16 rows by one, two and four tile
# pairs a block likewise
SHAPES = [
    (17, 8, 128),        # slices, one tile pair
    (17, 8, 5248),       # 1 x 1 x 16
    (16, 520, 9856),     # 1 x 1 x 16, past the tile-pair form
    (17, 8, 640),        # slices, one tile pair
    (17, 8, 2048),       # 1 x 2 x 8
    (33, 2568, 2688),    # slices, two tile pairs
    (33, 2568, 3712),    # 1 x 3 x 8
    (33, 2568, 1664),    # 1 x 4 x 4
    (33, 5128, 640),     # slices, four tile pairs
    (33, 5640, 640),     # 1 x 6 x 4
    (33, 9736, 1152),    # 1 x 8 x 4
    (33, 5128, 128),     # slices, four tile pairs
    (33, 5640, 128),     # 1 x 10 x 2
    (17, 12296, 640),    # 2 x 4 x 4
    (120, 5128, 1152),   # 2 x 6 x 4
    (50, 12296, 2688),   # 2 x 9 x 4
    (63, 19464, 640),    # 2 x 10 x 2
    (120, 5128, 640),    # 2 x 6 x 2
    (127, 19464, 640),   # 4 x 10 x 2
    (50, 1000, 3840),    # slices, one tile pair, two groups a wave but for two of them
    (40, 1032, 1536),    # slices, one tile pair, twelve of sixteen waves
    (97, 1032, 2176),    # slices, two tile pairs
    (127, 2040, 3200),   # slices, four tile pairs
    (255, 1016, 1280),   # slices, four tile pairs
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_linear_parity(cuda, m, n, k):
    print(f"gemm M={m} N={n} K={k}", flush=True)
    p, s = make_weight(n, k, seed=n + k)
    x = oracle.synth_activation(m, k, seed=m + n)
    w = w4a16.TiledWeight.from_artifact(p, s, n, k, device=cuda)
    out = from_dev(w4a16.gemm_int4_bf16(to_dev(x, cuda), w))
    assert_parity(out, oracle.gemm_bf16(x, p, s, n, k), f"gemm M={m} N={n} K={k}")


@pytest.mark.parametrize("m,hidden,inter", [
    (9, 640, 12296), (16, 1152, 12288), (15, 5248, 4104),  # many tile pairs, or K past the tile-pair form
    (6, 3584, 8196), (8, 2688, 8200),  # few rows whose staged copies leave a CU three blocks
])
def test_gate_up_parity(cuda, m, hidden, inter):
    print(f"gate/up M={m} H={hidden} I={inter}", flush=True)
    p, s = make_weight(2 * inter, hidden, seed=hidden + inter)
    x = oracle.synth_activation(m, hidden, seed=m)
    gu = w4a16.TiledWeight.from_artifact(p, s, 2 * inter, hidden, pair=True, device=cuda)
    act = from_dev(w4a16.gate_up_silu(to_dev(x, cuda), gu))
    want = oracle.silu_mul_packed(oracle.gemm_bf16(x, p, s, 2 * inter, hidden), m, inter)
    assert_parity(act, want, f"gate/up M={m} H={hidden} I={inter}")


@pytest.mark.parametrize("m,hidden,inter", [(17, 128, 128), (65, 640, 9728), (129, 640, 2176), (16, 256, 2176)])
def test_ffn_forms(cuda, m, hidden, inter):
    """The gate/up pair and the down projection, each stage against the oracle on its own inputs
    (end to end a BF16 rounding of the intermediate that falls the other way moves an output by
    up to 2^-8 |act| |w|, which is no error of either stage); then the forms around them, which
    run the same kernels and have to agree bit for bit: the FP32 partial rounds to the BF16
    output, and plan F2 is the MLP of the normed sum, with the residual gaining exactly it (at up to 16 rows
    its down projection is another kernel than the MLP's, so there it is held to the oracle)."""
    print(f"ffn M={m} H={hidden} I={inter}", flush=True)
    gup, gus, dp, ds = make_ffn(hidden, inter, layer=40)
    gu = w4a16.TiledWeight.from_artifact(gup, gus, 2 * inter, hidden, pair=True, device=cuda)
    dn = w4a16.TiledWeight.from_artifact(dp, ds, hidden, inter, device=cuda)
    x = oracle.synth_activation(m, hidden, seed=9)
    xd = to_dev(x, cuda)
    act = w4a16.gate_up_silu(xd, gu)
    mid = oracle.gemm_bf16(x, gup, gus, 2 * inter, hidden)
    assert_parity(from_dev(act), oracle.silu_mul_packed(mid, m, inter), f"gate/up M={m} I={inter}")
    down = w4a16.gemm_int4_bf16(act, dn)
    assert_parity(from_dev(down), oracle.gemm_bf16(from_dev(act), dp, ds, hidden, inter), f"down M={m} K={inter}")
    assert torch.equal(w4a16.mlp_int4(xd, gu, dn), down)
    f32 = w4a16.mlp_int4(xd, gu, dn, partial_f32=True)
    assert torch.equal(f32.to(torch.bfloat16).view(torch.int16), down.view(torch.int16))

    res, nw = norm_inputs(m, hidden, 1, seed=10)
    sub = oracle.synth_activation(m, hidden, seed=11)
    summed, _ = oracle.residual_norm_bf16(res, sub, nw, 1, 1e-6)
    resd = to_dev(res, cuda)
    got = w4a16.mlp_int4_residual_norm(resd, to_dev(sub, cuda), to_dev(nw, cuda), 1, 1e-6, gu, dn)
    normed = w4a16.rmsnorm(to_dev(summed, cuda), to_dev(nw, cuda), 1, 1e-6)
    if m > 16:
        assert torch.equal(got, w4a16.mlp_int4(normed, gu, dn))
    else:
        act = from_dev(w4a16.gate_up_silu(normed, gu))
        assert_parity(from_dev(got), oracle.gemm_bf16(act, dp, ds, hidden, inter), f"F2 down M={m} K={inter}")
    assert np.array_equal(from_dev(resd), oracle.residual_add_bf16(summed, from_dev(got)))


@pytest.mark.parametrize("m,n,k,more", [(16, 28672, 8192, 17), (11, 14344, 8192, 24)])
def test_few_rows_take_the_shape_of_their_width(cuda, m, n, k, more):
    """A long K whose rows rows_stream_kernel cannot hold runs in the shape that N asks for, as more rows do:
    the estimate gives both row counts four groups a step, so the shared rows have the same sums."""
    print(f"gemm M={m} and {more} N={n} K={k}", flush=True)
    gen = torch.Generator().manual_seed(n)
    packed = torch.randint(0, 256, (n, k // 2), generator=gen, dtype=torch.uint8)
    scales = (0.002 + 0.002 * torch.rand(n, k // 128, generator=gen)).to(torch.bfloat16).view(torch.int16)
    w = w4a16.TiledWeight.from_device_artifact(packed.to(cuda), scales.to(cuda), n, k)
    x = torch.randn(more, k, generator=gen).to(torch.bfloat16).to(cuda)
    few = w4a16.gemm_int4_bf16(x[:m], w)
    assert torch.equal(few, w4a16.gemm_int4_bf16(x, w)[:m])
    dense = w.dequantize().double()
    assert_parity(from_dev(few.view(torch.int16)), from_dev((x[:m].double() @ dense.T).to(torch.bfloat16).view(torch.int16)),
                  f"gemm M={m} N={n} K={k}")
