"""FP32 partials of a long K against the 64-bit product of the call's own intermediate, where a wave of
rows_gemm_kernel or rows_stream_kernel has more groups than one accumulator takes."""

import pytest
import torch

import w4a16

pytestmark = pytest.mark.gpu

# (hidden, inter, [(rows, draws of the activation, bound)]). The bound is the error on these inputs of the
# kernels that split K over more, shorter chains (sixteen accumulators a column beyond 3 rows, the few-row
# form up to 3), and 0.3 % for the scatter of a mean over so many outputs.
BOUNDS = [
    (5120, 17408, [(2, 40, 1.6058e-7), (3, 40, 1.6066e-7), (4, 20, 1.6911e-7), (33, 2, 1.6815e-7), (64, 2, 1.6675e-7),
                   (128, 2, 1.6784e-7), (200, 1, 1.6701e-7)]),
    (4096, 12288, [(33, 2, 1.6376e-7), (128, 2, 1.6341e-7), (200, 1, 1.6379e-7)]),
    (4096, 10240, [(33, 2, 1.6190e-7), (128, 2, 1.6351e-7), (200, 1, 1.6134e-7)]),
    (5120, 8064, [(5, 20, 1.5409e-7), (8, 20, 1.5636e-7)]),
    (5120, 8704, [(17, 4, 1.6370e-7), (64, 2, 1.6362e-7), (200, 1, 1.6335e-7)]),
    (5120, 5120, [(64, 2, 1.6175e-7), (200, 2, 1.6275e-7)]),
    (16384, 16384, [(2, 10, 1.6763e-7), (4, 10, 1.7397e-7)]),
]


def random_weight(gen, n, k, pair):
    codes = torch.randint(-7, 8, (2, n, k // 2), generator=gen, dtype=torch.int8).view(torch.uint8) & 15
    scales = (0.002 + 0.002 * torch.rand(n, k // 128, generator=gen)).to(torch.bfloat16)
    packed = codes[0] | codes[1] << 4
    return w4a16.TiledWeight.from_device_artifact(packed.cuda(), scales.view(torch.int16).cuda(), n, k, pair=pair)


def partial_error(lib, rows, gu, dn, dense, gen):
    """The relative error (2-norms) of one FP32 partial in the Python binding `lib`."""
    hidden, inter = dn.n, dn.k
    x = torch.randn(rows, hidden, generator=gen).to(torch.bfloat16).cuda()
    ws = torch.empty(rows, inter, device="cuda", dtype=torch.bfloat16)
    y = lib.mlp_int4(x, gu, dn, act_ws=ws, partial_f32=True).double()
    if 4 <= rows <= 16 and 64 <= inter // 128 <= 192:  # the intermediate is chunk-major
        ws = ws.view(inter // 8, rows, 8).permute(1, 0, 2).reshape(rows, inter)
    exact = ws.double() @ dense.T
    return float((y - exact).norm() / exact.norm())


@pytest.mark.parametrize("hidden,inter,rows", BOUNDS)
def test_partial_error(cuda, hidden, inter, rows):
    gen = torch.Generator().manual_seed(hidden + inter)
    gu = random_weight(gen, 2 * inter, hidden, True)
    dn = random_weight(gen, hidden, inter, False)
    dense = dn.dequantize().double()
    for m, draws, bound in rows:
        err = sum(partial_error(w4a16, m, gu, dn, dense, gen) for _ in range(draws)) / draws
        print(f"H={hidden} I={inter} M={m}: {err:.4e}, bound {bound:.4e}", flush=True)
        assert err <= 1.003 * bound
