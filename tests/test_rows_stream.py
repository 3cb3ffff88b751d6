"""Up to 16 rows on rows_stream_kernel (a block a CU over its tile pairs and K range): where
launch_rows and the chunk-major down projection send calls to it, at odd tile and group counts,
with and without a K split, against the oracle; and the same calls captured before anything was
allocated for them."""

import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import w4a16
from conftest import assert_parity
from oracle import oracle
from test_gpu_parity import from_dev, make_ffn, make_weight, norm_inputs, to_dev, ws_act

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (2, 4136, 12544),  # more tile pairs than CUs, the last half filled; K split
    (3, 4136, 10496),
    (5, 4104, 5376),   # one K range
    (8, 4136, 8704),
    (9, 4136, 9856),
    (16, 520, 9856),   # fewer tile pairs than CUs, K split until the rows fit LDS (77 groups)
    (16, 8, 8320),     # one half-filled tile pair: fewer units than waves in the last split
    (12, 16648, 2688), # many tile pairs, short K, past the tile-pair form
])
def test_linear_parity(cuda, m, n, k):
    print(f"gemm M={m} N={n} K={k}", flush=True)
    p, s = make_weight(n, k, seed=n + k)
    x = oracle.synth_activation(m, k, seed=m + n)
    w = w4a16.TiledWeight.from_artifact(p, s, n, k, device=cuda)
    out = from_dev(w4a16.gemm_int4_bf16(to_dev(x, cuda), w))
    assert_parity(out, oracle.gemm_bf16(x, p, s, n, k), f"gemm M={m} N={n} K={k}")


@pytest.mark.parametrize("m,hidden,inter", [(8, 4352, 8196), (6, 5120, 8448), (9, 5120, 8196), (16, 5120, 8448)])
def test_gate_up_parity(cuda, m, hidden, inter):
    print(f"gate/up M={m} H={hidden} I={inter}", flush=True)
    p, s = make_weight(2 * inter, hidden, seed=hidden + inter)
    x = oracle.synth_activation(m, hidden, seed=m)
    gu = w4a16.TiledWeight.from_artifact(p, s, 2 * inter, hidden, pair=True, device=cuda)
    act = from_dev(w4a16.gate_up_silu(to_dev(x, cuda), gu))
    want = oracle.silu_mul_packed(oracle.gemm_bf16(x, p, s, 2 * inter, hidden), m, inter)
    assert_parity(act, want, f"gate/up M={m} H={hidden} I={inter}")


@pytest.mark.parametrize("m", [4, 7, 16])
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


CAPTURED_FIRST = r"""
import sys
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/haskell-infer-demo_amd"]
import torch, w4a16
M, n, k = 16, 1032, 9856
gen = torch.Generator(device="cuda"); gen.manual_seed(5)
w = torch.randn(n, k, generator=gen, device="cuda") * 0.02
p, s = w4a16.quantize_device(w.to(torch.bfloat16).float())
tw = w4a16.TiledWeight.from_device_artifact(p, s, n, k)
x = torch.randn(M, k, generator=gen, device="cuda").to(torch.bfloat16)
out = torch.zeros((M, n), dtype=torch.bfloat16, device="cuda")
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    w4a16.gemm_int4_bf16(x, tw, out)
want = w4a16.gemm_int4_bf16(x, tw).float()
for _ in range(3):
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    rel = float((out.float() - want).norm() / want.norm())
    print("replay", rel)
    w4a16.gemm_int4_bf16(x, tw)
"""


def test_first_call_under_capture(cuda):
    """In a fresh process, a call whose plan wants split scratch that is not there yet, made under
    graph capture: it takes a kernel that needs none, and each replay agrees with the eager call
    to the order of the sums (BF16 roundings that fall the other way: well under 1e-3)."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    print("first call under capture, child process", flush=True)
    proc = subprocess.run([sys.executable, "-c", CAPTURED_FIRST, root], capture_output=True, text=True, timeout=110)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    rels = [float(ln.split()[1]) for ln in proc.stdout.splitlines() if ln.startswith("replay")]
    assert len(rels) == 3 and max(rels) < 1e-3, proc.stdout
