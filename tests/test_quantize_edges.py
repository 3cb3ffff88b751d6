"""The device quantizer and re-layout where their kernels branch: group counts that fill no block,
scales at both ends of BF16 (past the range of the reciprocal), quotients on rounding boundaries,
nonfinite values; bytes against the oracle's."""

import numpy as np
import pytest

import w4a16
from oracle import oracle
from test_gpu_parity import from_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(8, 128), (8, 1152), (24, 640), (72, 3968)])
@pytest.mark.parametrize("power", [-130, -61, -58, -3, 97, 103, 122])
def test_quantize_and_tiles(cuda, n, k, power):
    """Values that are halves of a code times the scale, and their neighbours in FP32, at scales of
    2^power (its neighbourhood: the group's peak is between 3.5 and 7 scales); then the tiles, against
    the host's."""
    import torch

    print(f"quantize n={n} k={k} power={power}", flush=True)
    rng = np.random.default_rng(n * k + power)
    scale = (rng.integers(128, 256, (n, k // 128, 1)) / 128).astype(np.float32)
    half = rng.integers(-14, 15, (n, k // 128, 128)).astype(np.float32) / 2
    half[:, :, 5] = 7
    w = np.ldexp(half * scale, power).astype(np.float32)
    step = rng.integers(-1, 2, w.shape)
    w = np.where(step < 0, np.nextafter(w, np.float32(-np.inf)), np.where(step > 0, np.nextafter(w, np.float32(np.inf)), w))
    w = w.astype(np.float32).reshape(n, k)
    w[0, :128] = 0.0
    p, s = w4a16.quantize_device(torch.from_numpy(w).to(cuda))
    hp, hs = oracle.quantize(w)
    assert np.array_equal(from_dev(s).reshape(n, -1), hs)
    assert np.array_equal(from_dev(p).reshape(n, -1), hp)
    for pair in (False, True):
        dev = w4a16.TiledWeight.from_device_artifact(p, s, n, k, pair=pair)
        tp, ts = w4a16.tile_pack_host(hp, hs, n, k, pair)
        assert np.array_equal(from_dev(dev.packed), tp) and np.array_equal(from_dev(dev.scales), ts)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf"), 1e-42])
def test_refused(cuda, value):
    """A nonfinite value anywhere, or a group whose scale rounds to zero, is refused."""
    import torch

    w = torch.zeros(8, 384, device=cuda)
    w[5, 255] = value
    with pytest.raises(w4a16.W4A16Error):
        w4a16.quantize_device(w)
