"""The int2 decode kernels' results to the bit: sums of (128 + code) x per group of 64, the bias taken off with the
zero point, in the kernels' fixed order. A change of the unpack or of the order of the sums shows here."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# M, N, K -> sha256 of the bf16 results (first 16 digits), row layout and line-tiled
WANT = {(1, 256, 8192): ("be01c1631ca4f53b", "be01c1631ca4f53b"), (2, 256, 8192): ("21f6454c9956ea52", "21f6454c9956ea52"),
        (4, 128, 2048): ("76033ea15c655ecf", "76033ea15c655ecf"), (8, 256, 8192): ("4e12fa61b114bed3", "4e12fa61b114bed3"),
        (16, 128, 28672): ("323cd87424fdbc96", "323cd87424fdbc96"), (3, 128, 28672): ("56046b7661d3ac4c", "b988e38bd18a5468")}


@pytest.mark.parametrize("M,N,K", list(WANT))
def test_decode_results_to_the_bit(dev, M, N, K):
    import torch
    from infinitemodel_amd import ops
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the K splits, and so the order of the sums, are those of 256 CUs")
    r = np.random.default_rng(M + N + K)
    q = torch.from_numpy(r.integers(0, 256, (N, K // 4), dtype=np.uint8)).to(dev)
    half = lambda lo, hi, d: torch.from_numpy(r.integers(lo, hi, (N, K // 64)).astype(np.float32) / d).to(torch.float16).to(dev)   # noqa: E731
    s, z = half(5, 50, 1024), half(0, 769, 256)
    x = torch.from_numpy(r.integers(-512, 513, (M, K)).astype(np.float32) / 128).to(torch.bfloat16).to(dev)
    got = [hashlib.sha256(y.view(torch.int16).cpu().numpy().tobytes()).hexdigest()[:16]
           for y in (ops.linear_w2(x, q, 64, (s, z)), ops.linear_w2_tiled(x, ops.line_tile(q), 64, (s, z)))]
    assert tuple(got) == WANT[M, N, K]
