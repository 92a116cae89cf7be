"""Device RTN packers (imq_pack_w4 / w2 / w8) are bit-identical to the host packers the cache
compiler and the load-time quantizer share (shard_compile.pack_linear_int4 / int2 / int8 on the
CPU, pinned to the oracle in test_oracle / test_packers): codes byte for byte, scale and zero bit
for bit -- including zero-padded last groups, all-zero groups (a -0.0 zero point), constant groups
(scale 1e-8) and the fp16 int8 quirk (fp16(1e-8) == 0)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DTS = ["bf16", "fp16", "fp32"]


def _tdt(dt):
    import torch
    return {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[dt]


def _bits(t):
    import torch
    t = t.detach().cpu()
    return t.view(torch.int16 if t.element_size() == 2 else torch.int32).numpy()


def _weights(N, K, dt, seed, std=0.02):
    """N(0, std) rows plus the special rows: an all-zero row, a constant row, a row with one large
    outlier, a row of tiny values (scale clamped to 1e-8)."""
    import torch
    g = torch.Generator().manual_seed(seed)
    W = torch.randn(N, K, generator=g) * std
    if N >= 4:
        W[0] = 0.0
        W[1] = 0.5
        W[2, K // 3] = 7.0
        W[3] = 1e-10
    return W.to(_tdt(dt))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("bits,G", [(4, 128), (4, 64), (4, 256), (2, 64), (2, 128)])
@pytest.mark.parametrize("N,K", [(64, 4096), (37, 300), (5, 64), (300, 1000)])
def test_group_packer_bit_identical(dev, dt, bits, G, N, K):
    from infinitemodel_amd import ops, shard_compile as sc
    W = _weights(N, K, dt, seed=N + K + G)
    host = (sc.pack_linear_int4 if bits == 4 else sc.pack_linear_int2)(W, G)
    devp = (ops.pack_w4 if bits == 4 else ops.pack_w2)(W.to(dev), G)
    assert devp[3] == host[3] == K
    assert np.array_equal(devp[0].cpu().numpy(), host[0].numpy())
    assert devp[1].dtype == host[1].dtype == W.dtype
    assert np.array_equal(_bits(devp[1]), _bits(host[1]))
    assert np.array_equal(_bits(devp[2]), _bits(host[2]))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("N,K", [(64, 4096), (37, 300), (4, 14336)])
def test_int8_packer_bit_identical(dev, dt, N, K):
    from infinitemodel_amd import ops, shard_compile as sc
    W = _weights(N, K, dt, seed=N * K)
    qh, sh = sc.pack_linear_int8(W)
    qd, sd = ops.pack_w8(W.to(dev))
    assert np.array_equal(qd.cpu().numpy(), qh.numpy())
    assert np.array_equal(_bits(sd), _bits(sh))


def test_packers_dispatch_to_the_device_and_match_the_oracle(dev):
    """shard_compile's packers take the device path for a ROCm tensor and agree with the numpy
    oracle at the C2 gate_up shape slice."""
    import torch
    from infinitemodel_amd import shard_compile as sc
    from oracle import quant as oq
    W = _weights(512, 4096, "bf16", seed=7)
    q, s, z, in_f = sc.pack_linear_int4(W.to(dev), 128)
    assert q.is_cuda and s.is_cuda
    qo, so, zo, _ = oq.pack_linear_int4(W.float().numpy(), 128, "bf16")
    assert np.array_equal(q.cpu().numpy(), qo)
    assert np.array_equal(s.float().cpu().numpy(), so) and np.array_equal(z.float().cpu().numpy(), zo)
    q8, s8 = sc.pack_linear_int8(W.to(dev))
    qo8, so8 = oq.pack_linear_int8(W.float().numpy(), "bf16")
    assert np.array_equal(q8.cpu().numpy(), qo8) and np.array_equal(s8.float().cpu().numpy(), so8)
    assert torch.equal(sc.pack_linear_int2(W.to(dev), 64)[0].cpu(), sc.pack_linear_int2(W, 64)[0])


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("K", [300, 4096, 6000, 20000])
def test_int8_packer_at_scale_zero_and_non_finite_weights(dev, dt, K):
    """Quotients outside the codes: an fp16 row whose scale rounds to 0 (w / 0 infinite, 0 / 0 NaN), infinite and NaN
    weights. Infinities clamp to +-127, NaN becomes 0, and a row's scale is that of its largest non-NaN weight."""
    import torch
    from infinitemodel_amd import ops
    W = (torch.randn(5, K, generator=torch.Generator().manual_seed(K)) * 0.02)
    W[0] = 0.0
    W[0, ::3], W[0, 1::3] = 2.0 ** -24, -2.0 ** -24          # the smallest fp16 subnormal: amax / 127 rounds to 0
    W[1, 5], W[1, K - 1] = float("nan"), float("nan")
    W[2, 7] = float("-inf")
    W = W.to(_tdt(dt))
    q, s = (t.cpu() for t in ops.pack_w8(W.to(dev)))
    v = W.double()                                           # on the host: torch's GPU divides by a scalar's reciprocal
    amax = torch.where(v.isnan(), torch.zeros_like(v), v).abs().amax(1, keepdim=True)
    want_s = torch.maximum((amax.float() / 127).to(W.dtype), torch.tensor(1e-8).to(W.dtype))
    assert torch.equal(s, want_s)
    quot = (W.float() / s.float()).to(W.dtype).float()
    want = torch.where(quot.isnan(), torch.zeros_like(quot), quot.round().clamp(-127, 127)).to(torch.int8)
    assert torch.equal(q, want)
    if dt == "fp16":
        assert float(s[0]) == 0 and set(q[0].unique().tolist()) == {-127, 0, 127}
    assert set(q[2].unique().tolist()) == {0} and float(s[2]) == float("inf")


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("N,K", [(1, 1), (9, 64), (33, 65), (17, 128), (300, 100), (5, 129), (40, 250), (7, 256), (6, 257), (21, 512), (6, 513)])
def test_int8_packer_short_rows(dev, dt, N, K):
    """Rows of 8, 16, 32 and 64 lanes, several to a wave: each row's scale and codes are its own (special rows beside
    ordinary ones), up to the last column and row."""
    from infinitemodel_amd import ops, shard_compile as sc
    W = _weights(N, K, dt, seed=N * K)
    qh, sh = sc.pack_linear_int8(W)
    qd, sd = ops.pack_w8(W.to(dev))
    assert np.array_equal(qd.cpu().numpy(), qh.numpy())
    assert np.array_equal(_bits(sd), _bits(sh))
