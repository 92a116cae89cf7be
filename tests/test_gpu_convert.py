"""Device packers and dequant at the sizes where their lane split can go wrong: rows shorter than a
lane's 16 (8) columns, ragged last groups, group counts that straddle waves, every row-length form of
the int8 packer, rows that no 16-byte load may touch (odd offsets and strides) and magnitudes past
the shared-reciprocal division's range. Bit for bit against the torch definitions on the CPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DTS = ["bf16", "fp16", "fp32"]


def _tdt(dt):
    import torch
    return {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[dt]


def _same(a, b):
    import torch
    a, b = a.detach().cpu(), b.detach().cpu()
    assert a.dtype == b.dtype and a.shape == b.shape
    if a.dtype.is_floating_point:
        iv = torch.int16 if a.element_size() == 2 else torch.int32
        a, b = a.contiguous().view(iv), b.contiguous().view(iv)
    return bool(torch.equal(a, b))


def _rows(N, K, dt, seed, wide):
    """N x K weights, magnitudes from 1e-30 to 1e30 where the dtype holds them; wide: a view at an odd
    offset of rows with an odd stride."""
    import torch
    g = torch.Generator().manual_seed(seed)
    W = torch.randn(N, K, generator=g) * 0.02
    if N >= 4:
        big = 1e30 if dt != "fp16" else 3e4
        W[0], W[1] = W[0] * big, W[1] * 1e-28
        W[2] = 0.25
        W[3, : K // 2] = big
    W = W.to(_tdt(dt))
    W = torch.where(W == 0, torch.zeros_like(W), W)     # the sign of a least value of zero is the host's own choice
    if wide:
        buf = torch.zeros(N, K + 5, dtype=W.dtype)
        buf[:, 3:3 + K] = W
        W = buf[:, 3:3 + K]
    return W


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("bits,G", [(4, 128), (4, 64), (2, 64), (2, 256)])
@pytest.mark.parametrize("N,K,wide", [(7, 1, False), (9, 24, False), (33, 129, True), (130, 1031, False), (5, 2880, True),
                                      (66, 640, False)])
def test_group_packer_and_dequant_edges(dev, dt, bits, G, N, K, wide):
    from infinitemodel_amd import ops, shard_compile as sc, worker_quant as wq
    W = _rows(N, K, dt, N + K + G, wide)
    q, s, z, in_f = (sc.pack_linear_int4 if bits == 4 else sc.pack_linear_int2)(W.contiguous(), G)
    Wd = W.to(dev)
    if wide:                                    # keep the odd offset and stride on the device
        buf = Wd.new_zeros(N, K + 5)
        buf[:, 3:3 + K] = Wd
        Wd = buf[:, 3:3 + K]
    qd, sd, zd, _ = (ops.pack_w4 if bits == 4 else ops.pack_w2)(Wd, G)
    assert _same(qd, q) and _same(sd, s) and _same(zd, z)
    for odt in DTS:
        f = ops.dequant_w4 if bits == 4 else ops.dequant_w2
        ref = wq._dequant_g_torch(q, s, z, in_f, G, _tdt(odt), bits)
        assert _same(f(qd, sd, zd, in_f, G, _tdt(odt)), ref), odt
        odd = qd.new_zeros(N, qd.shape[1] + 3)[:, 1:1 + qd.shape[1]]      # byte-aligned packed rows
        odd.copy_(qd)
        assert _same(f(odd, sd, zd, in_f, G, _tdt(odt)), ref), odt


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("N,K,wide", [(3, 5, False), (5, 1024, False), (6, 1032, True), (9, 2050, False), (4, 4096, False),
                                      (5, 4104, True), (3, 8192, False), (4, 16384, False), (2, 20001, True)])
def test_int8_packer_and_dequant_edges(dev, dt, N, K, wide):
    import torch
    from infinitemodel_amd import ops, shard_compile as sc
    W = _rows(N, K, dt, N * K, wide)
    q, s = sc.pack_linear_int8(W.contiguous())
    Wd = W.to(dev)
    if wide:
        buf = Wd.new_zeros(N, K + 5)
        buf[:, 3:3 + K] = Wd
        Wd = buf[:, 3:3 + K]
    qd, sd = ops.pack_w8(Wd)
    assert _same(qd, q) and _same(sd, s)
    for odt in DTS:
        ref = q.to(_tdt(odt)) * s
        assert _same(ops.dequant_w8(qd, sd, _tdt(odt)), ref), odt
        odd = torch.zeros(N, K + 3, dtype=torch.int8, device=dev)[:, 1:1 + K]
        odd.copy_(qd)
        assert _same(ops.dequant_w8(odd, sd, _tdt(odt)), ref), odt


@pytest.mark.parametrize("sdt", DTS)
def test_zero_products_keep_their_sign(dev, sdt):
    """Scales of zero (an fp16 group whose step underflows) and of either sign: a zero product has the sign of its
    factors, as torch's has, in every dtype written."""
    import torch
    from infinitemodel_amd import ops, worker_quant as wq
    g = torch.Generator().manual_seed(5)
    N, K = 24, 264
    s = torch.tensor([0.0, -0.0, 0.01, -0.01]).repeat(N // 4)[:, None].to(_tdt(sdt))
    q8 = torch.randint(-3, 4, (N, K), generator=g).to(torch.int8)
    for odt in DTS:
        assert _same(ops.dequant_w8(q8.to(dev), s.to(dev), _tdt(odt)), q8.to(_tdt(odt)) * s), odt
    for bits, G, f in ((4, 64, ops.dequant_w4), (2, 64, ops.dequant_w2)):
        Kp = 320
        q = torch.randint(0, 256, (N, Kp * bits // 8), generator=g, dtype=torch.uint8)
        sg, z = s.expand(N, Kp // G).contiguous(), torch.randint(0, 4, (N, Kp // G), generator=g).to(_tdt(sdt))
        for odt in DTS:
            ref = wq._dequant_g_torch(q, sg, z, K, G, _tdt(odt), bits)
            assert _same(f(q.to(dev), sg.to(dev), z.to(dev), K, G, _tdt(odt)), ref), (bits, odt)
