"""The register-B GEMM at every tile height it is built for (3 to 8 blocks of 32 rows), with and without K
splits, ragged rows and columns, each weight format and layout: against the oracle's product of the
once-rounded bf16 weights per element (int8: the exact integers), tiled against rows bit for bit."""
import numpy as np
import pytest

from oracle import quant as oq
from infinitemodel_amd import _lib
from tests import _cases as C
from tests.test_gpu_shortbatch import _check, _group_case

pytestmark = pytest.mark.gpu

# M, N, K, bits, G, dtype: on 256 CUs each pair (height, splits) below comes up
CASES = [(513, 1008, 1024, 4, 128, "bf16"), (777, 8200, 256, 4, 64, "fp16"), (1010, 1000, 4096, 4, 32, "bf16"),
         (513, 4096, 2048, 4, 128, "fp16"), (500, 16400, 256, 4, 128, "bf16"), (777, 14336, 256, 4, 128, "bf16"),
         (1010, 14336, 256, 4, 256, "fp16"), (601, 1000, 256, 2, 64, "fp16"), (777, 2000, 2048, 2, 64, "bf16"),
         (1010, 8200, 512, 2, 32, "fp16"), (601, 16400, 512, 2, 64, "bf16"), (150, 1008, 1024, 8, 0, "fp16"),
         (1010, 14336, 256, 8, 0, "bf16")]
# the heights those leave out of a format or a layout
CASES += [(150, 16, 1024, 4, 128, "fp16"), (1537, 4000, 256, 4, 128, "fp16"), (1537, 5008, 256, 4, 128, "bf16"),
          (777, 1500, 4096, 4, 64, "fp16"), (1010, 10000, 256, 4, 128, "fp16"), (1010, 11008, 256, 4, 128, "fp16"),
          (700, 16400, 256, 4, 128, "bf16"),
          (150, 16, 1024, 2, 64, "bf16"), (777, 8208, 512, 2, 64, "fp16"), (1537, 5008, 512, 2, 64, "bf16"),
          (1010, 10000, 512, 2, 64, "fp16"), (1010, 11008, 512, 2, 64, "fp16"), (700, 16400, 1024, 2, 64, "bf16"),
          (200, 8208, 4096, 2, 64, "bf16"),
          (150, 16, 384, 8, 0, "bf16"), (1537, 4000, 256, 8, 0, "fp16"), (1537, 5008, 256, 8, 0, "bf16"),
          (300, 8208, 2048, 8, 0, "fp16"), (1010, 10000, 256, 8, 0, "fp16"), (1010, 11008, 256, 8, 0, "bf16"),
          (700, 16400, 256, 8, 0, "fp16")]


def _tiles(N, K, bits, G):
    return N % 16 == 0 and (K * bits // 8) % 128 == 0 and G == {4: 128, 2: 64, 8: 0}[bits]


@pytest.mark.parametrize("M,N,K,bits,G,dt", CASES)
def test_tile_heights(dev, M, N, K, bits, G, dt):
    import torch
    from infinitemodel_amd import ops
    plan = _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, G, N, sqn=K * bits // 8)
    assert plan is not None and 3 <= plan[0] <= 8, plan
    x = C.bf16_normal(C.rng(M), (M, K))
    xt = C.to_torch(x, "bf16", dev)
    if bits == 8:
        r = C.rng(N)
        q = r.integers(-127, 128, (N, K), dtype=np.int8)
        s = oq.round_to(r.uniform(1e-4, 1e-3, (N, 1)).astype(np.float32), dt)
        qt, st = torch.from_numpy(q).to(dev), C.to_torch(s, dt, dev)
        y = ops.linear_w8(xt, qt, st)
        _check(y, x, q.astype(np.float64) * s)
        if _tiles(N, K, bits, G):
            assert torch.equal(ops.linear_w8_tiled(xt, ops.line_tile(qt), st), y)
        return
    q, s, z, w = _group_case(dev, bits, N, K, G, dt, dt, seed=N + K)
    y = (ops.linear_w4 if bits == 4 else ops.linear_w2)(xt, q, G, (s, z))
    _check(y, x, w)
    if _tiles(N, K, bits, G):
        f = ops.linear_w4_tiled if bits == 4 else ops.linear_w2_tiled
        assert torch.equal(f(xt, ops.line_tile(q), G, (s, z)), y)


def test_every_height_is_covered():
    heights = {_lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, G, N, sqn=K * b // 8)[0] for M, N, K, b, G, _ in CASES}
    assert heights == {3, 4, 5, 6, 7, 8}
    for bits in (4, 2, 8):                                     # of each format, in each layout
        of = lambda cases: {_lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, G, N, sqn=K * b // 8)[0]   # noqa: E731
                            for M, N, K, b, G, _ in cases if b == bits}
        assert of(CASES) == {3, 4, 5, 6, 7, 8}, bits
        assert of([c for c in CASES if _tiles(c[1], c[2], c[3], c[4])]) == {3, 4, 5, 6, 7, 8}, bits


@pytest.mark.parametrize("M,N,K,bits,G", [(241, 36480, 768, 4, 128), (241, 21440, 11776, 4, 128), (228, 38656, 1024, 2, 64)])
def test_rows_past_the_cus_run_taller_tiles(dev, M, N, K, bits, G):
    """Row-layout int4 and int2 calls whose short tiles outnumber the CUs run at another height than line-tiled ones, with
    the same splits: the same bits."""
    import torch
    from infinitemodel_amd import ops
    plan = _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, G, N, sqn=K * bits // 8)
    assert plan is not None and plan[0] <= 4 and -(-M // (32 * plan[0])) * -(-N // 256) * plan[1] > 256
    g = torch.Generator(device=dev).manual_seed(M)
    q = torch.randint(0, 256, (N, K * bits // 8), dtype=torch.uint8, device=dev, generator=g)
    s = (torch.rand(N, K // G, device=dev, generator=g) * 0.02 + 0.001).to(torch.bfloat16)
    z = torch.randint(0, 1 << bits, (N, K // G), device=dev, generator=g).to(torch.bfloat16)
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    op, tiled, deq = (ops.linear_w4, ops.linear_w4_tiled, ops.dequant_w4) if bits == 4 else (ops.linear_w2, ops.linear_w2_tiled, ops.dequant_w2)
    y = op(x, q, G, (s, z))
    assert torch.equal(tiled(x, ops.line_tile(q), G, (s, z)), y)
    rows = torch.cat([torch.arange(64), torch.arange(N - 64, N)]).to(dev)
    w = deq(q[rows].contiguous(), s[rows].contiguous(), z[rows].contiguous(), K, G, torch.bfloat16)
    ref = x.cpu().double() @ w.cpu().double().T
    err = (y[:, rows].cpu().double() - ref).abs().max() / ref.pow(2).mean().sqrt()
    assert err < 2.0 ** -8 * 5       # the output's own rounding, half a unit of 2^-8 at values up to 5 to 6 standard deviations
