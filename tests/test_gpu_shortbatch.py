"""The short-batch GEMM (16 < M <= 64) where it can go wrong: the first and last row counts of each row
block, ragged column tiles, K of one step and of fewer steps than waves, K ranges that end inside a
scale group, every group size, dtype pair and layout it takes, strided operands, and the plan without a
workspace. Against the oracle's product of the once-rounded bf16 weights, per element."""
import numpy as np
import pytest

from oracle import quant as oq
from tests import _cases as C

pytestmark = pytest.mark.gpu


def _check(y, x, w, acc_scale=1e-5):
    """bf16 result of an fp32 sum: half an ulp of bf16 plus the sum's own rounding."""
    exact = oq.linear_ref(x, w)
    tol = 2.0 ** -8 * np.abs(exact) + acc_scale * np.abs(exact).max()
    bad = np.abs(C.t2np(y) - exact) > tol
    assert not bad.any(), (int(bad.sum()), np.argwhere(bad)[:4].tolist())


def _group_case(dev, bits, N, K, G, sdt, zdt, seed):
    r = C.rng(seed)
    ng = K // G
    codes = r.integers(0, 1 << bits, (N, K), dtype=np.uint8)
    q = np.zeros((N, K * bits // 8), np.uint8)
    for i in range(8 // bits):
        q |= codes[:, i::8 // bits] << (bits * i)
    s = oq.round_to(r.uniform(0.005, 0.05, (N, ng)).astype(np.float32), sdt)
    z = oq.round_to(r.uniform(0, (1 << bits) - 1, (N, ng)).astype(np.float32), zdt)
    w = oq.round_to(oq.dequant_exact(codes, s, z, G, K).astype(np.float32), "bf16")
    return C.u8(q, dev), C.to_torch(s, sdt, dev), C.to_torch(z, zdt, dev), w


CASES = [
    # M, N, K, bits, G, scale dtype, zero dtype
    (17, 37, 64, 4, 64, "bf16", "bf16"), (32, 100, 448, 4, 64, "fp16", "bf16"), (33, 33, 576, 4, 32, "bf16", "fp32"),
    (64, 2944, 768, 4, 128, "fp32", "fp32"), (48, 4096, 4096, 4, 128, "bf16", "bf16"), (31, 257, 14336, 4, 256, "fp16", "fp16"),
    (20, 30000, 512, 4, 128, "bf16", "bf16"), (17, 96, 448, 2, 64, "fp16", "fp16"), (64, 1000, 8192, 2, 64, "fp16", "fp16"),
    (32, 16400, 1024, 2, 32, "bf16", "fp16"), (40, 300, 28672, 2, 128, "fp32", "bf16"),
    # each form on line-tiled weights too
    (17, 48, 512, 4, 128, "fp16", "fp16"), (32, 14336, 512, 4, 128, "bf16", "bf16"), (21, 2000, 8192, 4, 128, "fp16", "fp16"),
    (17, 48, 512, 2, 64, "bf16", "bf16"), (30, 48, 4096, 2, 64, "fp16", "fp16"), (32, 14336, 512, 2, 64, "fp32", "fp32"),
    (18, 30000, 512, 2, 64, "bf16", "bf16"), (33, 48, 512, 2, 64, "fp16", "fp16"), (64, 2000, 8192, 2, 64, "bf16", "bf16"),
]


def test_every_form_is_covered():
    """int4 and int2: one or two blocks of 32 rows with each count of column blocks, in both layouts."""
    from infinitemodel_amd import _lib
    want = {(1, 1), (1, 2), (1, 4), (2, 1), (2, 2)}
    for b in (4, 2):
        of = lambda M, N, K, G: (-(-M // 32), _lib.launch_plan(_lib.IMQ_PLAN_GEMM_WK, M, K, G, N, sqn=K * b // 8)[0])   # noqa: E731
        mine = [c for c in CASES if c[3] == b]
        assert {of(M, N, K, G) for M, N, K, _, G, _, _ in mine} == want
        assert {of(M, N, K, G) for M, N, K, _, G, s, z in mine if s == z and _tiles(N, K, b, G)} == want


def _tiles(N, K, bits, G):
    return N % 16 == 0 and (K * bits // 8) % 128 == 0 and G == (128 if bits == 4 else 64)


@pytest.mark.parametrize("M,N,K,bits,G,sdt,zdt", CASES)
def test_group_formats_match_the_oracle(dev, M, N, K, bits, G, sdt, zdt):
    import torch
    from infinitemodel_amd import ops
    q, s, z, w = _group_case(dev, bits, N, K, G, sdt, zdt, seed=M + N + K)
    x = C.bf16_normal(C.rng(M), (M, K))
    op = ops.linear_w4 if bits == 4 else ops.linear_w2
    y = op(C.to_torch(x, "bf16", dev), q, G, (s, z))
    _check(y, x, w)
    # strided operands: padded activation and weight rows, column-major scales, padded output rows
    xw = torch.zeros(M, K + 24, dtype=torch.bfloat16, device=dev)
    xw[:, 8:8 + K] = C.to_torch(x, "bf16", dev)
    qw = torch.zeros(N, q.shape[1] + 64, dtype=torch.uint8, device=dev)
    qw[:, :q.shape[1]] = q
    out = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device=dev)
    op(xw[:, 8:8 + K], qw[:, :q.shape[1]], G, (s.t().contiguous().t(), z.t().contiguous().t()), out=out[:, :N])
    assert torch.equal(out[:, :N], y) and bool((out[:, N:] == 7).all())
    if _tiles(N, K, bits, G) and sdt == zdt:
        tiled = ops.linear_w4_tiled if bits == 4 else ops.linear_w2_tiled
        assert torch.equal(tiled(C.to_torch(x, "bf16", dev), ops.line_tile(q), G, (s, z)), y)


@pytest.mark.parametrize("M,N,K,sdt", [(17, 40, 64, "bf16"), (33, 272, 1152, "fp16"), (64, 1008, 14336, "fp32"),
                                       (32, 14336, 4096, "fp16"), (5, 48, 128, "bf16"), (16, 4096, 14336, "fp16"),
                                       (8, 65552, 128, "bf16"), (9, 65552, 128, "bf16"), (12, 37, 192, "fp32")])
def test_int8_matches_the_oracle(dev, M, N, K, sdt):
    import torch
    from infinitemodel_amd import ops
    r = C.rng(N + K)
    q = r.integers(-127, 128, (N, K), dtype=np.int8)
    s = oq.round_to(r.uniform(1e-4, 1e-3, (N, 1)).astype(np.float32), sdt)
    x = C.bf16_normal(C.rng(M), (M, K))
    qt, st, xt = torch.from_numpy(q).to(dev), C.to_torch(s, sdt, dev), C.to_torch(x, "bf16", dev)
    y = ops.linear_w8(xt, qt, st)
    _check(y, x, q.astype(np.float64) * s)
    if N % 16 == 0 and K % 128 == 0:
        assert torch.equal(ops.linear_w8_tiled(xt, ops.line_tile(qt), st), y)


def test_without_a_workspace_and_repeated(dev):
    """A shape whose plan splits K: the same call without a workspace runs unsplit, and repeats and graph
    replays of the split call agree bit for bit."""
    import torch
    from infinitemodel_amd import _lib, ops
    M, N, K = 24, 256, 8192
    assert _lib.launch_plan(_lib.IMQ_PLAN_GEMM_WK, M, K, 128, N, sqn=K // 2)[1] > 1
    q, s, z, w = _group_case(dev, 4, N, K, 128, "bf16", "bf16", seed=5)
    x = C.bf16_normal(C.rng(M), (M, K))
    xt = C.to_torch(x, "bf16", dev)
    y = ops.linear_w4(xt, q, 128, (s, z))
    _check(y, x, w)
    y0 = torch.empty_like(y)
    _lib.call("imq_linear_w4", xt.data_ptr(), K, M, K, q.data_ptr(), K // 2, s.data_ptr(), s.stride(0), 1, 0, z.data_ptr(),
              z.stride(0), 1, 0, N, 128, y0.data_ptr(), N, None, 0, torch.cuda.current_stream(dev).cuda_stream)
    _check(y0, x, w)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        yg = ops.linear_w4(xt, q, 128, (s, z))
    for _ in range(3):
        yg.zero_()
        g.replay()
        assert torch.equal(yg, y) and torch.equal(ops.linear_w4(xt, q, 128, (s, z)), y)


@pytest.mark.parametrize("M,N,K,bits,G,sdt,zdt", [
    (1, 37, 64, 2, 64, "fp16", "fp16"), (3, 100, 192, 2, 64, "bf16", "fp32"), (16, 1344, 12096, 2, 64, "fp16", "fp16"),
    (7, 2560, 3520, 2, 64, "bf16", "bf16"), (5, 33, 28736, 2, 64, "fp16", "fp16"), (2, 70, 1152, 2, 128, "fp32", "bf16"),
    (1, 37, 448, 4, 64, "bf16", "bf16"), (16, 300, 1088, 4, 64, "fp16", "bf16"), (4, 96, 320, 4, 64, "bf16", "bf16"),
    (9, 300, 2944, 4, 128, "bf16", "bf16"), (16, 130, 11008, 2, 64, "fp16", "fp16")])
def test_decode_rows_of_odd_k_match_the_exact_product(dev, M, N, K, bits, G, sdt, zdt):
    """Decode rows whose K no decode kernel takes: the folded form rounds no weight, so its results are
    the exact (q - z) s product's to fp32 summation, strided operands included."""
    import torch
    from infinitemodel_amd import ops
    r = C.rng(M + N + K)
    codes = r.integers(0, 1 << bits, (N, K), dtype=np.uint8)
    q = np.zeros((N, K * bits // 8), np.uint8)
    for i in range(8 // bits):
        q |= codes[:, i::8 // bits] << (bits * i)
    s = oq.round_to(r.uniform(0.005, 0.05, (N, K // G)).astype(np.float32), sdt)
    z = oq.round_to(r.uniform(0, (1 << bits) - 1, (N, K // G)).astype(np.float32), zdt)
    x = C.bf16_normal(C.rng(M), (M, K))
    op = ops.linear_w4 if bits == 4 else ops.linear_w2
    st, zt = C.to_torch(s, sdt, dev), C.to_torch(z, zdt, dev)
    y = op(C.to_torch(x, "bf16", dev), C.u8(q, dev), G, (st, zt))
    _check(y, x, oq.dequant_exact(codes, s, z, G, K))
    xw = torch.full((M, K + 16), float("nan"), dtype=torch.bfloat16, device=dev)
    xw[:, 8:8 + K] = C.to_torch(x, "bf16", dev)
    qw = torch.zeros(N, q.shape[1] + 16, dtype=torch.uint8, device=dev)
    qw[:, :q.shape[1]] = C.u8(q, dev)
    assert torch.equal(op(xw[:, 8:8 + K], qw[:, :q.shape[1]], G, (st.t().contiguous().t(), zt.t().contiguous().t())), y)


@pytest.mark.parametrize("M,N,K", [(5, 272, 6784), (8, 2688, 6784), (14, 100, 13696), (16, 512, 10368)])
def test_int8_decode_rows_split_k_at_any_k(dev, M, N, K):
    """int8 rows 5 to 16 whose plan splits a K that is no multiple of 256 (no other format's planes are of that
    shape): the call gets its planes and matches the oracle, and a larger workspace changes nothing."""
    import torch
    from infinitemodel_amd import _lib, ops
    plan = _lib.launch_plan(_lib.IMQ_PLAN_GEMM_WK, M, K, 0, N, sqn=K)
    need = int(_lib.lib().imq_linear_workspace_bytes(M, N, K))
    assert plan[1] > 1 and need >= 4 * plan[1] * M * N
    r = C.rng(N + K)
    q = r.integers(-127, 128, (N, K), dtype=np.int8)
    s = oq.round_to(r.uniform(1e-4, 1e-3, (N, 1)).astype(np.float32), "bf16")
    x = C.bf16_normal(C.rng(M), (M, K))
    qt, st, xt = torch.from_numpy(q).to(dev), C.to_torch(s, "bf16", dev), C.to_torch(x, "bf16", dev)
    y = ops.linear_w8(xt, qt, st)
    _check(y, x, q.astype(np.float64) * s)
    for extra in (0, 4096):                                   # the planes lie in the workspace, nothing beyond the need
        ws = torch.full((need + extra,), 0x5a, dtype=torch.uint8, device=dev)
        y1 = torch.empty_like(y)
        _lib.call("imq_linear_w8", xt.data_ptr(), K, M, K, qt.data_ptr(), K, st.data_ptr(), 1, 0, N, y1.data_ptr(), N,
                  ws.data_ptr(), ws.numel(), torch.cuda.current_stream(dev).cuda_stream)
        assert torch.equal(y1, y) and bool((ws[need:] == 0x5a).all()) and bool((ws != 0x5a).any())


@pytest.mark.parametrize("M,N,K,bits,G", [(6, 37, 320, 4, 64), (8, 70, 192, 2, 64), (6, 33, 1152, 2, 128), (12, 100, 6272, 4, 128)])
def test_non_finite_activations_at_odd_k(dev, M, N, K, bits, G):
    """Decode rows of odd K with infinite and NaN activations: an output is the sum of its own products (q - z) s x, so
    one infinity gives an infinity of that product's sign (NaN at a zero weight), opposite ones and NaN give NaN, and
    the other rows are what they are without them."""
    import torch
    from infinitemodel_amd import ops
    r = C.rng(K)
    codes = r.integers(0, 1 << bits, (N, K), dtype=np.uint8)
    q = np.zeros((N, K * bits // 8), np.uint8)
    for i in range(8 // bits):
        q |= codes[:, i::8 // bits] << (bits * i)
    s = oq.round_to(r.uniform(0.005, 0.05, (N, K // G)).astype(np.float32), "bf16")
    z = r.integers(0, 1 << bits, (N, K // G)).astype(np.float32)          # whole zero points: zero weights come up
    x = C.bf16_normal(C.rng(M), (M, K))
    clean, inf = x.copy(), np.float32("inf")
    x[1, K - 3], x[2, 5], x[3, 70] = inf, -inf, np.nan
    x[4, 1], x[4, K // 2] = inf, -inf
    x[5] = np.nan
    w = oq.dequant_exact(codes, s, z, G, K).astype(np.float64)
    assert (w[:, K - 3] == 0).any() or (w[:, 5] == 0).any()
    with np.errstate(invalid="ignore"):
        want = (x.astype(np.float64)[:, None, :] * w[None]).sum(-1)
    op = ops.linear_w4 if bits == 4 else ops.linear_w2
    args = (C.u8(q, dev), G, (C.to_torch(s, "bf16", dev), C.to_torch(z, "bf16", dev)))
    y, y0 = op(C.to_torch(x, "bf16", dev), *args), op(C.to_torch(clean, "bf16", dev), *args)
    got = C.t2np(y)
    assert np.isinf(want).any() and np.isnan(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    at = np.isinf(want)
    assert np.array_equal(np.isinf(got), at) and np.array_equal(np.sign(got[at]), np.sign(want[at]))
    rest = [i for i in range(M) if i not in (1, 2, 3, 4, 5)]
    assert torch.equal(y[rest], y0[rest]) and bool(torch.isfinite(y0).all())
    # finite activations whose sum of codes overflows, their own products not: the exact sum, all its steps
    big = np.zeros((M, K), np.float32)
    big[M - 1, ::K // 8] = 2.0 ** 127                        # times a code of 2 or more: past fp32's range
    sx = oq.round_to(np.full((N, K // G), 2.0 ** -7, np.float32), "bf16")
    got = C.t2np(op(C.to_torch(big, "bf16", dev), args[0], G, (C.to_torch(sx, "bf16", dev), args[2][1])))
    want = big.astype(np.float64) @ oq.dequant_exact(codes, sx, z, G, K).astype(np.float64).T
    assert np.isfinite(want).all()
    assert np.abs(got - want).max() <= 2.0 ** -8 * np.abs(want).max()


@pytest.mark.parametrize("M,N,K,bits,G", [(17, 33000, 64, 4, 64), (64, 20000, 64, 4, 32), (33, 33008, 512, 2, 64), (24, 131072, 64, 2, 64),
                                          (64, 33000, 192, 8, 0), (8, 16400, 192, 8, 0), (16, 16400, 64, 8, 0)])
def test_short_k_and_wide_n_are_other_kernels_calls(dev, M, N, K, bits, G):
    """Row counts of the short-batch GEMM whose plan it declines (workgroups for more than the CUs, few K steps each): the
    LDS-dequant GEMM's (int8 decode rows: the skinny kernel's), against the oracle."""
    import torch
    from infinitemodel_amd import _lib, ops
    assert _lib.launch_plan(_lib.IMQ_PLAN_GEMM_WK, M, K, G, N, sqn=K * bits // 8) is None
    x = C.bf16_normal(C.rng(M), (M, K))
    xt = C.to_torch(x, "bf16", dev)
    if bits == 8:
        r = C.rng(N + K)
        q = r.integers(-127, 128, (N, K), dtype=np.int8)
        s = oq.round_to(r.uniform(1e-4, 1e-3, (N, 1)).astype(np.float32), "bf16")
        return _check(ops.linear_w8(xt, torch.from_numpy(q).to(dev), C.to_torch(s, "bf16", dev)), x, q.astype(np.float64) * s)
    q, s, z, w = _group_case(dev, bits, N, K, G, "bf16", "bf16", seed=M + N + K)
    _check((ops.linear_w4 if bits == 4 else ops.linear_w2)(xt, q, G, (s, z)), x, w)


@pytest.mark.parametrize("M,N,K,bits,G", [(1, 40, 64, 4, 64), (16, 2048, 64, 2, 64), (12, 33, 128, 2, 64), (13, 33, 128, 2, 64), (2, 100, 320, 4, 64),
                                          (7, 64, 11136, 4, 128), (6, 64, 11136, 4, 128), (16, 33, 2304, 2, 64), (9, 4128, 2944, 4, 128), (9, 4096, 2944, 4, 128), (5, 48, 6912, 2, 64), (4, 33, 12096, 2, 64)])
def test_decode_rows_on_both_sides_of_the_folded_forms_lines(dev, M, N, K, bits, G):
    """Decode rows of odd K at the lines between the generic, skinny and folded kernels: no weight is rounded on any
    side, so each matches the exact product."""
    from infinitemodel_amd import ops
    r = C.rng(M + N + K)
    codes = r.integers(0, 1 << bits, (N, K), dtype=np.uint8)
    q = np.zeros((N, K * bits // 8), np.uint8)
    for i in range(8 // bits):
        q |= codes[:, i::8 // bits] << (bits * i)
    s = oq.round_to(r.uniform(0.005, 0.05, (N, K // G)).astype(np.float32), "bf16")
    z = oq.round_to(r.uniform(0, (1 << bits) - 1, (N, K // G)).astype(np.float32), "bf16")
    x = C.bf16_normal(C.rng(M), (M, K))
    y = (ops.linear_w4 if bits == 4 else ops.linear_w2)(C.to_torch(x, "bf16", dev), C.u8(q, dev), G,
                                                       (C.to_torch(s, "bf16", dev), C.to_torch(z, "bf16", dev)))
    _check(y, x, oq.dequant_exact(codes, s, z, G, K))
