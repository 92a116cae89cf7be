"""The native host path of the eager calls: the same bits as the Python path wherever it takes a call, None
(so the Python path's conversions, results and errors) wherever that path does anything but launch."""
import threading

import pytest

from tests import _cases as C

pytestmark = pytest.mark.gpu


def _case(dev, bits, N=64, K=1024, dt="bf16"):
    import torch
    if bits == 8:
        c = C.int8_case(N, K, seed=1, dt=dt)
        return torch.from_numpy(c["q"].astype("int8")).to(dev), C.to_torch(c["s"], dt, dev)
    c = (C.int4_case(N, K, 128, seed=1) if bits == 4 else C.int2_case(N, K, 64, seed=1))
    return C.u8(c["q"], dev), (C.to_torch(c["s"], dt, dev), C.to_torch(c["z"], dt, dev))


def _ops(bits, tiled):
    from infinitemodel_amd import ops
    f = getattr(ops, f"linear_w{bits}" + ("_tiled" if tiled else ""))
    G = {4: 128, 2: 64, 8: 0}[bits]
    return (lambda x, q, sz: f(x, q, sz)) if bits == 8 else (lambda x, q, sz: f(x, q, G, sz)), G


@pytest.mark.parametrize("bits", [4, 2, 8])
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("M", [1, 3, 16, 17, 70])
def test_same_bits_as_the_python_path(dev, monkeypatch, bits, tiled, M):
    import torch
    from infinitemodel_amd import ops
    q, sz = _case(dev, bits)
    q = ops.line_tile(q) if tiled else q
    op, G = _ops(bits, tiled)
    wide = torch.randn(M, 1024 + 16, device=dev).to(torch.bfloat16)
    for x in (wide[:, :1024].contiguous(), wide[:, 8:8 + 1024]):
        y = ops._fast_linear(bits + 16 * tiled, x, q, sz, G, False)
        assert y is not None and not y.requires_grad
        nd = ops._fast_linear(bits + 16 * tiled, x.contiguous().reshape(1, M, 1, 1024), q, sz, G, True)
        assert nd.shape == (1, M, 1, 64) and torch.equal(nd.reshape(M, 64), y)
        a = op(x, q, sz)
        with monkeypatch.context() as m:
            m.setattr(ops, "_fast_linear", lambda *a: None)
            assert torch.equal(op(x, q, sz), y) and torch.equal(a, y)


def test_what_the_python_path_converts_or_refuses_is_left_to_it(dev):
    import torch
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from infinitemodel_amd import ops
    q, (s, z) = _case(dev, 4)
    x = torch.randn(2, 1024, device=dev).to(torch.bfloat16)
    fast = lambda x=x, q=q, s=s, z=z, k=4, g=128, nd=False: ops._fast_linear(k, x, q, (s, z), g, nd)   # noqa: E731
    y = fast()
    assert y is not None
    class Sub(torch.Tensor):
        pass
    odd = torch.empty(2 * 1024 + 8, dtype=torch.bfloat16, device=dev)[1:2049].view(2, 1024)
    for bad in (dict(x=x.float()), dict(x=x[:, :512]), dict(x=x.reshape(1, 2, 1024)), dict(x=x.t().contiguous().t()),
                dict(x=odd), dict(x=x.cpu()), dict(x=x.as_subclass(Sub)), dict(x=x[:0]), dict(q=q.cpu()), dict(q=q.to(torch.int8)),
                dict(s=s[:, :4]), dict(z=z.double()), dict(g=0), dict(g=100), dict(k=20, g=64), dict(k=3), dict(s=None)):
        assert fast(**bad) is None, list(bad)
    assert ops._fast_linear(4, x, q, [s, z], 128, False) is None and ops._fast_linear(4, x) is None
    assert torch.equal(ops.linear_w4(x.reshape(1, 2, 1024), q, 128, (s, z)), y)          # flattened, as before
    assert ops.linear_w4(x[:, :1000], q, 128, (s, z)).shape == (2, 64)                   # padded, as before
    for bad in (lambda: ops.linear_w4(x, q, 128, (s[:, :4], z)), lambda: ops.linear_w4(x.cpu(), q, 128, (s, z))):
        with pytest.raises(ValueError):
            bad()

    class F(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class D(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    for mode in (F(), D()):
        with mode:
            assert fast() is None
    seen = []
    torch.vmap(lambda v: (seen.append(fast(x=v)), v)[1])(x.reshape(1, 2, 1024))
    assert seen == [None]


def test_streams_threads_and_capture(dev):
    import torch
    from infinitemodel_amd import ops
    q, sz = _case(dev, 4)
    t = ops.line_tile(q)
    xs = [torch.randn(8, 1024, device=dev).to(torch.bfloat16) for _ in range(4)]
    want = [ops.linear_w4_tiled(x, t, 128, sz) for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                y = ops.linear_w4_tiled(xs[i], t, 128, sz)
            torch.cuda.current_stream().synchronize()
            if not torch.equal(y, want[i]):
                bad.append(i)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [th.start() for th in ts]
    [th.join() for th in ts]
    assert not bad
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = ops.linear_w4_tiled(xs[0], t, 128, sz)
    for i in (1, 2, 3):
        xs[0].copy_(xs[i])
        g.replay()
        assert torch.equal(y, want[i])


def test_what_torch_throws_stays_inside_the_call(dev):
    """An operand whose address torch refuses (as a fake tensor's): the native calls return None instead of ending the
    process, and the Python path raises torch's error."""
    import torch
    from infinitemodel_amd import ops
    q, sz = _case(dev, 4)
    x = torch.randn(2, 1024, device=dev).to(torch.bfloat16)
    y = ops.linear_w4(x, q, 128, sz)
    for bad in ("x", "q"):
        xb, qb = x.clone(), q.clone()
        torch._C._set_throw_on_mutable_data_ptr(xb if bad == "x" else qb)
        assert ops._fast_linear(4, xb, qb, sz, 128, False) is None
        assert ops._fast_linear(4, xb.reshape(1, 2, 1024) if bad == "q" else xb, qb, sz, 128, True) is None
        with pytest.raises(RuntimeError):
            ops.linear_w4(xb, qb, 128, sz)
    gu, dn = (torch.zeros(2, 64, 64, dtype=torch.uint8, device=dev), *[torch.ones(2, 64, 1, dtype=torch.bfloat16, device=dev)] * 2, 128), \
        (torch.zeros(2, 128, 64, dtype=torch.uint8, device=dev), *[torch.ones(2, 128, 1, dtype=torch.bfloat16, device=dev)] * 2, 32)
    h = torch.zeros(1, 128, dtype=torch.bfloat16, device=dev)
    torch._C._set_throw_on_mutable_data_ptr(h)
    idx, w = torch.zeros(1, 1, dtype=torch.int64, device=dev), torch.ones(1, 1, dtype=torch.bfloat16, device=dev)
    assert ops._fast_moe(h, idx, w, gu, dn, 128, 0, None, None, 1.702, 7.0) is None
    assert torch.equal(ops.linear_w4(x, q, 128, sz), y)


@pytest.mark.parametrize("native", [True, False])
def test_threads_that_share_a_stream(dev, monkeypatch, native):
    """Calls that split K into the shared workspace, from several threads on torch's default stream: another thread's
    kernel never comes between a call's partials and their sum, on either host path or between the two."""
    import torch
    from infinitemodel_amd import _lib, ops
    N, K, M = 4096, 14336, 8
    assert _lib.launch_plan(_lib.IMQ_PLAN_GEMM_WK, M, K, 0, N, sqn=K)[1] > 1          # int8 splits K
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    x = [torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16) for _ in range(4)]
    q8 = torch.randint(-127, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    q4 = torch.randint(0, 256, (N, K // 2), generator=g, device=dev, dtype=torch.uint8)
    s8 = torch.full((N, 1), 1e-3, dtype=torch.bfloat16, device=dev)
    s4 = torch.full((N, K // 128), 1e-2, dtype=torch.bfloat16, device=dev)
    q2, s2 = q4[:, :K // 4].contiguous(), torch.full((N, K // 64), 1e-2, dtype=torch.bfloat16, device=dev)
    if not native:
        monkeypatch.setattr(ops, "_fast_linear", lambda *a: None)
    out = [torch.empty(M, N, dtype=torch.bfloat16, device=dev) for _ in x]
    ops_ = [lambda i: ops.linear_w8(x[i], q8, s8), lambda i: ops.linear_w4(x[i], q4, 128, (s4, s4)),
            lambda i: ops.linear_w2(x[i], q2, 64, (s2, s2)), lambda i: ops.linear_w8(x[i], q8, s8, out=out[i])]
    want = [[f(i).clone() for f in ops_] for i in range(4)]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        for _ in range(50):
            ys = [f(i) for f in ops_]
            bad.extend((i, j) for j, y in enumerate(ys) if not torch.equal(y, want[i][j]))
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [th.start() for th in ts]
    [th.join() for th in ts]
    assert not bad, bad[:8]


@pytest.mark.parametrize("T,act", [(1, "silu_glu"), (5, "gptoss"), (40, "silu_glu")])
def test_experts_same_bits_as_the_python_path(dev, monkeypatch, T, act):
    import torch
    from infinitemodel_amd import ops, shard_compile as sc
    E, H, I = 8, 256, 128
    gu = sc.pack_linear_int4_3d((torch.randn(E, 2 * I, H, device=dev) * 0.05).to(torch.bfloat16))
    dn = sc.pack_linear_int4_3d((torch.randn(E, H, I, device=dev) * 0.05).to(torch.bfloat16))
    gu, dn = (*gu[:3], H), (*dn[:3], I)
    pad = lambda p: tuple(torch.nn.functional.pad(t, (0, t.shape[2])) if p[0].shape[2] * 2 % 256 else t for t in p[:3])   # noqa: E731
    dn = (*pad(dn), I)
    x = torch.randn(T, H, device=dev).to(torch.bfloat16)
    w, idx = torch.topk(torch.softmax(torch.randn(T, E, device=dev), -1), 2)
    w = w.to(torch.bfloat16)
    b = (torch.randn(E, 2 * I, device=dev).to(torch.bfloat16), torch.randn(E, H, device=dev).to(torch.bfloat16)) if act == "gptoss" else (None, None)
    kw = dict(act=act, gu_bias=b[0], dn_bias=b[1])
    assert ops._fast_moe(x, idx, w, gu, dn, 128, ops._ACT[act], b[0], b[1], 1.702, 7.0) is not None
    y = ops.moe_experts_w4(x, idx, w, gu, dn, 128, check_ids=False, **kw)
    monkeypatch.setattr(ops, "_fast_moe", lambda *a: None)
    assert torch.equal(ops.moe_experts_w4(x, idx, w, gu, dn, 128, check_ids=False, **kw), y)
    assert torch.equal(ops.moe_experts_w4(x, idx, w, gu, dn, 128, **kw), y)
