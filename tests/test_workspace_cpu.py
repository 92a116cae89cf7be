"""The shared workspaces of the eager ops (ops._scratch), without a device: a call that uses one keeps every other
thread's call on the same stream out until its last launch, calls on other streams and calls that need none
go ahead, and no buffer that was handed out is ever dropped."""
import contextlib
import threading
import time

import pytest


@pytest.fixture
def cpu_ops(monkeypatch):
    """ops with host tensors, the launch replaced by ``calls`` (entry, stream, workspace pointer) and a pause."""
    import torch
    from infinitemodel_amd import ops
    at = threading.local()
    log, inside, worst = [], {}, {}
    guard = threading.Lock()

    def call(name, *args):
        stream, ws = args[-1], args[-3]
        with guard:
            log.append((name, stream, ws))
            if ws:
                inside[stream] = inside.get(stream, 0) + 1
                worst[stream] = max(worst.get(stream, 0), inside[stream])
        time.sleep(0.01)
        with guard:
            if ws:
                inside[stream] -= 1
    monkeypatch.setattr(ops, "_check_dev", lambda *a: torch.device("cpu"))
    monkeypatch.setattr(ops, "_stream", lambda dev: at.stream)
    monkeypatch.setattr(ops, "call", call)
    monkeypatch.setattr(ops, "_fast_linear", lambda *a: None)
    monkeypatch.setattr(ops, "_fast_moe", lambda *a: None)
    monkeypatch.setattr(ops, "_WS", {})
    monkeypatch.setattr(ops, "_WS_RETIRED", [])
    monkeypatch.setattr(torch.cuda, "device", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: type("S", (), {"cuda_stream": at.stream}))
    return ops, at, log, worst


def _in_threads(fns):
    errs = []

    def guarded(f):
        try:
            f()
        except Exception as exc:      # noqa: BLE001
            errs.append(exc)
    ts = [threading.Thread(target=guarded, args=(f,)) for f in fns]
    [t.start() for t in ts]
    [t.join(30) for t in ts]
    assert not errs and not any(t.is_alive() for t in ts), errs


def _calls(torch, ops):
    x = torch.zeros(8, 14336, dtype=torch.bfloat16)
    q8, s8 = torch.zeros(256, 14336, dtype=torch.int8), torch.ones(256, 1, dtype=torch.bfloat16)
    q4 = torch.zeros(256, 14336 // 2, dtype=torch.uint8)
    s4 = torch.ones(256, 112, dtype=torch.bfloat16)
    q2 = torch.zeros(256, 14336 // 4, dtype=torch.uint8)
    s2 = torch.ones(256, 224, dtype=torch.bfloat16)
    E, H, I = 4, 256, 128
    moe = (x[:, :H].contiguous(), torch.zeros(8, 2, dtype=torch.int64), torch.ones(8, 2, dtype=torch.bfloat16),
           (torch.zeros(E, 2 * I, H // 2, dtype=torch.uint8), *[torch.ones(E, 2 * I, 2, dtype=torch.bfloat16)] * 2, H),
           (torch.zeros(E, H, I // 2, dtype=torch.uint8), *[torch.ones(E, H, 1, dtype=torch.bfloat16)] * 2, I), 128)
    return [lambda: ops.linear_w8(x, q8, s8), lambda: ops.linear_w8_tiled(x, q8, s8),
            lambda: ops.linear_w4(x, q4, 128, (s4, s4)), lambda: ops.linear_w2(x, q2, 64, (s2, s2)),
            lambda: ops.moe_experts_w4(*moe, check_ids=False)]


def test_calls_that_share_a_workspace_do_not_overlap(cpu_ops):
    import torch
    ops, at, log, worst = cpu_ops
    calls = _calls(torch, ops)

    def work(stream):
        at.stream = stream
        for f in calls:
            f()
    _in_threads([lambda: work(11)] * 3 + [lambda: work(22)])
    assert len(log) == 4 * len(calls) and all(ws for _, _, ws in log)
    assert worst == {11: 1, 22: 1}
    assert {ws for _, s, ws in log if s == 11}.isdisjoint({ws for _, s, ws in log if s == 22})


def test_calls_without_a_workspace_take_no_lock(cpu_ops):
    import torch
    ops, at, log, _ = cpu_ops
    at.stream = 5
    _calls(torch, ops)[0]()
    x, q, s = torch.zeros(1, 256, dtype=torch.bfloat16), torch.zeros(16, 256, dtype=torch.int8), torch.ones(16, 1, dtype=torch.bfloat16)

    def work():
        at.stream = 5
        ops.linear_w8(x, q, s)
    with ops._WS[(None, 5)][1]:
        _in_threads([work])
    assert not log[-1][2]


def test_no_buffer_handed_out_is_dropped(cpu_ops, monkeypatch):
    """Threads that ask for a key's first or a larger workspace at once: every pointer handed out (the native path and
    captured graphs keep them) belongs to a buffer that is still held, and a key keeps its one lock."""
    import torch
    ops, at, _, _ = cpu_ops
    empty, got = torch.empty, []

    def slow(*a, **k):
        time.sleep(0.005)
        return empty(*a, **k)
    monkeypatch.setattr(torch, "empty", slow)

    def work(need):
        at.stream = 7
        for n in (need, 2 * need, 3 * need):
            got.append(ops._scratch(torch.device("cpu"), n))
    _in_threads([lambda n=n: work(n) for n in (64, 96, 128, 160)])
    held = {b.data_ptr() for b in ops._WS_RETIRED} | {ops._WS[(None, 7)][0].data_ptr()}
    assert {g[0].data_ptr() for g in got} <= held and len({id(g[1]) for g in got}) == 1
    assert len(held) <= 9        # sizes at least double


def test_a_workspace_taken_while_one_is_allocated_is_kept(cpu_ops, monkeypatch):
    """A finalizer that runs inside the allocation may itself make a call on the same stream."""
    import torch
    ops, at, _, _ = cpu_ops
    at.stream = 9
    empty, inner = torch.empty, []

    def nested(*a, **k):
        if not inner:
            inner.append(None)
            inner[0] = ops._scratch(torch.device("cpu"), 512)
        return empty(*a, **k)
    monkeypatch.setattr(torch, "empty", nested)
    outer = ops._scratch(torch.device("cpu"), 64)
    assert outer[1] is inner[0][1]
    assert any(b is inner[0][0] for b in [*ops._WS_RETIRED, ops._WS[(None, 9)][0]])
