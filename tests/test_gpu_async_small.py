"""Small asynchronous calls, which stay on their caller's stream while the communication stream is idle: the same
results as synchronous ones on both sides of the bound, and the order that one stream for all calls would give."""

import ctypes
import threading
import time

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu

E, K, R, TP = 32, 4, 4, 16


def _make(cuda, S, H, seed=1):
    from moonep_amd import Buffer, EmulatedWorld

    g = torch.Generator(device="cuda").manual_seed(seed)
    topk = torch.topk(torch.randn(R, S, E, device=cuda, generator=g), K, dim=-1)[1].to(torch.int32)
    counts = torch.zeros(R, E, dtype=torch.int32, device=cuda)
    counts.scatter_add_(1, topk.reshape(R, -1).long(), torch.ones(R, S * K, dtype=torch.int32, device=cuda))
    world = EmulatedWorld(S, H, K, E, R, TP)
    world.hidden_buf.zero_()
    buf = Buffer(S, H, K, E, R, token_padding=TP, rank=1, world=world)
    xs = [torch.randn(S, H, device=cuda, generator=g).to(torch.bfloat16) for _ in range(2)]
    return world, buf, xs, torch.rand(S, K, device=cuda, generator=g), topk, counts


def _pass(buf, x, w, topk, counts, wait, zero_copy):
    modes = dict(zero_copy=zero_copy, router_weights_zero_copy=zero_copy, async_finish=wait)
    res = buf.dispatch(x, w, topk, counts, **modes)
    if wait:
        torch.cuda.current_stream().wait_event(res[4])
    out = buf.combine(res[3], res[0], res[1], **modes)
    if wait:
        torch.cuda.current_stream().wait_event(out[2])
    return res, out


@pytest.mark.parametrize("S,H", [(1, 512), (300, 1024), (4000, 2048), (4200, 2048)])   # 64 MiB lie between the last
@pytest.mark.parametrize("zero_copy", [True, False])
def test_same_as_synchronous(cuda, S, H, zero_copy):
    print(f"async {S} x {H} zero_copy={zero_copy}", flush=True)
    world, buf, (x, _), w, topk, counts = _make(cuda, S, H)
    got = []
    for wait in (False, True, True):
        world.hidden_buf.fill_(3)
        res, out = _pass(buf, x, w, topk[1].contiguous(), counts, wait, zero_copy)
        torch.cuda.synchronize()
        got.append([t.clone() for t in (world.hidden_buf, res[1], res[2], res[3].dst, out[0], out[1])])
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))


def test_calls_from_several_streams_keep_their_order(cuda):
    """A call whose stream is held comes before calls that are made later on other streams, small or through the
    communication stream, as if all of them went through that one."""
    S, H = 200, 1024
    world, buf, (x, y), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    wants = []
    for t in (x, y):
        res, out = _pass(buf, t, w, mine, counts, False, True)
        wants.append((res[0].clone(), out[0].clone()))
    (rows_x, want_x), (rows_y, want_y) = wants
    shard = res[0]
    assert not torch.equal(rows_x, rows_y)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for rounds in range(3):
        print(f"round {rounds}", flush=True)
        torch.cuda.synchronize()
        # held dispatch of x on one stream, combine on another
        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)
            plan, ev = buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)[3:5]
        with torch.cuda.stream(b):
            out, _, done = buf.combine(plan, shard, zero_copy=True, async_finish=True)
        done.synchronize()
        assert ev.query() and torch.equal(out, want_x)
        # held dispatch of x, then one of y whose routing is every rank's: that one goes through the communication stream
        with torch.cuda.stream(b):
            torch.cuda._sleep(20_000_000)
            buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)
        with torch.cuda.stream(a):
            rows, _, _, plan, _ = buf.dispatch(y, w, topk, counts, zero_copy=True, async_finish=True)
        with torch.cuda.stream(b):   # the communication stream is not idle
            out, _, done = buf.combine(plan, shard, zero_copy=True, async_finish=True)
        done.synchronize()
        torch.cuda.synchronize()
        assert torch.equal(out, want_y) and torch.equal(rows, rows_y)


def test_call_of_another_thread_while_one_comes_to_the_communication_stream(cuda):
    """A dispatch with every rank's routing takes the communication stream in steps: first it is ordered, then the work
    follows.  A small call of another thread in between finds that stream idle; the calls after both of them still come
    behind the work."""
    S, H = 200, 1024
    world, buf, (x, y), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    rows, _, _, plan = buf.dispatch(y, w, topk, counts, zero_copy=True)
    want = buf.combine(plan, rows, zero_copy=True)[0].clone()
    a, streams = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(6)]   # some share a hardware queue
    failures = []

    def other():
        try:
            with torch.cuda.device(cuda), torch.cuda.stream(b):
                buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)[4].synchronize()
        except Exception as e:  # noqa: BLE001 - shown by the assertion below
            failures.append(e)

    run = buf._run_dispatch

    def slowly(*args):
        for _ in range(100):
            time.sleep(0.001)
            if buf._comm_stream.query():
                break
        thread = threading.Thread(target=other)
        thread.start()
        thread.join()
        torch.cuda._sleep(20_000_000)
        run(*args)

    buf._run_dispatch = slowly
    for b in streams:
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            rows, _, _, plan, done = buf.dispatch(y, w, topk, counts, zero_copy=True, async_finish=True)
        assert not failures
        with torch.cuda.stream(b):
            out, _, last = buf.combine(plan, rows, zero_copy=True, async_finish=True)
        last.synchronize()
        assert done.query() and torch.equal(out, want)


def test_part_of_a_call_that_fails_keeps_its_place(cuda):
    """A call whose second launch is refused leaves its first one on the caller's stream: later calls come behind it.
    (The planner has run when the dispatch is refused: the context says that a rank's weight slots lie one apart.)"""
    from moonep_amd.api import _native_context

    S, H = 200, 1024
    world, buf, (x, _), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    want = buf.dispatch(x, None, mine, counts, zero_copy=True)[0].clone()
    buf._native = _native_context({**buf._ctx, "meta_chunk_padded": 1}, buf._comm_stream)
    a = torch.cuda.Stream()
    for b in [torch.cuda.Stream() for _ in range(6)]:   # some share a hardware queue with the first
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)
            with pytest.raises(RuntimeError, match="mep_dispatch failed"):
                buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)
            first = a.record_event()
        with torch.cuda.stream(b):
            rows, _, _, _, done = buf.dispatch(x, None, mine, counts, zero_copy=True, async_finish=True)
        done.synchronize()
        assert first.query() and torch.equal(rows, want)


def test_streams_of_others_may_end(cuda):
    """Calls on a stream that torch did not make go through the communication stream: the allocator is not told of a stream that
    may end before the memory does, and nothing is kept by its handle."""
    S, H = 200, 1024
    world, buf, (x, _), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    want = buf.dispatch(x, w, mine, counts, zero_copy=True)[0].clone()
    lib = _lib.lib()
    for _ in range(6):    # some share a hardware queue with the communication stream
        handle = ctypes.c_void_p()
        _lib.check(lib.mep_stream_create_limited(64, ctypes.byref(handle)), "mep_stream_create_limited")
        copy, weights = x.clone(), w.clone()
        torch.cuda.synchronize()
        with torch.cuda.stream(buf._comm_stream):
            torch.cuda._sleep(20_000_000)
            held = buf._comm_stream.record_event()
        with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
            rows, _, _, _, done = buf.dispatch(copy, weights, mine, counts, zero_copy=True, async_finish=True)
        done.synchronize()
        assert held.query() and torch.equal(rows, want)
        torch.cuda.synchronize()
        _lib.check(lib.mep_stream_destroy(handle), "mep_stream_destroy")
        del copy, weights
        again = [torch.empty_like(x) for _ in range(4)]     # the allocator looks whether their memory is free
        torch.cuda.synchronize()
        del again


def test_memory_of_another_stream_outlives_the_call(cuda):
    """Tensors that were allocated on a stream other than the caller's may be dropped as soon as the call returns: their
    memory is not handed out again while the call's work is to come."""
    S, H = 200, 1024
    world, buf, (x, _), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    want = buf.dispatch(x, w, mine, counts, zero_copy=True)[0].clone()
    side = torch.cuda.Stream()
    for _ in range(3):
        copy = x.clone()
        place = copy.data_ptr()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(20_000_000)
            rows, _, _, _, done = buf.dispatch(copy, w, mine, counts, zero_copy=True, async_finish=True)
        del copy
        others = [torch.full_like(x, 7.0) for _ in range(4)]
        assert not done.query() and place not in [t.data_ptr() for t in others]
        done.synchronize()
        assert torch.equal(rows, want)


@pytest.mark.parametrize("way", ["small", "prefetch", "all ranks"])
def test_calls_behind_those_of_the_default_stream(cuda, way):
    """A call on the default stream, then one on another: on that stream itself, where the first call of another stream finds
    no event behind the held one yet, and through the communication stream, as a prefetch and as a dispatch that knows every
    rank's routing."""
    S, H = 200, 1024
    world, buf, (x, y), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    want = {}
    for name, t in (("x", x), ("y", y)):
        res, out = _pass(buf, t, w, mine, counts, False, True)
        want[name] = res[0].clone(), out[0].clone()
    shard = res[0]
    local = torch.ones(E // R, 128, 128, dtype=torch.bfloat16, device=cuda)
    pools = [torch.zeros(R, E // R, 128, 128, dtype=torch.bfloat16, device=cuda) for _ in range(3)]
    for rounds, b in enumerate([torch.cuda.Stream() for _ in range(5)]):     # some share the default stream's hardware queue
        print(f"{way} round {rounds}", flush=True)
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)
        plan, ev = buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)[3:5]
        expect = want["x"]
        with torch.cuda.stream(b):
            if way == "prefetch":
                buf.prefetch_weight(plan, True, local_gate_weight=local, local_up_weight=local, local_down_weight=local,
                                    gate_prefetch_buffer=pools[0], up_prefetch_buffer=pools[1], down_prefetch_buffer=pools[2])
            elif way == "all ranks":
                plan = buf.dispatch(y, w, topk, counts, zero_copy=True, async_finish=True)[3]
                expect = want["y"]
            out, _, done = buf.combine(plan, shard, zero_copy=True, async_finish=True)
        done.synchronize()
        assert ev.query() and torch.equal(out, expect[1])
        torch.cuda.synchronize()
        assert torch.equal(shard, expect[0])


def test_capture_behind_a_call_of_the_default_stream(cuda):
    """A call is captured while one on the default stream is still running, and without the wait that torch.cuda.graph
    begins with: replays give what an eager call gives, and later calls keep their order."""
    S, H = 200, 1024
    world, buf, (x, y), w, topk, counts = _make(cuda, S, H)
    mine = topk[1].contiguous()
    rows_y = _pass(buf, y, w, mine, counts, True, True)[0][0].clone()
    rows_x = _pass(buf, x, w, mine, counts, True, True)[0][0].clone()
    a, held = torch.cuda.Stream(), x.clone()
    with torch.cuda.stream(a):
        buf.dispatch(y, w, mine, counts, zero_copy=True, async_finish=True)[4].wait()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    torch.cuda._sleep(20_000_000)
    ev = buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)[4]
    with torch.cuda.stream(a):
        graph.capture_begin()
        buf.dispatch(y, w, mine, counts, zero_copy=True, async_finish=True)[4].wait()
        graph.capture_end()
    ev.synchronize()
    shard = buf.hidden_nvsh_buffer_view
    for _ in range(3):
        torch.cuda.synchronize()
        assert torch.equal(shard, rows_x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(shard, rows_y)
        buf.dispatch(x, w, mine, counts, zero_copy=True, async_finish=True)[4].synchronize()
