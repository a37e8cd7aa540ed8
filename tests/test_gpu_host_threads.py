"""The native host path lets other Python threads run while a call waits: for a place in a full launch
queue here."""

import sys
import threading
import time

import pytest
import torch

from moonep_amd import Buffer, ffn

pytestmark = pytest.mark.gpu


def _prefetch(cuda):
    E, R, H, Hp = 8, 2, 128, 128
    buf = Buffer(64, 8, 2, E, R, rank=1)
    topk = (torch.arange(128, dtype=torch.int32, device=cuda) % E).view(64, 2)
    counts = torch.bincount(topk.flatten(), minlength=E).to(torch.int32).repeat(R, 1)
    plan = buf.dispatch(torch.zeros(64, 8, dtype=torch.bfloat16, device=cuda), None, topk, counts, zero_copy=True)[3]
    local = [torch.zeros(E // R, H, Hp, dtype=torch.bfloat16, device=cuda) for _ in range(3)]
    pools = [torch.zeros(R, E // R, H, Hp, dtype=torch.bfloat16, device=cuda) for _ in range(3)]
    names = ("gate", "up", "down")
    kw = {f"local_{n}_weight": t for n, t in zip(names, local)} | {f"{n}_prefetch_buffer": t for n, t in zip(names, pools)}
    return buf, lambda: buf.prefetch_weight(plan, **kw)


def _exchange(cuda):
    E, R, S, H, K = 8, 2, 16, 64, 2
    buf = Buffer(S, H, K, E, R, rank=1)
    topk = (torch.arange(S * K, dtype=torch.int32, device=cuda) % E).view(S, K)
    counts = torch.bincount(topk.flatten(), minlength=E).to(torch.int32).repeat(R, 1)
    x = torch.zeros(S, H, dtype=torch.bfloat16, device=cuda)

    def call():
        rows, _, _, plan = buf.dispatch(x, None, topk, counts, zero_copy=True)
        buf.combine(plan, rows, zero_copy=True)
    return buf, call


def _ffn(cuda):
    M, H, Hp, G = 256, 256, 256, 2
    rows = torch.zeros(M, H, dtype=torch.bfloat16, device=cuda)
    cu = torch.tensor([128, 256], dtype=torch.int32, device=cuda)
    gate, up, down = (torch.zeros(G, 256, 256, dtype=torch.bfloat16, device=cuda) for _ in range(3))
    args = (rows, None, cu, gate, up, down)

    def call():
        _, saved = ffn.grouped_ffn_hip_forward(*args)
        ffn.grouped_ffn_hip_backward(rows, *args, saved)
    return None, call


@pytest.mark.parametrize("make", [_prefetch, _exchange, _ffn])
def test_other_threads_run_while_a_launch_waits(cuda, make):
    buf, call = make(cuda)
    for _ in range(3):
        call()
    torch.cuda.synchronize()
    gaps, stop = [], threading.Event()

    def watch():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.001)
            now = time.perf_counter()
            gaps.append((now - last, now))
            last = now

    interval = sys.getswitchinterval()
    sys.setswitchinterval(0.001)
    thread = threading.Thread(target=watch)
    thread.start()
    try:
        torch.cuda._sleep(1_200_000_000)     # half a second in front of the calls
        longest = (0.0, 0.0)
        for _ in range(40_000):              # until one of them has waited
            t0 = time.perf_counter()
            call()
            t1 = time.perf_counter()
            longest = max(longest, (t1 - t0, t1))
            if t1 - t0 > 0.1:
                break
    finally:
        stop.set()
        thread.join()
        sys.setswitchinterval(interval)
        torch.cuda.synchronize()
    waited, end = longest
    during = max(g for g, now in gaps if end - waited < now)
    print(f"{make.__name__}: a call waited {waited * 1e3:.0f} ms, the other thread at most {during * 1e3:.1f} ms", flush=True)
    assert waited > 0.05, "no call had to wait: the queue was not full"
    assert during < waited / 2
    if buf is not None:
        buf.destroy()
