"""The whole-group launches (mep_*_ranks, mep_grad_reduce_batch, mep_cast_bf16 behind
moonep_amd.moe) against the per-rank operators on the same inputs: the same bits.  Sizes: rows
that are no whole wave tiles, paddings with and without rows behind the last group, one expert per
rank, projections of different sizes."""

import pytest
import torch

from moonep_amd import Buffer, EmulatedWorld, moe, routing
from moonep_amd.grad_reduce import launch_grad_reduce
from moonep_amd.prefetch import launch_prefetch_pull

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,epn,S,K,H,tp,sigma", [
    (2, 1, 1, 1, 8, 1, 0.0),            # the smallest: no padding, one entry per rank
    (4, 3, 37, 3, 136, 16, 1.0),        # H no multiple of 512
    (8, 4, 64, 8, 512, 128, 2.0),       # skewed: slots in use, long tails behind the last group
])
def test_dispatch_and_combine_of_a_group(cuda, R, epn, S, K, H, tp, sigma):
    E = R * epn
    print(f"group R={R} epn={epn} S={S} K={K} H={H}", flush=True)
    topk = torch.stack([routing.popularity_biased(S, K, E, R, r, sigma, seed=3) for r in range(R)])
    tpe = routing.tokens_per_expert(topk, E).to(cuda)
    topk = topk.to(cuda)
    g = torch.Generator().manual_seed(R + S)
    x = torch.randn(R, S, H, generator=g).to(torch.bfloat16).to(cuda)
    w = torch.rand(R, S, K, generator=g).to(cuda)
    group = moe.EmulatedGroup(S, H, K, E, R, token_padding=tp)
    rows, slots, cu, plans = moe.group_dispatch(group, x, w, topk, tpe)

    world = EmulatedWorld(S, H, K, E, R, tp)
    world.hidden_buf.zero_()
    world.meta_buf.zero_()
    bufs = [Buffer(S, H, K, E, R, token_padding=tp, rank=r, world=world) for r in range(R)]
    mine = [bufs[r].dispatch(x[r], w[r], topk, tpe, zero_copy=True, router_weights_zero_copy=True) for r in range(R)]
    for r in range(R):
        p, q = plans[r], mine[r][3]
        assert torch.equal(rows[r], bufs[r].hidden_nvsh_buffer_view)
        assert torch.equal(slots[r], bufs[r].router_weight_buffer_view)
        assert torch.equal(cu[r], mine[r][2])
        n, d = (int(v) for v in q.dup_counts)
        assert torch.equal(p.dup_counts, q.dup_counts)
        assert torch.equal(p.dup_groups[:n], q.dup_groups[:n]) and torch.equal(p.dup_loffs[:d], q.dup_loffs[:d])
        for a, b in ((p.dst, q.dst), (p.experts_to_copy, q.experts_to_copy), (p.remote_stats, q.remote_stats),
                     (p.zero_fill_ranges, q.zero_fill_ranges)):
            assert torch.equal(a, b)
    out = moe.group_combine(group, plans, rows)
    stacked = moe.group_combine(group, [m[3] for m in mine], rows)     # plans of another origin
    for r in range(R):
        want = bufs[r].combine(mine[r][3], bufs[r].hidden_nvsh_buffer_view, zero_copy=True)[0]
        assert torch.equal(out[r], want) and torch.equal(stacked[r], want)
    for b in (group, *bufs):
        b.destroy()


@pytest.mark.parametrize("R,epn,shapes", [(2, 2, ((128, 128), (128, 256), (256, 128))), (4, 5, ((256, 256),) * 3)])
def test_views_and_gradient_sums_of_a_group(cuda, R, epn, shapes):
    g = torch.Generator().manual_seed(R * epn)
    etc = torch.full((R, epn), -1, dtype=torch.int32)
    for d in range(R):
        for b in range(epn - 1):
            etc[d, b] = int(torch.randint(0, R * epn, (1,), generator=g))
    etc = etc.to(cuda)

    class Group:
        pass

    group = Group()
    group.R, group.epn = R, epn
    master = [torch.randn(R, epn, *s, generator=g).to(cuda) for s in shapes]
    views = moe._fill_views(group, etc, master)
    for m, v in zip(master, views):
        local = m.to(torch.bfloat16)
        pool = torch.zeros_like(local)
        for r in range(R):
            launch_prefetch_pull((local,) * 3, (pool,) * 3, etc, rank=r)
        assert torch.equal(v[:, :epn], local)
        for d, b in (etc >= 0).nonzero().tolist():
            assert torch.equal(v[d, epn + b], pool[d, b])
    # sums: one launch for all projections and ranks against one per projection and rank
    import ctypes as C

    from moonep_amd import _lib
    own = [torch.randn(R, epn, *s, generator=g).to(cuda) for s in shapes]
    pool = [torch.randn(R, epn, *s, generator=g).to(cuda) for s in shapes]
    want = [t.clone() for t in own]
    for o, p in zip(want, pool):
        for r in range(R):
            launch_grad_reduce(o[r], p, etc, rank=r, phase="reduce")
    arr_p, arr_i = C.c_void_p * 3, C.c_int64 * 3
    n = [a * b for a, b in shapes]
    rc = _lib.lib().mep_grad_reduce_batch(3, arr_p(*[t.data_ptr() for t in own]), arr_p(*[t.data_ptr() for t in pool]),
                                          arr_i(*[epn * k for k in n]), arr_i(*n), etc.data_ptr(), 0, R, epn, R,
                                          _lib.REDUCE_NO_CLEAR, _lib.current_stream())
    assert rc == 0
    torch.cuda.synchronize()
    for a, b in zip(own, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("R,epn,elems,owner,rank0,nranks", [
    (8, 8, 4096, 3, 0, 8),       # every hosted expert belongs to one rank
    (4, 3, 36868, 0, 0, 4),      # experts past a 128 KiB block, few experts, the first rank's
    (16, 5, 1028, 15, 9, 7),     # some of the ranks, the last rank's experts
    (4, 2, 256, 1, 2, 2),        # none of theirs
    (64, 96, 64, 37, 0, 64),     # a table that takes a list for each rank
])
def test_sums_of_several_ranks_where_one_owns_the_hosted_experts(cuda, R, epn, elems, owner, rank0, nranks):
    import ctypes as C

    from moonep_amd import _lib
    g = torch.Generator().manual_seed(R + epn)
    etc = torch.full((R, epn), -1, dtype=torch.int32)
    for d in range(min(R, 12)):
        etc[d, d % epn] = owner * epn + int(torch.randint(0, min(epn, 3), (1,), generator=g))
    own = torch.randn(nranks, epn, elems, generator=g)
    pool = torch.randn(R, epn, elems, generator=g)
    want = own.clone()
    for d, b in (etc >= 0).nonzero().tolist():      # slots are added in ascending order, in fp32
        e = int(etc[d, b])
        if rank0 <= e // epn < rank0 + nranks:
            want[e // epn - rank0, e % epn] += pool[d, b]
    etc, got, slots = etc.to(cuda), own.to(cuda), pool.to(cuda)
    arr_p, arr_i = C.c_void_p * 1, C.c_int64 * 1
    rc = _lib.lib().mep_grad_reduce_batch(1, arr_p(got.data_ptr()), arr_p(slots.data_ptr()), arr_i(epn * elems),
                                          arr_i(elems), etc.data_ptr(), rank0, nranks, epn, R, _lib.REDUCE_NO_CLEAR,
                                          _lib.current_stream())
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), want) and torch.equal(slots.cpu(), pool)


@pytest.mark.parametrize("R,epn,nbytes,full,rank0,nranks", [
    (8, 8, 16384, (5,), 0, 8),           # every occupied slot on one rank
    (4, 3, 147472, (0, 3), 0, 4),        # experts past a 128 KiB block
    (16, 70, 1040, (9, 15), 9, 7),       # some of the ranks, more slots than a wave has lanes
    (4, 2, 256, (0, 1), 2, 2),           # no slot of theirs
    (96, 86, 16, (0, 50, 95), 0, 96),    # a list that takes more than one launch
])
def test_slots_of_several_ranks_where_few_ranks_host(cuda, R, epn, nbytes, full, rank0, nranks):
    import ctypes as C

    from moonep_amd import _lib
    g = torch.Generator().manual_seed(R + epn)
    etc = torch.full((R, epn), -1, dtype=torch.int32)
    for d in full:
        etc[d, : epn - epn // 3] = torch.randint(0, R * epn, (epn - epn // 3,), generator=g).to(torch.int32)
    local = torch.randint(0, 256, (R, epn, nbytes), dtype=torch.uint8, generator=g)
    want = torch.randint(0, 256, (R, epn, nbytes), dtype=torch.uint8, generator=g)
    src, got = local.to(cuda), want.to(cuda)
    for d, b in (etc >= 0).nonzero().tolist():
        if rank0 <= d < rank0 + nranks:
            want[d, b] = local.view(-1, nbytes)[int(etc[d, b])]
    etc = etc.to(cuda)
    arr_p, arr_i = C.c_void_p * 1, C.c_int64 * 1
    stride = arr_i(epn * nbytes)
    rc = _lib.lib().mep_prefetch_pull_ranks(1, arr_p(src.data_ptr()), stride, arr_p(got.data_ptr()), stride, arr_i(nbytes),
                                            etc.data_ptr(), rank0, nranks, epn, R, _lib.current_stream())
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), want) and torch.equal(src.cpu(), local)


def _routed(cuda, R, E, S, K, H, seed):
    topk = torch.stack([routing.popularity_biased(S, K, E, R, r, 1.0, seed=seed) for r in range(R)])
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(R, S, H, generator=g).to(torch.bfloat16).to(cuda).requires_grad_()
    return x, topk.to(cuda), routing.tokens_per_expert(topk, E).to(cuda)


@pytest.mark.parametrize("used", ["rows", "slots", "both"])
def test_dispatch_backward_where_only_some_outputs_are_used(cuda, used):
    """An output that nobody used counts as one with a gradient of zeroes."""
    R, epn, S, K, H, tp = 4, 2, 21, 3, 136, 16
    group = moe.EmulatedGroup(S, H, K, R * epn, R, token_padding=tp)
    x, topk, tpe = _routed(cuda, R, R * epn, S, K, H, seed=3)
    w = torch.rand(R, S, K, device=cuda).requires_grad_()
    rows, slots, _, _ = moe.group_dispatch(group, x, w, topk, tpe)
    g_rows = torch.randn_like(rows) * (used != "slots")
    g_slots = torch.randn_like(slots) * (used != "rows")
    want = torch.autograd.grad((rows, slots), (x, w), (g_rows, g_slots), retain_graph=True)
    outs = {"rows": ((rows,), (g_rows,)), "slots": ((slots,), (g_slots,)), "both": ((rows, slots), (g_rows, g_slots))}[used]
    got = torch.autograd.grad(outs[0], (x, w), outs[1])
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_two_dispatches_of_a_group_in_flight(cuda, monkeypatch):
    """Micro-batches: the first one's combine and its backward work from the first one's plans."""
    R, epn, S, K, H, tp = 4, 2, 21, 3, 136, 16
    group = moe.EmulatedGroup(S, H, K, R * epn, R, token_padding=tp)
    batches = [_routed(cuda, R, R * epn, S, K, H, seed) for seed in (1, 2)]
    gout = torch.randn(R, S, H, device=cuda).to(torch.bfloat16)

    def finish(x, rows, plans):
        out = moe.group_combine(group, plans, rows * 2)
        return (out.detach(), *torch.autograd.grad(out, (rows, x), gout))

    want = []
    for x, topk, tpe in batches:
        rows, _, cu, plans = moe.group_dispatch(group, x, None, topk, tpe)
        want.append(finish(x, rows, plans))
    seen = []
    run = moe._dispatch_all
    monkeypatch.setattr(moe, "_dispatch_all", lambda *a: seen.append(a[3:]) or run(*a))
    flying = [moe.group_dispatch(group, x, None, topk, tpe) for x, topk, tpe in batches]
    del seen[:]
    for (x, _, _), (rows, _, cu, plans), w in zip(batches, flying, want):
        for a, b in zip(finish(x, rows, list(plans)), w):
            assert torch.equal(a, b)
        dst, zero_fill, ends = seen.pop()
        # the plans' own tensors, nothing stacked, and the groups' ends known
        assert dst.data_ptr() == plans[0].dst.data_ptr() and zero_fill.data_ptr() == plans[0].zero_fill_ranges.data_ptr()
        assert ends is not None and torch.equal(ends, cu)
    group.destroy()


def test_combine_of_a_group_takes_the_ranges_of_the_plans_it_is_given(cuda):
    import dataclasses
    R, epn, S, K, H, tp = 4, 2, 21, 3, 136, 16
    group = moe.EmulatedGroup(S, H, K, R * epn, R, token_padding=tp)
    x, topk, tpe = _routed(cuda, R, R * epn, S, K, H, 1)
    _, _, _, plans = moe.group_dispatch(group, x, None, topk, tpe)
    other = [dataclasses.replace(p, zero_fill_ranges=p.zero_fill_ranges * 0) for p in plans]
    t = moe._plan_tensors(group, other)
    assert torch.equal(t.zero_fill, torch.zeros_like(t.zero_fill)) and t.dst.data_ptr() == plans[0].dst.data_ptr()
    cloned = moe._plan_tensors(group, [p.clone() for p in plans])
    assert torch.equal(cloned.dst, t.dst) and cloned.cu is None
    turned = moe._plan_tensors(group, plans[::-1])
    assert torch.equal(turned.dst, t.dst.flip(0))
    group.destroy()


def test_shards_of_a_group_hold_what_its_operators_worked_on(cuda):
    R, epn, S, K, H, tp = 4, 2, 21, 3, 136, 16
    group = moe.EmulatedGroup(S, H, K, R * epn, R, token_padding=tp)
    x, topk, tpe = _routed(cuda, R, R * epn, S, K, H, 1)
    w = torch.rand(R, S, K, device=cuda)
    rows, slots, _, plans = moe.group_dispatch(group, x, w, topk, tpe)
    assert torch.equal(group.shards(), rows) and torch.equal(group.weight_slots(), slots)
    assert group.shards().data_ptr() == group.buffers[0].hidden_nvsh_buffer_view.data_ptr()
    # what a rank's own Buffer makes of them
    one = group.buffers[1].combine(plans[1], group.buffers[1].hidden_nvsh_buffer_view, zero_copy=True)[0]
    y = rows * 2
    out = moe.group_combine(group, plans, y)
    assert torch.equal(group.shards(), y.detach()) and torch.equal(group.weight_slots(), slots)
    assert torch.equal(out[1], one * 2)      # doubled throughout: every rounding is the same
    g_y, = torch.autograd.grad(out, y, torch.ones_like(out), retain_graph=True)
    assert torch.equal(group.shards(), g_y)
    g_rows = torch.randn(R, group.NvS, H, device=cuda).to(torch.bfloat16)
    torch.autograd.grad(rows, x, g_rows)
    assert torch.equal(group.shards(), g_rows)
    rows, none, _, _ = moe.group_dispatch(group, x, None, topk, tpe)
    assert none is None and torch.equal(group.shards(), rows) and not group.weight_slots().any()
    group.destroy()
