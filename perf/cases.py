"""The workloads whose speed this package is judged by.

A case is one pass that a training or serving program makes through the public entry points:

* ``exchange``  -- ``Buffer.dispatch`` then ``Buffer.combine`` of one rank: a layer's forward (fresh plan)
  or its backward (saved plan; tokens only on the way out, route-weight gradients on the way back);
* ``prefetch``  -- ``Buffer.prefetch_weight``: the three projections of the experts that other ranks host;
* ``reduce``    -- ``Buffer.reduce_grad``: the fp32 gradients of those experts summed home;
* ``ffn``       -- the grouped expert FFN of one rank's rows, for inference;
* ``ffn_train`` -- the same with the backward pass, weight gradients in fp32;
* ``layer``     -- a whole MoE layer of an emulated group, forward and backward through autograd.

Sizes are those of this repository's benchmark (S=4096/8192, H=4096/7168, E=128/256/384, K=8, R=8,
H'=2048), its tests' small and ragged ones, and decode batches of a few tokens.  ``skew`` is the
standard deviation of the per-expert logit bias: 0.1 gives maxvio ~ 1, 0.3 maxvio ~ 4.
"""

from __future__ import annotations

import dataclasses
import math

import torch

from moonep_amd import Buffer, EmulatedWorld, ffn, moe

# the bounds of what draw() gives: one rank's share of the largest benchmark shapes
_MOST_EXCHANGE = 8192 * 8 * 4096          # S * K * H
_MOST_SHARDS = 10 * 10**9                 # bytes of all ranks' shards
_MOST_FFN = 4096 * 8 * 7168 * 2048        # S * K * H * H'
_MOST_POOL = 8 * 32 * 7168 * 2048         # elements of an all-rank weight pool
_MOST_LAYER = 8 * 512 * 8 * 2048 * 1024   # R * S * K * H * H'


def listed():
    exchange = dict(kind="exchange", plan="fresh", weights=True, copy=False, wait="stream", tp=128, skew=0.1)
    return [
        # one decode step of a small batch: latency of the launches and of the host path
        dict(exchange, name="decode 8 tokens", S=8, H=4096, K=8, E=128, R=8),
        # a ragged batch of a model whose sizes are no powers of two, other top-k and padding
        dict(exchange, name="ragged 333 tokens", S=333, H=2880, K=6, E=96, R=4, tp=64, skew=0.3),
        # a training or prefill step at the benchmark's main configuration, zero-copy views
        dict(exchange, name="forward 4096 tokens", S=4096, H=7168, K=8, E=256, R=8),
        # the same with the call's defaults, which copy the rows out of and back into the shard
        dict(exchange, name="forward 8192 copied", S=8192, H=4096, K=8, E=128, R=8, copy=True, skew=0.2),
        # the backward of the main configuration on the communication stream
        dict(exchange, name="backward 4096 tokens", S=4096, H=7168, K=8, E=256, R=8, plan="saved", wait="event"),
        # quantised weights with their scales, small experts: a serving step's prefetch
        dict(kind="prefetch", name="prefetch small uint8", dtype="uint8", H=1024, Hp=512, E=64, R=4, slots=3, fan=1),
        # the benchmark's expert shape, bf16, some experts wanted by two ranks
        dict(kind="prefetch", name="prefetch large bf16", dtype="bfloat16", H=7168, Hp=2048, E=256, R=8, slots=6, fan=2),
        # the matching gradient reduction of a training step
        dict(kind="reduce", name="reduce large", H=7168, Hp=2048, E=256, R=8, slots=4, fan=2),
        # expert FFN of a decode batch: a few rows per expert, bound by the weights
        dict(kind="ffn", name="ffn decode", S=64, H=4096, Hp=2048, K=8, E=128, R=8, tp=128, skew=0.1),
        # expert FFN of a prefill at the main configuration
        dict(kind="ffn", name="ffn prefill", S=4096, H=7168, Hp=2048, K=8, E=256, R=8, tp=128, skew=0.1),
        # forward and backward of the second benchmark shape: more rows per expert
        dict(kind="ffn_train", name="ffn train", S=4096, H=4096, Hp=2048, K=8, E=128, R=8, tp=128, skew=0.1),
        # a training step of a whole layer, every rank of the group on this GPU
        dict(kind="layer", name="layer train", S=512, H=2048, Hp=1024, K=8, E=64, R=8, tp=128, skew=0.1),
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _routing_sizes(rng):
    R = rng.choice((2, 4, 8, 8, 16))
    epn = rng.choice((2, 4, 8, 12, 16, 32, 48))
    E = R * epn
    K = min(rng.choice((1, 2, 4, 6, 8, 8, 8)), E)
    return dict(R=R, E=E, K=K, skew=round(rng.uniform(0.0, 0.3), 3))


def _padded_rows(c):
    epn = c["E"] // c["R"]
    return -(-(c["S"] * c["K"] + (c["tp"] - 1) * 2 * epn) // c["tp"]) * c["tp"]


def draw(rng):
    kind = rng.choice(("exchange", "exchange", "exchange", "exchange", "prefetch", "reduce", "ffn", "ffn_train", "layer"))
    while True:
        if kind == "exchange":
            c = dict(_routing_sizes(rng), kind=kind, S=_log_int(rng, 1, 8192), tp=rng.choice((16, 64, 128, 128)),
                     H=rng.choice((_log_int(rng, 512, 8192, 8), _log_int(rng, 512, 8192, 512))),
                     plan=rng.choice(("fresh", "fresh", "saved")), weights=rng.random() < 0.8,
                     copy=rng.random() < 0.3)
            # a program that overlaps its communication works on the views
            c["wait"] = "stream" if c["copy"] else rng.choice(("stream", "stream", "event"))
            if c["S"] * c["K"] * c["H"] <= _MOST_EXCHANGE and c["R"] * _padded_rows(c) * c["H"] * 2 <= _MOST_SHARDS:
                return c
        elif kind in ("prefetch", "reduce"):
            R, epn = rng.choice((2, 4, 8, 8)), rng.choice((4, 8, 16, 32))
            c = dict(kind=kind, R=R, E=R * epn, H=_log_int(rng, 512, 7168, 128), Hp=_log_int(rng, 256, 2048, 128),
                     slots=_log_int(rng, 1, min(epn, 8)), fan=rng.choice((1, 1, min(2, R - 1))))
            if kind == "prefetch":
                c["dtype"] = rng.choice(("bfloat16", "bfloat16", "uint8"))
            if c["E"] * c["H"] * c["Hp"] <= _MOST_POOL:
                return c
        elif kind in ("ffn", "ffn_train"):
            c = dict(_routing_sizes(rng), kind=kind, S=_log_int(rng, 8, 8192), H=_log_int(rng, 512, 7168, 256),
                     Hp=_log_int(rng, 256, 2048, 256), tp=rng.choice((128, 128, 256)))
            # the backward counts three times; half the size keeps it under the largest listed case
            if c["S"] * c["K"] * c["H"] * c["Hp"] <= _MOST_FFN // (1 if kind == "ffn" else 2) and \
                    c["E"] // c["R"] * c["H"] * c["Hp"] <= 16 * 4096 * 2048:
                return c
        else:
            c = dict(_routing_sizes(rng), kind=kind, S=_log_int(rng, 32, 1024), H=_log_int(rng, 512, 2048, 256),
                     Hp=_log_int(rng, 256, 1024, 256), tp=128)
            if c["R"] * c["S"] * c["K"] * c["H"] * c["Hp"] <= _MOST_LAYER and c["E"] * c["H"] * c["Hp"] <= 64 * 2048 * 1024:
                return c


# -- inputs ------------------------------------------------------------------------------------

def _routing(c, g):
    """Every rank's top-k experts, their softmax weights and the gathered counts."""
    S, K, E, R = c["S"], c["K"], c["E"], c["R"]
    bias = torch.randn(E, device="cuda", generator=g) * c["skew"]
    logits = torch.randn(R, S, E, device="cuda", generator=g) + bias
    v, topk = torch.topk(logits, K, dim=-1)
    counts = torch.zeros(R, E, dtype=torch.int32, device="cuda")
    counts.scatter_add_(1, topk.reshape(R, -1), torch.ones(R, S * K, dtype=torch.int32, device="cuda"))
    return topk.to(torch.int32), torch.softmax(v, dim=-1), counts


def _normal(shape, scale, g, dtype=torch.bfloat16):
    out = torch.empty(shape, dtype=dtype, device="cuda")
    out.normal_(0.0, scale, generator=g)
    return out


def _prepare_exchange(c, g):
    S, H, K, E, R = (c[k] for k in ("S", "H", "K", "E", "R"))
    topk, w, counts = _routing(c, g)
    rank = R // 2
    world = EmulatedWorld(S, H, K, E, R, c["tp"])
    world.hidden_buf.normal_(0.0, 1.0, generator=g)   # the rows that the other ranks sent
    buf = Buffer(S, H, K, E, R, token_padding=c["tp"], rank=rank, world=world)
    st = dict(c=c, world=world, buf=buf, x=_normal((S, H), 1.0, g), w=w[rank].contiguous(),
              topk=topk[rank].contiguous(), counts=counts)
    if c["plan"] == "saved":
        st["plan"] = buf.dispatch(st["x"], st["w"], st["topk"], counts, zero_copy=True, router_weights_zero_copy=True)[3]
    return st


def _plan_of(E, R, S=64, K=2):
    """A plan and the Buffer that made it; the operators on weights use the plan's slot table only."""
    buf = Buffer(S, 8, K, E, R, rank=R // 2)
    topk = (torch.arange(S * K, dtype=torch.int32, device="cuda") % E).view(S, K)
    counts = torch.bincount(topk.flatten(), minlength=E).to(torch.int32).repeat(R, 1)
    return buf, buf.dispatch(torch.zeros(S, 8, dtype=torch.bfloat16, device="cuda"), None, topk, counts, zero_copy=True)[3]


def _slot_table(c, g):
    """[R, epn]: every rank hosts ``slots`` experts of the other ranks, ``fan`` ranks the same one."""
    R, epn, slots = c["R"], c["E"] // c["R"], c["slots"]
    table = torch.full((R, epn), -1, dtype=torch.int32)
    order = torch.stack([torch.randperm(epn, device="cuda", generator=g) for _ in range(R)]).cpu()
    given = [0] * R
    for b in range(slots):
        for d in range(R):
            owner = (d + 1 + b % (R - 1)) % R
            table[d, b] = owner * epn + int(order[owner, given[owner] // c["fan"]])
            given[owner] += 1
    return table.cuda()


def _active(c):
    return -(-c["slots"] // c["fan"])


def _prepare_weights(c, g):
    R, epn, H, Hp = c["R"], c["E"] // c["R"], c["H"], c["Hp"]
    buf, plan = _plan_of(c["E"], R)
    plan = dataclasses.replace(plan, experts_to_copy=_slot_table(c, g))
    st = dict(c=c, buf=buf, plan=plan)
    if c["kind"] == "reduce":
        st["local"] = [_normal((epn, H, Hp), 1e-3, g, torch.float32) for _ in range(3)]
        st["pools"] = [_normal((R, epn, H, Hp), 1e-3, g, torch.float32) for _ in range(3)]
    elif c["dtype"] == "bfloat16":
        st["local"] = [_normal((epn, H, Hp), 0.02, g) for _ in range(3)]
        st["pools"] = [torch.zeros(R, epn, H, Hp, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    else:
        # packed low-bit weights and one scale byte per 32 of them, padded to what the copy takes
        scale = -(-(H * Hp // 32) // 16384) * 128
        for key, shape in (("local", (H, Hp)), ("scales", (128, scale))):
            st[key] = [torch.randint(0, 256, (epn, *shape), dtype=torch.uint8, device="cuda", generator=g) for _ in range(3)]
        st["pools"] = [torch.zeros(R, epn, H, Hp, dtype=torch.uint8, device="cuda") for _ in range(3)]
        st["scale_pools"] = [torch.zeros(R, epn, 128, scale, dtype=torch.uint8, device="cuda") for _ in range(3)]
    return st


def _prepare_ffn(c, g):
    S, H, Hp, K, E, R = (c[k] for k in ("S", "H", "Hp", "K", "E", "R"))
    G = 2 * (E // R)
    topk, _, counts = _routing(c, g)
    rank = R // 2
    buf = Buffer(S, 8, K, E, R, token_padding=c["tp"], rank=rank)   # the groups come from the planner; rows are made below
    _, _, cu, plan = buf.dispatch(torch.zeros(S, 8, dtype=torch.bfloat16, device="cuda"), None,
                                  topk[rank].contiguous(), counts, zero_copy=True)
    NvS = plan.NvS
    rows, slots = _normal((NvS, H), 1.0, g), torch.rand(NvS, device="cuda", generator=g) * 0.3 + 0.02
    for start, n in plan.zero_fill_ranges.tolist() + [[int(cu[-1]), NvS - int(cu[-1])]]:
        rows[start:start + n] = 0
        slots[start:start + n] = 0
    buf.destroy()
    st = dict(c=c, rows=rows, slots=slots, cu=cu, gate=_normal((G, Hp, H), 0.02, g), up=_normal((G, Hp, H), 0.02, g),
              down=_normal((G, H, Hp), 0.02, g))
    if c["kind"] == "ffn_train":
        st["dy"] = _normal((NvS, H), 1.0, g)
        st["dy"][int(cu[-1]):] = 0
    return st


def _prepare_layer(c, g):
    S, H, Hp, K, E, R = (c[k] for k in ("S", "H", "Hp", "K", "E", "R"))
    topk, w, counts = _routing(c, g)
    epn = E // R
    master = [_normal((R, epn, *shape), 0.02, g, torch.float32).requires_grad_() for shape in ((Hp, H), (Hp, H), (H, Hp))]
    return dict(c=c, group=moe.EmulatedGroup(S, H, K, E, R, token_padding=c["tp"]), topk=topk, counts=counts,
                x=_normal((R, S, H), 1.0, g).requires_grad_(), w=w.contiguous().requires_grad_(), master=master,
                gout=_normal((R, S, H), 1.0, g))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    make = {"exchange": _prepare_exchange, "prefetch": _prepare_weights, "reduce": _prepare_weights,
            "ffn": _prepare_ffn, "ffn_train": _prepare_ffn, "layer": _prepare_layer}[case["kind"]]
    return make(case, g)


# -- one pass ----------------------------------------------------------------------------------

def _run_exchange(st):
    c, buf = st["c"], st["buf"]
    zero_copy, wait = not c["copy"], c["wait"] == "event"
    modes = dict(zero_copy=zero_copy, router_weights_zero_copy=zero_copy, async_finish=wait)
    if c["plan"] == "fresh":
        res = buf.dispatch(st["x"], st["w"] if c["weights"] else None, st["topk"], st["counts"], **modes)
    else:
        res = buf.dispatch(st["x"], plan=st["plan"], **modes)
    rows, slots, cu, plan = res[:4]
    if wait:
        torch.cuda.current_stream().wait_event(res[4])
    # the experts would rewrite `rows` here; the gradients of the route weights lie in their slots
    if c["plan"] == "saved" and c["weights"]:
        slots = buf.router_weight_buffer_view
        modes["router_weights_zero_copy"] = True
    out, w_back, done = buf.combine(plan, rows, slots, **modes)
    if wait:
        torch.cuda.current_stream().wait_event(done)
    return dict(shards=st["world"].hidden_buf, rows=rows if c["copy"] else None, slots=slots, cu=cu, dst=plan.dst,
                experts_to_copy=plan.experts_to_copy, zero_fill_ranges=plan.zero_fill_ranges,
                remote_stats=plan.remote_stats, out=out, w_back=w_back)


def _run_prefetch(st):
    scales = {}
    if "scales" in st:
        s, p = st["scales"], st["scale_pools"]
        scales = dict(local_gate_scale=s[0], local_up_scale=s[1], local_down_scale=s[2],
                      gate_scale_prefetch_buffer=p[0], up_scale_prefetch_buffer=p[1], down_scale_prefetch_buffer=p[2])
    local, pools = st["local"], st["pools"]
    st["buf"].prefetch_weight(st["plan"], local_gate_weight=local[0], local_up_weight=local[1], local_down_weight=local[2],
                              gate_prefetch_buffer=pools[0], up_prefetch_buffer=pools[1], down_prefetch_buffer=pools[2],
                              **scales)
    return dict(pools=pools, scale_pools=st.get("scale_pools"))


def _run_reduce(st):
    local, pools = st["local"], st["pools"]
    st["buf"].reduce_grad(st["plan"], local_gate_grad=local[0], local_up_grad=local[1], local_down_grad=local[2],
                          gate_reduce_buffer=pools[0], up_reduce_buffer=pools[1], down_reduce_buffer=pools[2])
    return dict(local=local, pools=pools)


def _run_ffn(st):
    return ffn.grouped_ffn_hip(st["rows"], st["slots"], st["cu"], st["gate"], st["up"], st["down"],
                               token_padding=st["c"]["tp"])


def _run_ffn_train(st):
    args = (st["rows"], st["slots"], st["cu"], st["gate"], st["up"], st["down"])
    y, saved = ffn.grouped_ffn_hip_forward(*args, token_padding=st["c"]["tp"])
    return (y, *ffn.grouped_ffn_hip_backward(st["dy"], *args, saved, token_padding=st["c"]["tp"]))


def _run_layer(st):
    group = st["group"]
    rows, slots, cu, plans = moe.group_dispatch(group, st["x"], st["w"], st["topk"], st["counts"])
    y = moe.group_expert_ffn_hip(group, plans[0].experts_to_copy, cu, rows, slots, *st["master"])
    out = moe.group_combine(group, plans, y)
    return (out.detach(), *torch.autograd.grad(out, (st["x"], st["w"], *st["master"]), st["gout"]))


def run(state):
    return {"exchange": _run_exchange, "prefetch": _run_prefetch, "reduce": _run_reduce, "ffn": _run_ffn,
            "ffn_train": _run_ffn_train, "layer": _run_layer}[state["c"]["kind"]](state)


# -- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    c = case
    if c["kind"] == "exchange":
        N, row = c["S"] * c["K"], 2 * c["H"]
        # tokens read, copies written, copies read, sums written; the routing, its slots and the weights
        b = 2 * (c["S"] + N) * row + 4 * N * (2 + (c["plan"] == "fresh") + 4 * c["weights"])
        if c["copy"]:   # the shard copied out after dispatch and in before combine
            b += 4 * _padded_rows(c) * row
        return dict(bytes=b, flops=N * c["H"])
    if c["kind"] in ("prefetch", "reduce"):
        n = c["H"] * c["Hp"]
        if c["kind"] == "reduce":   # slots read, gradients read and written, own slots cleared
            return dict(bytes=3 * 4 * n * (2 * c["slots"] + 2 * _active(c)), flops=3 * n * c["slots"])
        per = 2 * n if c["dtype"] == "bfloat16" else n + n // 32
        return dict(bytes=3 * per * (c["slots"] + _active(c)), flops=0)
    N = c["S"] * c["K"]
    groups = min(c["E"] // c["R"], N * c["R"])
    weights, rows = 3 * groups * c["H"] * c["Hp"], N * c["H"]
    if c["kind"] == "ffn":
        return dict(bytes=2 * (weights + rows + _padded_rows(c) * c["H"]), flops=6 * N * c["H"] * c["Hp"])
    if c["kind"] == "ffn_train":
        # weights in, fp32 gradients of all groups out; rows and dy in, y and the rows' gradient out
        return dict(bytes=2 * weights + 4 * 3 * 2 * (c["E"] // c["R"]) * c["H"] * c["Hp"] +
                    2 * (2 * rows + 2 * _padded_rows(c) * c["H"]), flops=18 * N * c["H"] * c["Hp"])
    # fp32 masters in, their gradients out; tokens and their gradients in and out, every copy of a row
    # written and read by dispatch and combine in both directions
    R = c["R"]
    return dict(bytes=2 * 4 * R * weights + R * (4 * c["S"] + 8 * N) * 2 * c["H"], flops=18 * R * N * c["H"] * c["Hp"])


def tolerance(case):
    """Planning, copies and sums in a fixed order are exact; products of bf16 rows are rounded to bf16."""
    return {"rel": 1e-2} if case["kind"] in ("ffn", "ffn_train", "layer") else "exact"
