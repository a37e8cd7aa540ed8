"""The four-wave 256 x 256 GEMM kernel: one K step and few, tiles of 128 rows first, last and alone, more
groups than a wave has lanes, several ranks' groups, every product that takes it.

Sizes leave more than a quarter of the CUs a tile (below that another kernel runs).  Tolerance: bf16
operands, fp32 sums, one rounding to bf16 (2^-9 relative): 5e-3 in the 2-norm of every 128-row block; the
activation of a SwiGLU rounds once, too."""

import ctypes

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu

HEIGHTS = {"short tiles": (1, 0, 3, 2, 0, 5, 1, 1, 7), "short alone": (1,) * 12, "whole": (8, 0, 0, 4, 6),
           "many groups": tuple((0, 1, 0, 2)[i % 4] for i in range(150))}


@pytest.mark.parametrize("K", [64, 128, 192, 832])
@pytest.mark.parametrize("heights", HEIGHTS, ids=lambda h: h.replace(" ", "-"))
@pytest.mark.parametrize("form", ["swiglu", "swiglu saved", "plain", "scaled", "dual", "kn", "kn scaled", "kn dual"])
def test_products(cuda, form, heights, K):
    h = HEIGHTS[heights]
    G, M = len(h), 128 * (sum(h) + 2)
    N = 2304 if K == 64 else 2560 if G > 100 else 4352
    print(f"{form} {heights} K={K} N={N} M={M}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K + G)

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, device=cuda, generator=g) * scale).to(torch.bfloat16)

    kn = form.startswith("kn")
    x1, x2 = normal(M, K), normal(M, K)
    w1, w2 = (normal(G, *((K, N) if kn else (N, K)), scale=K ** -0.5) for _ in range(2))
    ends = torch.tensor([128 * sum(h[:i + 1]) for i in range(G)], dtype=torch.int32, device=cuda)
    scale = torch.rand(M, device=cuda, generator=g) + 0.1 if "scaled" in form else None
    outs = [torch.full((M, N), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(3 if form == "swiglu saved" else 1)]
    lib, p, s = _lib.lib(), _lib.ptr, _lib.current_stream()
    _lib.check(lib.mep_set_gemm_row_tile(256), "mep_set_gemm_row_tile")
    try:
        if form == "swiglu saved":
            rc = lib.mep_grouped_swiglu_nt(p(x1), p(w1), p(w2), p(ends), G, *map(p, outs), M, N, K, s)
        elif form in ("swiglu", "plain", "scaled"):
            rc = lib.mep_grouped_gemm_nt(p(x1), p(w1), p(w2) if form == "swiglu" else None, p(ends), G, p(outs[0]), p(scale), M,
                                         N, K, form == "swiglu", s)
        elif "dual" in form:
            fn = lib.mep_grouped_gemm_dual_nn if kn else lib.mep_grouped_gemm_dual_nt
            rc = fn(p(x1), p(w1), p(x2), p(w2), p(ends), G, p(outs[0]), M, N, K, s)
        else:
            rc = lib.mep_grouped_gemm_nn(p(x1), p(w1), p(ends), G, p(outs[0]), p(scale), M, N, K, s)
    finally:
        _lib.check(lib.mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
    _lib.check(rc, form)
    beg = 0
    for i, end in enumerate(ends.tolist()):
        if end == beg:
            continue
        rows = slice(beg, end)
        mats = [w[i].float() if kn else w[i].float().t() for w in (w1, w2)]
        one, two = x1[rows].float() @ mats[0], (x2 if "dual" in form else x1)[rows].float() @ mats[1]
        want = [one]
        if "dual" in form:
            want = [one + two]
        elif form.startswith("swiglu"):
            want = [torch.nn.functional.silu(one) * two, one, two]
        if scale is not None:
            want = [one * scale[rows, None]]
        for out, w in zip(outs, want):
            for b in range(0, end - beg, 128):
                d = out[beg + b:beg + b + 128].float() - w[b:b + 128]
                assert float(d.norm() / w[b:b + 128].norm()) < 5e-3, (i, b)
                # 64 columns by 16 rows, the smallest piece that one wave stores: nothing swapped
                d, n = (t.view(8, 16, N // 64, 64).square().sum((1, 3)).sqrt() for t in (d, w[b:b + 128]))
                assert float((d / n).max()) < 1e-2, (i, b)
        beg = end
    for out in outs:
        assert (out[beg:] == 7.0).all()


# row blocks of each rank's groups: ends that differ between the ranks, empty groups first, last and side by side,
# more groups in all than a wave has lanes
RANKS = {"three": ((3, 0, 5, 2, 0, 1), (0, 0, 1, 1, 9, 4), (7, 2, 1, 0, 0, 0)),
         "ten": tuple(tuple((r + 3 * i) % 5 % 3 for i in range(8)) for r in range(10))}


@pytest.mark.parametrize("slots", [True, False])
@pytest.mark.parametrize("ranks,H,Hp", [("three", 2048, 1792), ("ten", 1024, 2304)])
def test_groups_of_several_ranks(cuda, ranks, H, Hp, slots):
    """The row-tiled products of an FFN's forward and backward pass of all ranks of a group: SwiGLU with saved
    pre-activations, down (scaled and plain), dy * down and the two pairs with [K, N] weights."""
    heights = RANKS[ranks]
    n, G, M = len(heights), len(heights[0]), 128 * (max(map(sum, heights)) + 1)
    print(f"{n} ranks H={H} Hp={Hp} M={M} slots={slots}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, device=cuda, generator=g) * scale).to(torch.bfloat16)

    rows, dy = normal(n, M, H), normal(n, M, H)
    gate, up, down = normal(n, G, Hp, H, scale=H ** -0.5), normal(n, G, Hp, H, scale=H ** -0.5), normal(n, G, H, Hp, scale=Hp ** -0.5)
    cu = torch.tensor([[128 * sum(h[:i + 1]) for i in range(G)] for h in heights], dtype=torch.int32, device=cuda)
    scale = torch.rand(n, M, device=cuda, generator=g) + 0.1 if slots else None
    act, gate_pre, up_pre, dh, dgate, dup, hs = (torch.full((n, M, Hp), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(7))
    y, drows = (torch.full((n, M, H), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(2))
    dslots = torch.empty(n, M, device=cuda) if slots else None
    split = G // 2
    grads = [[torch.empty(n, s, *shape, device=cuda) for shape in ((Hp, H), (Hp, H), (H, Hp))] for s in (split, G - split)]
    lib, p, s = _lib.lib(), _lib.ptr, _lib.current_stream()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        _lib.check(lib.mep_ffn_forward(p(rows), p(scale), p(cu), G, p(gate), p(up), p(down), p(act), p(gate_pre), p(up_pre), p(y),
                                       n, M, H, Hp, s), "mep_ffn_forward")
        _lib.check(lib.mep_ffn_backward(p(dy), p(rows), p(scale), p(cu), G, p(gate), p(up), p(down), p(gate_pre), p(up_pre), p(dh),
                                        p(dgate), p(dup), p(hs), p(dslots), p(drows), *((ctypes.c_void_p * 3)(*map(p, t)) for t in grads),
                                        split, n, M, H, Hp, G, s), "mep_ffn_backward")
        torch.cuda.synchronize()
    assert sum(e.count for e in prof.key_averages() if "gemm_wide_kernel" in e.key) == 4
    for r in range(n):
        ends = cu[r].tolist()
        for i, end in enumerate(ends):
            beg = ends[i - 1] if i else 0
            t = slice(beg, end)
            if end == beg:
                continue
            x = rows[r, t].float()
            one, two = x @ gate[r, i].float().t(), x @ up[r, i].float().t()
            by = scale[r, t, None] if slots else 1.0
            checks = [(gate_pre, one), (up_pre, two), (act, torch.nn.functional.silu(one) * two),
                      (y, act[r, t].float() @ down[r, i].float().t() * by), (dh, dy[r, t].float() @ down[r, i].float()),
                      (drows, dgate[r, t].float() @ gate[r, i].float() + dup[r, t].float() @ up[r, i].float())]
            for k, (out, want) in enumerate(checks):
                d, norm = (v.view((end - beg) // 128, 128, -1, 64).square().sum((1, 3)).sqrt() for v in (out[r, t].float() - want, want))
                assert float((d / norm).max()) < 1e-2, (r, i, k)
        assert not y[r, ends[-1]:].any() and not drows[r, ends[-1]:].any()
        assert (act[r, ends[-1]:] == 7.0).all() and (dh[r, ends[-1]:] == 7.0).all()
