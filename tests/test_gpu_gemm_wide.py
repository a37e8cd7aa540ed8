"""The four-wave 256 x 256 GEMM kernel: one K step and few, tiles of 128 rows first, last and alone, more
groups than a wave has lanes, several ranks' groups, every product that takes it.

Sizes leave more than a quarter of the CUs a tile (below that another kernel runs).  Tolerance: bf16
operands, fp32 sums, one rounding to bf16 (2^-9 relative): 5e-3 in the 2-norm of every 128-row block; the
activation of a SwiGLU rounds once, too."""

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
