"""The last, partial round of 256 x 256 tiles, which goes out in halves where at most half of the CUs get a tile:
rounds that are just that, one more, a few and none, with and without a single block at a group's end.

Tolerance: bf16 operands, fp32 sums, one rounding to bf16 (2^-9 relative): 5e-3 in the 2-norm of a block."""

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heights", [(34,), (33,), (5, 0, 7, 1, 20), (1,) * 17, (48,), (47, 1), (50,), (64,), (65,), (18,), (17,)],
                         ids=lambda h: "+".join(map(str, h)) if len(h) < 9 else f"{len(h)}x{h[0]}")
@pytest.mark.parametrize("form", ["plain", "swiglu", "kn dual"])
def test_partial_rounds(cuda, form, heights):
    G, M, K, N = len(heights), 128 * (sum(heights) + 1), 128, 4096
    cols = N // 2 if form == "swiglu" else N   # as many tiles: one of them is 128 gate and 128 up columns
    print(f"{form} {heights}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(heights))

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, device=cuda, generator=g) * scale).to(torch.bfloat16)

    x1, x2 = normal(M, K), normal(M, K)
    w1, w2 = (normal(G, *((K, cols) if form == "kn dual" else (cols, K)), scale=K ** -0.5) for _ in range(2))
    ends = torch.tensor([128 * sum(heights[:i + 1]) for i in range(G)], dtype=torch.int32, device=cuda)
    out = torch.full((M, cols), 7.0, dtype=torch.bfloat16, device=cuda)
    lib, p, s = _lib.lib(), _lib.ptr, _lib.current_stream()
    _lib.check(lib.mep_set_gemm_row_tile(256), "mep_set_gemm_row_tile")
    try:
        if form == "kn dual":
            rc = lib.mep_grouped_gemm_dual_nn(p(x1), p(w1), p(x2), p(w2), p(ends), G, p(out), M, cols, K, s)
        else:
            rc = lib.mep_grouped_gemm_nt(p(x1), p(w1), p(w2) if form == "swiglu" else None, p(ends), G, p(out), None, M, cols, K,
                                         form == "swiglu", s)
    finally:
        _lib.check(lib.mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
    _lib.check(rc, form)
    beg = 0
    for i, end in enumerate(ends.tolist()):
        a, b = x1[beg:end].float(), x2[beg:end].float()
        m1, m2 = (w[i].float() if form == "kn dual" else w[i].float().t() for w in (w1, w2))
        want = a @ m1 + b @ m2 if form == "kn dual" else torch.nn.functional.silu(a @ m1) * (a @ m2) if form == "swiglu" else a @ m1
        for r in range(0, end - beg, 128):
            d, n = (t.view(128, cols // 64, 64).square().sum((0, 2)).sqrt() for t in (out[beg + r:beg + r + 128].float() - want[r:r + 128],
                                                                                  want[r:r + 128]))
            assert float((d / n).max()) < 5e-3, (i, r)
        beg = end
    assert bool((out[beg:] == 7).all())
