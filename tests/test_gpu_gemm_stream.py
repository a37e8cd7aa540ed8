"""Forward products of groups of about one 128-row block on the streaming kernel, at every number of
units that a tile can have (one to nine), one and two rounds of tiles, K from one step (fewer than
the loads in flight) to ten, against fp32 products and the 256 x 256 kernel.

Tolerance: bf16 operands, fp32 sums, one rounding to bf16 (2^-9 relative) and the fast exponential:
5e-3 in the 2-norm."""

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu


# blocks of 128 rows; N weight rows: units per tile 1, 2 and 3, 3 and 4, 4 and 5, 5 and 6, 6 and 7, 7 and 8, 8 and 9
@pytest.mark.parametrize("blocks,K", [(2, 64), (5, 192), (7, 128), (9, 640), (20, 192), (24, 64), (28, 128), (33, 256), (17, 640)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_every_tile_width(cuda, blocks, K, swiglu):
    N = 2048 if swiglu else 4096
    # groups of one and two blocks, empty ones between
    height = [1, 0, 2, 1, 0] * 16
    cu, G, left = [], 0, blocks
    while left:
        h = min(height[G], left)
        left -= h
        cu.append(blocks - left)
        G += 1
    M = 128 * (blocks + 1)
    print(f"stream blocks={blocks} G={G} M={M} N={N} K={K} swiglu={swiglu}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(blocks * K)
    A = torch.randn(M, K, device=cuda, generator=g).to(torch.bfloat16)
    B, B2 = (torch.randn(G, N, K, device=cuda, generator=g).to(torch.bfloat16) * K ** -0.5 for _ in range(2))
    scale = torch.rand(M, device=cuda, generator=g) + 0.1
    ends = torch.tensor([128 * c for c in cu], dtype=torch.int32, device=cuda)
    got = {}
    for tile in (128, 256):
        C = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=cuda)
        _lib.check(_lib.lib().mep_set_gemm_row_tile(tile), "mep_set_gemm_row_tile")
        try:
            rc = _lib.lib().mep_grouped_gemm_nt(A.data_ptr(), B.data_ptr(), B2.data_ptr() if swiglu else None, ends.data_ptr(), G,
                                                C.data_ptr(), None if swiglu else scale.data_ptr(), M, N, K, int(swiglu),
                                                _lib.current_stream())
        finally:
            _lib.check(_lib.lib().mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
        _lib.check(rc, "mep_grouped_gemm_nt")
        got[tile] = C
    assert (got[128][128 * blocks:] == 7.0).all()      # the rows of no group are left alone
    beg = 0
    for i, c in enumerate(cu):
        end = 128 * c
        if end > beg:
            x = A[beg:end].float()
            want = x @ B[i].float().t()
            want = torch.nn.functional.silu(want) * (x @ B2[i].float().t()) if swiglu else want * scale[beg:end, None]
            for tile in (128, 256):
                assert float((got[tile][beg:end].float() - want).norm() / want.norm()) < 5e-3, (i, tile)
        beg = end
