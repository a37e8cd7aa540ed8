"""Forward products whose K is a multiple of 2048: their K steps go through the two halves of every 4 KB of a row in turn.  Every step
has to come once: one piece of 4 KB, two and three, beside the shapes next to them whose steps go up, with tiles of one
unit and of nine, on the streaming kernel and the 256 x 256 ones (few tiles and many, short ones and tall).  All agree to the bit, and
the sums of a row tile do not depend on the tiles beside it.

Tolerance: bf16 operands, fp32 sums, one rounding to bf16 (2^-9 relative) and the fast exponential: 5e-3 in the
2-norm.  A step left out or taken twice is off by sqrt(64 / K), 0.1 at K = 6144."""

import pytest
import torch

from moonep_amd import _lib, ffn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [1, 17])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("K", [1984, 2048, 2112, 4096, 6144])
def test_every_step_once(cuda, K, swiglu, blocks):
    N = 512 if blocks == 1 else 2048 if swiglu else 4096
    print(f"stream fold blocks={blocks} N={N} K={K} swiglu={swiglu}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randn(128 * blocks, K, device=cuda, generator=g).to(torch.bfloat16)
    B, B2 = (torch.randn(2, N, K, device=cuda, generator=g).to(torch.bfloat16) * K ** -0.5 for _ in range(2))
    ends = torch.tensor([128, 128 * blocks], dtype=torch.int32, device=cuda)
    _lib.check(_lib.lib().mep_set_gemm_row_tile(256), "mep_set_gemm_row_tile")
    try:
        wide = ffn.launch_grouped_gemm_nt(A, B, ends, up_weights=B2 if swiglu else None)
        _lib.check(_lib.lib().mep_set_gemm_row_tile(128), "mep_set_gemm_row_tile")
        got = ffn.launch_grouped_gemm_nt(A, B, ends, up_weights=B2 if swiglu else None)
        alone = ffn.launch_grouped_gemm_nt(A[:128].contiguous(), B[:1].contiguous(), ends[:1].contiguous(),
                                           up_weights=B2[:1].contiguous() if swiglu else None)
    finally:
        _lib.check(_lib.lib().mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
    assert torch.equal(got[:128], alone) and torch.equal(got, wide)
    for i, rows in enumerate((slice(0, 128), slice(128, 128 * blocks))):
        x = A[rows].float()
        want = x @ B[i].float().t()
        if swiglu:
            want = torch.nn.functional.silu(want) * (x @ B2[i].float().t())
        assert float((got[rows].float() - want).norm()) <= 5e-3 * float(want.norm()), i
