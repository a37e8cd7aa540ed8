"""Row scales begin at any element: the streaming kernels read four at a time.  The same bits from every offset, with
weights given as [N, K] and as [K, N], for tiles of one to nine and of one to four units (the fp32 products are test_gpu_gemm_stream.py's)."""

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,blocks,K", [(form, *size) for form in ("nt", "nn")
                                            for size in [(2, 64), (5, 192), (9, 64), (17, 128), (33, 64)]])
def test_any_first_element(cuda, form, blocks, K):
    M, N = 128 * blocks, 4096
    print(f"row scales {form} blocks={blocks} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(blocks)
    A = torch.randn(M, K, device=cuda, generator=g).to(torch.bfloat16)
    B = torch.randn(blocks, N, K, device=cuda, generator=g).to(torch.bfloat16)
    ends = torch.arange(128, M + 1, 128, dtype=torch.int32, device=cuda)
    scale = torch.rand(M, device=cuda, generator=g) + 0.1
    got = []
    for first in range(5):
        shifted = torch.full((M + 8,), float("nan"), device=cuda)
        shifted[first:first + M] = scale
        C = torch.empty(M, N, dtype=torch.bfloat16, device=cuda)
        _lib.check(_lib.lib().mep_set_gemm_row_tile(128), "mep_set_gemm_row_tile")
        try:
            rows = shifted.data_ptr() + 4 * first
            if form == "nt":
                rc = _lib.lib().mep_grouped_gemm_nt(A.data_ptr(), B.data_ptr(), None, ends.data_ptr(), blocks, C.data_ptr(), rows,
                                                    M, N, K, 0, _lib.current_stream())
            else:   # the same numbers, read as [K, N]
                rc = _lib.lib().mep_grouped_gemm_nn(A.data_ptr(), B.data_ptr(), ends.data_ptr(), blocks, C.data_ptr(), rows,
                                                    M, N, K, _lib.current_stream())
        finally:
            _lib.check(_lib.lib().mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
        _lib.check(rc, form)
        got.append(C)
    assert torch.isfinite(got[0]).all() and all(torch.equal(got[0], c) for c in got[1:])
