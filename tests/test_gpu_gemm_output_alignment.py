"""bf16 outputs of the grouped products may start at any element: the same bits as on a 16-byte
boundary, from each kernel, and nothing written beside the output."""

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu

M, G = 640, 3
ENDS = (256, 256, 512)      # two row blocks of a 256-row tile and a short last one; a row block of no group


def _out(n, cols, offset, cuda):
    """(flat buffer, [n, cols] view that starts `offset` elements past a 16-byte boundary)"""
    flat = torch.full((n * cols + 64,), 7.0, dtype=torch.bfloat16, device=cuda)
    return flat, flat[16 + offset:16 + offset + n * cols].view(n, cols)


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("product", ["nt", "swiglu", "dual_nt", "nn", "dual_nn"])
def test_output_at_any_element(cuda, product, tile):
    N, K = 512, 192
    lib = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(3)
    A, A2 = (torch.randn(M, K, device=cuda, generator=g).to(torch.bfloat16) for _ in range(2))
    B, B2 = (torch.randn(G, N * K, device=cuda, generator=g).to(torch.bfloat16) for _ in range(2))
    ends = torch.tensor(ENDS, dtype=torch.int32, device=cuda)
    a, a2, b, b2, e, st = A.data_ptr(), A2.data_ptr(), B.data_ptr(), B2.data_ptr(), ends.data_ptr(), _lib.current_stream()
    got = {}
    for offset in (0, 1, 2, 5):
        print(product, tile, offset, flush=True)
        outs = [_out(M, N, offset + (i if offset else 0), cuda) for i in range(3 if product == "swiglu" else 1)]
        c = [v.data_ptr() for _, v in outs]
        _lib.check(lib.mep_set_gemm_row_tile(tile), "mep_set_gemm_row_tile")
        try:
            rc = {"nt": lambda: lib.mep_grouped_gemm_nt(a, b, None, e, G, c[0], None, M, N, K, 0, st),
                  "swiglu": lambda: lib.mep_grouped_swiglu_nt(a, b, b2, e, G, *c, M, N, K, st),
                  "dual_nt": lambda: lib.mep_grouped_gemm_dual_nt(a, b, a2, b2, e, G, c[0], M, N, K, st),
                  "nn": lambda: lib.mep_grouped_gemm_nn(a, b, e, G, c[0], None, M, N, K, st),
                  "dual_nn": lambda: lib.mep_grouped_gemm_dual_nn(a, b, a2, b2, e, G, c[0], M, N, K, st)}[product]()
        finally:
            _lib.check(lib.mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
        _lib.check(rc, product)
        for flat, view in outs:
            start = view.storage_offset()
            assert (flat[:start] == 7.0).all() and (flat[start + M * N:] == 7.0).all()
            assert (view[ENDS[-1]:] == 7.0).all() and not (view[:ENDS[-1]] == 7.0).all()
        got[offset] = [v.clone().view(torch.int16) for _, v in outs]
        for x, y in zip(got[offset], got[0]):
            assert torch.equal(x, y)


def test_ffn_output_at_any_element(cuda):
    H, Hp, Gf = 256, 256, 4
    lib = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(4)
    rows = torch.randn(M, H, device=cuda, generator=g).to(torch.bfloat16)
    gate, up, down = (torch.randn(Gf, 256, 256, device=cuda, generator=g).to(torch.bfloat16) for _ in range(3))
    ends = torch.tensor((*ENDS, ENDS[-1]), dtype=torch.int32, device=cuda)
    want = None
    for offset in (0, 1, 2, 5):
        print("ffn", offset, flush=True)
        flat, y = _out(M, H, offset, cuda)
        act = torch.empty(M, Hp, dtype=torch.bfloat16, device=cuda)
        _lib.check(lib.mep_ffn_forward(rows.data_ptr(), None, ends.data_ptr(), Gf, gate.data_ptr(), up.data_ptr(), down.data_ptr(),
                                       act.data_ptr(), None, None, y.data_ptr(), 1, M, H, Hp, _lib.current_stream()), "mep_ffn_forward")
        start = y.storage_offset()
        assert (flat[:start] == 7.0).all() and (flat[start + M * H:] == 7.0).all()
        assert (y[ENDS[-1]:] == 0).all()
        want = y.clone() if want is None else want
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
