"""The expert FFN in one call (mep_ffn_forward / mep_ffn_backward behind grouped_ffn_hip and its
training pair) against fp32 autograd on the CPU, on both tilings: tile remainders, more than 64
groups, empty groups, unused rows at the end (zero in y and drows whatever memory they land in),
and weight gradients split over two sets of buffers.

Tolerance: operands are bf16, sums fp32; the intermediate activation and its gradient round to bf16
once more (2^-8 relative), so a result's error is a few times 2^-8 of its own size in the 2-norm:
1e-2 covers two roundings and the fast exponential."""

import pytest
import torch

from moonep_amd import _lib, ffn

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=[128, 256])
def row_tile(request):
    _lib.check(_lib.lib().mep_set_gemm_row_tile(request.param), "mep_set_gemm_row_tile")
    yield request.param
    _lib.check(_lib.lib().mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")


def _rel(got, want):
    return float((got.float().cpu() - want).norm() / want.norm().clamp(min=1e-20))


@pytest.mark.parametrize("H,Hp,blocks,tail", [
    (256, 256, (1, 0), 0),                             # one 128-row block, an empty group
    (256, 512, (3, 0, 2, 0, 1, 5), 3),                 # odd and even heights
    (768, 256, (0,) * 70 + (1, 9) + (0,) * 24, 1),     # 96 groups: two rounds of the group search; a group of panels
    (512, 256, (2, 2, 17, 0), 2),                      # more row tiles than a panel holds
])
def test_forward_and_backward(cuda, H, Hp, blocks, tail):
    G, M = len(blocks), 128 * (sum(blocks) + tail)
    print(f"ffn H={H} Hp={Hp} G={G} M={M}", flush=True)
    g = torch.Generator().manual_seed(H + Hp + G)
    cu = torch.tensor([128 * sum(blocks[:i + 1]) for i in range(G)], dtype=torch.int32)
    bf = lambda *s, sc=1.0: (torch.randn(*s, generator=g) * sc).to(torch.bfloat16)  # noqa: E731
    rows, dy = bf(M, H), bf(M, H)
    slots = torch.rand(M, generator=g) + 0.1
    gate, up, down = bf(G, Hp, H, sc=H ** -0.5), bf(G, Hp, H, sc=H ** -0.5), bf(G, H, Hp, sc=Hp ** -0.5)
    rows[int(cu[-1]):] = 0
    ref = [t.float().requires_grad_() for t in (rows, slots, gate, up, down)]
    out, beg = torch.zeros(M, H), 0
    pieces = []
    for i in range(G):
        end = int(cu[i])
        if end > beg:
            x, s = ref[0][beg:end], ref[1][beg:end, None]
            h = torch.nn.functional.silu(x @ ref[2][i].t()) * (x @ ref[3][i].t())
            pieces.append(s * (h @ ref[4][i].t()))
        beg = end
    out = torch.cat([*pieces, torch.zeros(M - beg, H)])
    grads = torch.autograd.grad(out, ref, dy.float())
    d = [t.to(cuda) for t in (rows, slots, cu, gate, up, down)]

    def poison():      # what the next allocations of these sizes find
        t = [torch.full((M, n), float("nan"), dtype=torch.bfloat16, device=cuda) for n in (H, H, H, Hp, Hp, Hp)]
        torch.cuda.synchronize()
        del t

    poison()
    y = ffn.grouped_ffn_hip(*d)
    poison()
    y2, saved = ffn.grouped_ffn_hip_forward(*d)
    assert torch.equal(y, y2) and _rel(y, out.detach()) < 1e-2
    assert not y[beg:].any()
    poison()
    drows, dslots, *dw = ffn.grouped_ffn_hip_backward(dy.to(cuda), *d, saved)
    assert not drows[beg:].any() and not dslots[beg:].any()
    for got, want in zip((drows, dslots, *dw), grads):
        assert _rel(got, want) < 1e-2
    # gradients into two sets of buffers, empty groups of the upper half left alone
    own, other = ([torch.full((G // 2, *t.shape[1:]), 7.0, device=cuda) for t in dw] for _ in range(2))
    res = _lib.host().ffn_backward(*d, 128, dy.to(cuda), *saved, True, tuple(own), tuple(other))
    assert torch.equal(res[0], drows) and res[2] is None
    for lo, hi, want in zip(own, other, dw):
        assert torch.equal(lo, want[:G // 2])
        for i in range(G // 2):
            assert torch.equal(hi[i], want[G // 2 + i]) if blocks[G // 2 + i] else bool((hi[i] == 7.0).all())
