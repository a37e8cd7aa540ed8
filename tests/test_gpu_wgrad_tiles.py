"""Tile list of the weight gradients: products with fewer tiles than XCDs, numbers of tiles and groups that
eight does not divide, three products in one launch, several ranks' groups, and more tiles than one workgroup
lists."""

import ctypes

import pytest
import torch

from moonep_amd import _lib, ffn

pytestmark = pytest.mark.gpu


def _ends(lens, cuda):
    return (torch.tensor(lens).cumsum(0) * 128).to(torch.int32).to(cuda)


@pytest.mark.parametrize("Ma,Nb", [(256, 256), (512, 512), (768, 768), (1280, 512), (256, 2304), (1024, 1792)])
@pytest.mark.parametrize("G", [2, 10, 16])
def test_every_tile_of_every_group(cuda, Ma, Nb, G):
    """Against the fp64 product: a sum of n products in fp32, in any order, is off by at most n 2^-24 of the
    sum of their magnitudes; skipped groups keep what they hold."""
    print(f"wgrad {Ma}x{Nb}, {G} groups", flush=True)
    lens = [(3 * i + 1) % 4 for i in range(G)]  # blocks: 1 0 3 2 1 ...
    ends = _ends(lens, cuda)
    rows = 128 * (sum(lens) + 1)
    g = torch.Generator(device=cuda).manual_seed(Ma + Nb + G)
    x1, x2 = (torch.randn(rows, n, generator=g, device=cuda).to(torch.bfloat16) for n in (Ma, Nb))
    got = torch.full((G, Ma, Nb), float("nan"), device=cuda)
    kept = got.clone()
    ffn.launch_grouped_gemm_wgrad_tn(x1, x2, ends, got)
    ffn.launch_grouped_gemm_wgrad_tn(x1, x2, ends, kept, skip_empty_from=G // 2)
    torch.cuda.synchronize()
    at = 0
    for i, n in enumerate(lens):
        a, b = (x[128 * at:128 * (at + n)].double() for x in (x1, x2))
        bound = 128 * n * 2.0 ** -24 * (a.abs().t() @ b.abs())
        assert bool(((got[i].double() - a.t() @ b).abs() <= bound).all()), f"group {i}"
        if n or i < G // 2:
            assert torch.equal(kept[i], got[i]), f"group {i} with empty ones skipped"
        else:
            assert bool(kept[i].isnan().all()), f"group {i} was written"
        at += n


@pytest.mark.parametrize("H,Hp,G", [(512, 256, 4), (768, 768, 10), (512, 1280, 6)])
def test_three_products_of_a_backward_are_the_single_ones(cuda, H, Hp, G):
    print(f"backward {H}x{Hp}, {G} groups", flush=True)
    lens = [(2 * i + 1) % 3 for i in range(G)]
    ends = _ends(lens, cuda)
    M = 128 * (sum(lens) + 2)
    g = torch.Generator(device=cuda).manual_seed(H + Hp + G)
    rows, dy = (torch.randn(M, H, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
    slots = torch.rand(M, generator=g, device=cuda)
    gate, up = (torch.randn(G, Hp, H, generator=g, device=cuda).to(torch.bfloat16) / 32 for _ in range(2))
    down = torch.randn(G, H, Hp, generator=g, device=cuda).to(torch.bfloat16) / 32
    _, saved = ffn.grouped_ffn_hip_forward(rows, slots, ends, gate, up, down)
    got = ffn.grouped_ffn_hip_backward(dy, rows, slots, ends, gate, up, down, saved)[2:]
    dh = ffn.launch_grouped_gemm_nn(dy, down, ends)
    dg, du, hs, _ = ffn.launch_swiglu_bwd(dh, *saved, slots, ends)
    torch.cuda.synchronize()
    for what, a, b, c in zip(("gate", "up", "down"), (dg, du, dy), (rows, rows, hs), got):
        assert torch.equal(ffn.launch_grouped_gemm_wgrad_tn(a, b, ends), c), what


# row blocks of each rank's groups: ends that differ between the ranks, empty groups on either side of the split
RANKS = {"three": ((3, 0, 1, 2, 0, 1), (0, 0, 1, 1, 2, 0), (1, 2, 0, 0, 0, 0)),
         "eleven": tuple(tuple((r + 3 * i) % 5 % 3 for i in range(10)) for r in range(11))}


@pytest.mark.parametrize("ranks", list(RANKS))
@pytest.mark.parametrize("H,Hp", [(768, 512), (2560, 1280), (256, 1024)])
def test_several_ranks_are_the_single_ones(cuda, ranks, H, Hp):
    """Each rank's six tensors of one backward call of all ranks: its own experts' and its slots', of
    which the empty ones are left as they are."""
    heights = RANKS[ranks]
    n, G, M = len(heights), len(heights[0]), 128 * (max(map(sum, heights)) + 1)
    split = G // 2
    print(f"backward of {n} ranks {H}x{Hp}, {G} groups", flush=True)
    g = torch.Generator(device=cuda).manual_seed(H + Hp + n)

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, device=cuda, generator=g) * scale).to(torch.bfloat16)

    rows, dy = normal(n, M, H), normal(n, M, H)
    gate, up = (normal(n, G, Hp, H, scale=H ** -0.5) for _ in range(2))
    down = normal(n, G, H, Hp, scale=Hp ** -0.5)
    gate_pre, up_pre = normal(n, M, Hp), normal(n, M, Hp)
    cu = torch.tensor([[128 * sum(h[:i + 1]) for i in range(G)] for h in heights], dtype=torch.int32, device=cuda)
    scale = torch.rand(n, M, device=cuda, generator=g) + 0.1
    dh, dgate, dup, hs = (torch.zeros(n, M, Hp, dtype=torch.bfloat16, device=cuda) for _ in range(4))
    drows, dslots = torch.zeros(n, M, H, dtype=torch.bfloat16, device=cuda), torch.zeros(n, M, device=cuda)
    shapes = ((Hp, H), (Hp, H), (H, Hp))
    grads = [[torch.full((n, k, *s), -3.0, device=cuda) for s in shapes] for k in (split, G - split)]
    p = _lib.ptr
    _lib.check(_lib.lib().mep_ffn_backward(
        p(dy), p(rows), p(scale), p(cu), G, p(gate), p(up), p(down), p(gate_pre), p(up_pre), p(dh), p(dgate), p(dup), p(hs),
        p(dslots), p(drows), *((ctypes.c_void_p * 3)(*map(p, t)) for t in grads), split, n, M, H, Hp, split,
        _lib.current_stream()), "mep_ffn_backward")
    torch.cuda.synchronize()
    for r, lens in enumerate(heights):
        for k, (x1, x2) in enumerate(((dgate, rows), (dup, rows), (dy, hs))):
            one = torch.full((G, *shapes[k]), -3.0, device=cuda)
            ffn.launch_grouped_gemm_wgrad_tn(x1[r], x2[r], cu[r], one, skip_empty_from=split)
            got = torch.cat([grads[0][k][r], grads[1][k][r]])
            assert torch.equal(got, one), (r, k)
            for i, blocks in enumerate(lens):
                kept = bool((got[i] == -3.0).all())
                assert kept == (blocks == 0 and i >= split) and bool(got[i].any()) == (blocks > 0 or kept), (r, k, i)


def test_more_tiles_than_a_workgroup_lists(cuda):
    """1100 groups of 16 tiles, nearly all without rows: a workgroup's share by K steps alone would be
    more than the 64 tiles that its lanes hold."""
    G, n = 1100, 1024
    lens = [1 if i in (0, 7, 549, 1099) else 0 for i in range(G)]
    ends = _ends(lens, cuda)
    g = torch.Generator(device=cuda).manual_seed(3)
    x1, x2 = (torch.randn(128 * 4, n, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
    out = torch.full((G, n, n), float("nan"), device=cuda)
    ffn.launch_grouped_gemm_wgrad_tn(x1, x2, ends, out)
    torch.cuda.synchronize()
    at = 0
    for i, full in enumerate(lens):
        if full:
            a, b = (x[128 * at:128 * (at + 1)].double() for x in (x1, x2))
            assert bool(((out[i].double() - a.t() @ b).abs() <= 2.0 ** -17 * (a.abs().t() @ b.abs())).all()), f"group {i}"
            out[i].zero_()
            at += 1
    assert not bool(out.any())
