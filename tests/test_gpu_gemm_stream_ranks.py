"""The streaming GEMM kernel on several ranks' groups: both input gradients of an FFN's backward pass
against the 256 x 256 kernels on the same inputs.  Both add K in ascending order: the same bits.  Ends that differ
between the ranks, ranks without a row first, in the middle and last, ranks whose groups are more than a
wave has lanes, the most ranks it takes (64) and one more (which the 256 x 256 kernels take)."""

import ctypes

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu

# row blocks of each rank's groups
RANKS = {"two": ((1, 0, 0, 2), (0, 1, 1, 0)),
         "empty ranks": ((0, 0), (1, 1), (0, 0), (3, 0), (0, 0)),
         "many groups": tuple(tuple((i + r) % 9 == 0 for i in range(70)) for r in range(3)),
         "sixty-four": tuple(((r % 3 == 1), (r % 5 == 0)) for r in range(64)),
         "sixty-five": tuple(((r % 3 == 1), (r % 5 == 0)) for r in range(65))}


@pytest.mark.parametrize("slots", [True, False])
@pytest.mark.parametrize("ranks,H,Hp", [("two", 768, 512), ("two", 2560, 1280), ("empty ranks", 1024, 256),
                                        ("many groups", 256, 512), ("sixty-four", 512, 256), ("sixty-five", 512, 256)],
                         ids=lambda v: str(v).replace(" ", "-"))
def test_same_bits_as_the_256_row_kernels(cuda, ranks, H, Hp, slots):
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
    lib, p, s = _lib.lib(), _lib.ptr, _lib.current_stream()
    split = G // 2
    both = []
    for tile in (128, 256):
        act, gate_pre, up_pre, dh, dgate, dup, hs = (torch.full((n, M, Hp), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(7))
        y, drows = (torch.full((n, M, H), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(2))
        dslots = torch.zeros(n, M, device=cuda) if slots else None
        grads = [[torch.zeros(n, k, *shape, device=cuda) for shape in ((Hp, H), (Hp, H), (H, Hp))] for k in (split, G - split)]
        lib.mep_set_gemm_row_tile(tile)
        try:
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
                _lib.check(lib.mep_ffn_forward(p(rows), p(scale), p(cu), G, p(gate), p(up), p(down), p(act), p(gate_pre), p(up_pre),
                                               p(y), n, M, H, Hp, s), "mep_ffn_forward")
                _lib.check(lib.mep_ffn_backward(
                    p(dy), p(rows), p(scale), p(cu), G, p(gate), p(up), p(down), p(gate_pre), p(up_pre), p(dh), p(dgate), p(dup),
                    p(hs), p(dslots), p(drows), *((ctypes.c_void_p * 3)(*map(p, t)) for t in grads), split, n, M, H, Hp, G, s),
                    "mep_ffn_backward")
                torch.cuda.synchronize()
        finally:
            lib.mep_set_gemm_row_tile(0)
        streaming = sum(e.count for e in prof.key_averages() if "gemm_stream_kernel" in e.key)
        assert streaming == (2 if tile == 128 and n <= 64 else 0)
        both.append([act, gate_pre, up_pre, y, dh, dgate, dup, drows] + ([dslots] if slots else []))
    for k, (a, b) in enumerate(zip(*both)):
        assert torch.equal(a, b), k
    y, drows = both[0][3], both[0][7]
    for r in range(n):
        end = int(cu[r, -1])
        assert not y[r, end:].any() and not drows[r, end:].any()
        if end:
            assert y[r, :end].any()


# ranks, experts of a rank, blocks of each of a rank's experts, H, H', does the streaming kernel run
@pytest.mark.parametrize("n,epn,each,H,Hp,streaming", [(4, 2, 1, 512, 256, True),      # less than a block a group
                                                       (4, 2, 2, 512, 256, False),
                                                       (2, 2, 1, 2048, 1024, True),
                                                       (2, 2, 1, 2304, 1024, False)])  # larger experts
def test_the_kernel_of_these_sizes(cuda, n, epn, each, H, Hp, streaming):
    """Which kernel brings both input gradients is a rule on sizes; the result is the other's to the bit."""
    print(f"{n} ranks of {epn} experts, {each} blocks each, {H} x {Hp}", flush=True)
    G, M = 2 * epn, 128 * (each * epn + 2 * epn)
    g = torch.Generator(device="cuda").manual_seed(n)

    def normal(*shape):
        return torch.randn(*shape, device=cuda, generator=g).to(torch.bfloat16)

    rows, dy, gate, up, down = normal(n, M, H), normal(n, M, H), normal(n, G, Hp, H), normal(n, G, Hp, H), normal(n, G, H, Hp)
    cu = (128 * each * (torch.arange(G, device=cuda) + 1).clamp(max=epn)).to(torch.int32).expand(n, G).contiguous()
    lib, p, s = _lib.lib(), _lib.ptr, _lib.current_stream()
    drows = []
    for tile in (0, 256 if streaming else 128):
        mid = [normal(n, M, Hp) * 0 for _ in range(6)]
        out = normal(n, M, H)
        grads = [[torch.zeros(n, epn, *shape, device=cuda) for shape in ((Hp, H), (Hp, H), (H, Hp))] for _ in range(2)]
        lib.mep_set_gemm_row_tile(tile)
        try:
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
                _lib.check(lib.mep_ffn_backward(
                    p(dy), p(rows), None, p(cu), G, p(gate), p(up), p(down), p(rows), p(dy), *map(p, mid[:4]), None, p(out),
                    *((ctypes.c_void_p * 3)(*map(p, t)) for t in grads), epn, n, M, H, Hp, G, s), "mep_ffn_backward")
                torch.cuda.synchronize()
        finally:
            lib.mep_set_gemm_row_tile(0)
        seen = sum(e.count for e in prof.key_averages() if "gemm_stream_kernel" in e.key)
        assert seen == (2 if streaming == (tile == 0) else 0)
        drows.append(out)
    assert torch.equal(*drows) and drows[0].any()
