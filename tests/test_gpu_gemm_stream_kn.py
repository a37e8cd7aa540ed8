"""Streaming kernel for weights given as [K, N]: every width of a tile, K shorter than its ring of LDS
stages, blocks that share a group, groups without rows, both pairs.  K goes up in every kernel, so the
result is that of the 256 x 256 kernels to the bit."""

import pytest
import torch

from moonep_amd import _lib, ffn

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def any_row_tile():
    yield
    _lib.check(_lib.lib().mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")


# blocks, groups, N, K: tiles of 1; 2; 3; 4 units; two rounds of 2 and 3; one K step, more than the ring
@pytest.mark.parametrize("blocks,G,N,K", [(1, 2, 256, 64), (64, 9, 512, 128), (64, 65, 768, 192), (85, 40, 768, 320),
                                          (90, 12, 768, 64), (3, 8, 2816, 640)])
def test_bits_of_the_256_kernels(cuda, blocks, G, N, K):
    print(f"stream kn {blocks} blocks, {G} groups, {N} x {K}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(blocks + G + N + K)
    cuts = torch.randint(0, blocks + 1, (G - 1,), generator=g, device=cuda).sort().values
    ends = (torch.cat([cuts, torch.tensor([blocks], device=cuda)]) * 128).to(torch.int32)
    M = 128 * (blocks + 1)
    a1, a2 = (torch.randn(M, K, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
    w1, w2 = ((torch.randn(G, K, N, generator=g, device=cuda) / K ** 0.5).to(torch.bfloat16) for _ in range(2))
    scale = torch.rand(M, generator=g, device=cuda) + 0.5
    out = []
    for tile in (128, 256):
        _lib.check(_lib.lib().mep_set_gemm_row_tile(tile), "mep_set_gemm_row_tile")
        plain, scaled = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(2))
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            ffn.launch_grouped_gemm_nn(a1, w1, ends, out=plain)
            ffn.launch_grouped_gemm_nn(a1, w1, ends, out=scaled, row_scale=scale)
            out.append((plain, scaled, ffn.launch_grouped_gemm_dual_nn(a1, w1, a2, w2, ends)))
            torch.cuda.synchronize()
        assert sum(e.count for e in prof.key_averages() if "gemm_stream_kernel" in e.key) == (3 if tile == 128 else 0)
    for what, x, y in zip(("plain", "scaled", "both pairs"), *out):
        assert torch.equal(x, y), what
    assert bool(out[0][0][:128 * blocks].any()) and not bool(out[0][2][128 * blocks:].any())
    assert all(bool((x[128 * blocks:] == 7.0).all()) for x in out[0][:2])   # rows behind the last group
