"""The weight gradients' list of tiles: which groups have rows, which come out as zeros and which are left alone.  Beside
more groups than one wave looks at, of one round, where all groups stay in their places, and of several, and
beside more groups than there are tables for."""

import pytest
import torch

from moonep_amd import ffn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("full", ["few", "half", "all", "last"])
@pytest.mark.parametrize("G", [64, 66, 130, 1030])
def test_groups_with_and_without_rows(cuda, G, full):
    check(cuda, G, full, 512, 256)


@pytest.mark.parametrize("full", ["few", "half", "all", "last"])
@pytest.mark.parametrize("G,M,N", [(32, 1024, 512), (34, 1024, 512), (64, 512, 1024), (66, 1024, 512), (256, 256, 256), (258, 256, 256),
                                   (30, 1280, 512), (34, 768, 768), (66, 256, 1280)])    # numbers of tiles that eight does not divide
def test_both_sides_of_one_round(cuda, G, M, N, full):
    check(cuda, G, full, M, N)


def check(cuda, G, full, M, N):
    """Against the fp64 product: a sum of n products in fp32, in any order, is off by at most n 2^-24 of the
    sum of their magnitudes."""
    print(f"wgrad list, {G} groups of {M} x {N}, rows in {full}", flush=True)
    g = torch.Generator().manual_seed(G)
    share = {"few": 0.05, "half": 0.5, "all": 1.0, "last": 0.0}[full]
    lens = ((torch.rand(G, generator=g) < share) * torch.randint(1, 3, (G,), generator=g)).tolist()
    lens[-1] = 1
    ends = (torch.tensor(lens).cumsum(0) * 128).to(torch.int32).to(cuda)
    rows = 128 * (sum(lens) + 1)
    gc = torch.Generator(device=cuda).manual_seed(G)
    x1, x2 = (torch.randn(rows, n, generator=gc, device=cuda).to(torch.bfloat16) for n in (M, N))
    got = torch.full((G, M, N), float("nan"), device=cuda)
    kept = got.clone()
    ffn.launch_grouped_gemm_wgrad_tn(x1, x2, ends, got)
    ffn.launch_grouped_gemm_wgrad_tn(x1, x2, ends, kept, skip_empty_from=G // 3)
    torch.cuda.synchronize()
    at = 0
    for i, n in enumerate(lens):
        if n:
            a, b = (x[128 * at:128 * (at + n)].double() for x in (x1, x2))
            assert bool(((got[i].double() - a.t() @ b).abs() <= 128 * n * 2.0 ** -24 * (a.abs().t() @ b.abs())).all()), f"group {i}"
            at += n
    empty = torch.tensor(lens, device=cuda) == 0
    kept_alone = empty & (torch.arange(G, device=cuda) >= G // 3)
    assert bool((got[empty] == 0).all())
    assert torch.equal(kept[~kept_alone], got[~kept_alone])
    assert bool(kept[kept_alone].isnan().all())


@pytest.mark.parametrize("skip", [False, True])
def test_more_groups_than_the_tables_hold(cuda, skip):
    """262146 groups, five with rows: 69 GB of gradients, in which the others come out as zeros or are not touched."""
    G, full = 262146, (0, 1, 70_000, 262_143, 262_145)
    if torch.cuda.mem_get_info()[0] < 90 << 30:
        pytest.skip("needs 69 GB")
    print(f"wgrad list, {G} groups, skip={skip}", flush=True)
    lens = torch.zeros(G, dtype=torch.int32)
    lens[list(full)] = 128
    ends = lens.cumsum(0).to(torch.int32).to(cuda)
    g = torch.Generator(device=cuda).manual_seed(2)
    x1, x2 = (torch.randn(128 * len(full), 256, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
    out = torch.full((G, 256, 256), 3.0, device=cuda)
    ffn.launch_grouped_gemm_wgrad_tn(x1, x2, ends, out, skip_empty_from=0 if skip else None)
    torch.cuda.synchronize()
    for at, i in enumerate(full):
        a, b = (x[128 * at:128 * (at + 1)].double() for x in (x1, x2))
        assert bool(((out[i].double() - a.t() @ b).abs() <= 2.0 ** -17 * (a.abs().t() @ b.abs())).all()), f"group {i}"
        out[i].fill_(3.0 if skip else 0.0)
    low, high = torch.aminmax(out)
    assert float(low) == float(high) == (3.0 if skip else 0.0)
    del out
    torch.cuda.empty_cache()
