"""Combine of few tokens (all rows of a token asked for at once) against the oracle and against the
kernel for many tokens: the same tokens as part of a call that is too large for the first."""

import pytest
import torch

from moonep_amd import _lib
from oracle import ops_oracle as oo

pytestmark = pytest.mark.gpu


def _call(shards, wslots, dst, S, H, K):
    R, NvS, _ = shards.shape
    out = torch.full((S, H), 3.0, dtype=torch.bfloat16, device="cuda")
    w = torch.full((S, K), 5.0, device="cuda")
    _lib.check(_lib.lib().mep_combine(shards.data_ptr(), NvS, wslots.data_ptr(), NvS, dst.data_ptr(), out.data_ptr(),
                                      w.data_ptr(), S, H, K, R, NvS, _lib.COMBINE_TWO_LEVEL, _lib.current_stream()), "mep_combine")
    return out.cpu().view(torch.int16), w.cpu().view(torch.int32)


# K on both sides of each unrolled length, rows of one vector, just under, at and past whole pieces
@pytest.mark.parametrize("S,H,K,R", [(1, 8, 1, 2), (3, 504, 2, 4), (5, 512, 4, 8), (7, 520, 5, 4), (8, 4096, 8, 8),
                                     (33, 2880, 6, 4), (6, 1032, 7, 3), (4, 1024, 9, 8)])
@pytest.mark.parametrize("skipped", [False, True])
def test_few_tokens(cuda, S, H, K, R, skipped):
    g = torch.Generator().manual_seed(S * 131 + H + K)
    NvS = 64
    large = 6144 // ((H + 511) // 512) + 1 + S     # one token more than the rule for few tokens takes
    shards = torch.randn(R, NvS, H, generator=g).to(torch.bfloat16)
    shards[0, 3] = float("inf")
    shards[0, 5, ::3] = float("nan")
    wslots = torch.randn(R, NvS, generator=g)
    ranks = torch.randint(0, R, (large, K), generator=g)
    raw = ranks * NvS + torch.randint(0, NvS, (large, K), generator=g)
    first = torch.ones(large, K, dtype=torch.bool)
    for k in range(1, K):
        first[:, k] = (ranks[:, :k] != ranks[:, k:k + 1]).all(1)
    if skipped:     # what the planner makes of an invalid expert id
        gone = torch.rand(large, K, generator=g) < 0.3
        raw[gone] = R * NvS
    dst = torch.where(first, raw, -raw - 1).to(torch.int32).contiguous()
    print(f"S={S} H={H} K={K} R={R} skipped={skipped}", flush=True)
    dev = shards.cuda(), wslots.cuda()
    few = _call(*dev, dst[:S].contiguous().cuda(), S, H, K)
    many = _call(*dev, dst.cuda(), large, H, K)
    assert torch.equal(few[0], many[0][:S]) and torch.equal(few[1], many[1][:S])
    if not skipped:
        want, w = oo.combine(shards, wslots, dst[:S].reshape(-1), K, mode="two_level")
        nan = want.isnan()
        assert torch.equal(few[0][~nan], want.view(torch.int16)[~nan])
        assert few[0].view(torch.bfloat16)[nan].isnan().all()
        assert torch.equal(few[1].view(-1), w.reshape(-1).view(torch.int32))
