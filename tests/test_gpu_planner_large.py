"""The planner with more than 64 KB of tables: those that fill a CU's LDS and those just beyond it, the only ones
that callers bring scratch for."""

import numpy as np
import pytest
import torch

from moonep_amd import Buffer, _lib, routing
from moonep_amd.planning import launch_planning_all_ranks
from tests.util import oracle_world_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,K,E,R,tp", [
    (700, 8, 512, 16, 128),    # 90 KB, several workgroups a rank
    (300, 8, 768, 16, 64),     # 133 KB
    (150, 6, 624, 8, 16),      # 68 KB
    (140, 8, 1528, 8, 16),     # the most that 160 KB hold at eight ranks ...
    (140, 8, 1536, 8, 16),     # ... in scratch
    (60, 3, 576, 24, 32),      # ranks and top-k that no variant is compiled for
    (33, 1, 1100, 4, 8),
])
def test_large_tables_match_the_oracle(cuda, S, K, E, R, tp):
    print(f"planner S={S} K={K} E={E} R={R}", flush=True)
    topk = torch.stack([routing.popularity_biased(S, K, E, R, r, 0.7, seed=5) for r in range(R)])
    tpe = routing.tokens_per_expert(topk, E)
    gp, plans, dst = oracle_world_plan(topk.numpy(), tpe.numpy(), tp)
    tables = 4 * ((6 + 4) * E + 6 * R + 1024 + 2 * E * R)
    want = 0 if tables <= 163840 else -(-S // (256 // K)) * 2 * E * R * 4
    assert _lib.lib().mep_plan_scratch_bytes(S, K, E, R, 1) == want
    buf = Buffer(S, 16, K, E, R, token_padding=tp, rank=0)
    dst_all, cu, etc, zfr, stats = launch_planning_all_ranks(buf._require_ctx(), topk.to(cuda), tpe.to(cuda))
    torch.cuda.synchronize()
    assert np.array_equal(dst_all.cpu().numpy(), dst)
    assert np.array_equal(cu.cpu().numpy(), gp.cu_seqlens)
    assert np.array_equal(etc.cpu().numpy(), gp.experts_to_copy)
    assert np.array_equal(zfr.cpu().numpy(), gp.zero_fill)
    assert np.array_equal(stats.cpu().numpy(), gp.remote_stats)
    buf.destroy()
