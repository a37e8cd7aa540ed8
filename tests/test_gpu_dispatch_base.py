"""Shards that begin anywhere at which 16 bytes may begin: rows are written from the 128-byte line that holds their
first byte on, which depends on the base as much as on the row's length.  Every byte of the shards, of what lies
between the ranks' and of a margin on both sides against an index copy (nothing is rounded)."""

import pytest
import torch

from moonep_amd import _lib
from oracle import ops_oracle as oo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("base", [0, 16, 64, 112])
# 16 bytes to four whole pieces of 4 KB; both sides of what a row takes in one and in two KB from a line's beginning on
@pytest.mark.parametrize("H", [8, 448, 456, 464, 520, 960, 968, 976, 1024, 2048, 2880, 4096, 4104, 6144, 8192])
@pytest.mark.parametrize("one_launch", [False, True])
def test_every_byte_of_the_shards(cuda, H, base, one_launch):
    S, K, E, R, rank, tp = 21, 3, 8, 2, 1, 16
    print(f"H={H} base={base} one_launch={one_launch}", flush=True)
    epn = E // R
    NvS = -(-(S * K + (tp - 1) * 2 * epn) // tp) * tp
    stride, margin = NvS + 3, 256
    g = torch.Generator(device="cuda").manual_seed(H + base)
    topk = torch.topk(torch.randn(R, S, E, device=cuda, generator=g), K, dim=-1)[1].to(torch.int32)
    counts = torch.zeros(R, E, dtype=torch.int32, device=cuda)
    counts.scatter_add_(1, topk.reshape(R, -1).long(), torch.ones(R, S * K, dtype=torch.int32, device=cuda))
    mine = topk[rank].contiguous()
    x = torch.randint(-2**15, 2**15, (S, H), device=cuda, generator=g, dtype=torch.int16)
    w = torch.rand(S, K, device=cuda, generator=g)
    ints = [torch.empty(shape, dtype=torch.int32, device=cuda)
            for shape in ((S * K,), (2 * epn,), (R, epn), (2 * epn, 2), (2,), (2,))]
    memory = torch.full((margin + R * stride * H + margin,), 77, dtype=torch.int16, device=cuda)
    shards = memory[margin // 2 + base // 2:]
    assert memory.data_ptr() % 128 == 0 and shards.data_ptr() % 128 == base
    slots = torch.full((R, NvS), 7.0, device=cuda)
    lib, p, s = _lib.lib(), _lib.ptr, _lib.current_stream()
    dst, cu, etc, zf, stats, dup = map(p, ints)
    if one_launch:
        rc = lib.mep_dispatch_fresh(p(counts), p(mine), p(x), p(w), rank, S, H, K, E, R, tp, NvS, dst, cu, etc, zf, stats, dup,
                                    p(shards), stride, p(slots), NvS, None, 0, s)
    else:
        rc = lib.mep_plan(p(counts), p(mine), rank, S, K, E, R, tp, NvS, dst, cu, etc, zf, stats, None, 0, s)
        _lib.check(rc, "mep_plan")
        rc = lib.mep_dispatch(p(x), p(w), dst, zf, p(shards), stride, p(slots), NvS, rank, S, H, K, R, epn, NvS, tp,
                              _lib.DISPATCH_WRITE_DUPS, s)
    _lib.check(rc, "dispatch")
    torch.cuda.synchronize()
    want, want_slots = torch.full_like(memory.cpu(), 77), torch.full((R, NvS), 7.0)
    rows, at = torch.full((R, NvS, H), 77, dtype=torch.int16), margin // 2 + base // 2
    oo.dispatch(x.cpu(), w.cpu(), ints[0].cpu(), ints[3].cpu(), rows, want_slots, rank, K, include_dups=True)
    want[at:at + R * stride * H].view(R, stride, H)[:, :NvS] = rows
    assert int((rows != 77).sum()) > S * H
    assert torch.equal(memory.cpu(), want) and torch.equal(slots.cpu(), want_slots)
