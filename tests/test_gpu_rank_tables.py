"""Sums and copies of several ranks' slots where the table is large: more than one list of ranks (and a
last one of fewer), more entries than a wave has lanes, experts in many slots, experts of less than a
tile, so that a workgroup's next tile lies several experts on."""

import ctypes as C

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu


def _table(R, epn, used, g):
    """Every rank's occupied slots, of which an eighth hold one of three experts."""
    etc = torch.full((R, epn), -1, dtype=torch.int32)
    take = torch.rand(R, epn, generator=g) < used
    experts = torch.randint(0, R * epn, (R, epn), generator=g, dtype=torch.int32)
    few = torch.rand(R, epn, generator=g) < 0.125
    return torch.where(take, torch.where(few, experts % 3 * (R * epn // 3), experts), etc)


@pytest.mark.parametrize("R,epn,rank0,nranks", [(64, 48, 0, 64),   # two lists
                                                (64, 48, 3, 41),   # two lists of 21 and 20 ranks
                                                (16, 48, 0, 16),
                                                (3, 67, 1, 2),
                                                (64, 48, 5, 1)])
@pytest.mark.parametrize("used", [0.02, 1.0])
def test_sums(cuda, R, epn, rank0, nranks, used):
    print(f"sums of ranks {rank0} + {nranks} of {R}, {epn} experts, {used} of the slots", flush=True)
    g = torch.Generator().manual_seed(R + epn + nranks)
    etc = _table(R, epn, used, g)
    elems = (64, 4100, 8192)       # less than a tile, a tile and a rest, two tiles
    own = [torch.randn(nranks, epn, n, generator=g) for n in elems]
    pool = [torch.randn(R, epn, n, generator=g) for n in elems]
    want = [t.clone() for t in own]
    for d, b in (etc >= 0).nonzero().tolist():      # slots are added in ascending order, in fp32
        r, le = divmod(int(etc[d, b]), epn)
        if rank0 <= r < rank0 + nranks:
            for w, p in zip(want, pool):
                w[r - rank0, le] += p[d, b]
    etc, got, slots = etc.to(cuda), [t.to(cuda) for t in own], [t.to(cuda) for t in pool]
    arr_p, arr_i = C.c_void_p * 3, C.c_int64 * 3
    rc = _lib.lib().mep_grad_reduce_batch(3, arr_p(*[t.data_ptr() for t in got]), arr_p(*[t.data_ptr() for t in slots]),
                                          arr_i(*[epn * n for n in elems]), arr_i(*elems), etc.data_ptr(), rank0, nranks,
                                          epn, R, _lib.REDUCE_NO_CLEAR, _lib.current_stream())
    _lib.check(rc, "mep_grad_reduce_batch")
    torch.cuda.synchronize()
    for a, b, c, d in zip(got, want, slots, pool):
        assert torch.equal(a.cpu(), b) and torch.equal(c.cpu(), d)


@pytest.mark.parametrize("R,epn,rank0,nranks", [(64, 48, 0, 64), (64, 48, 3, 41), (16, 48, 0, 16), (3, 67, 1, 2),
                                                (16, 17, 0, 16)])
@pytest.mark.parametrize("used", [0.0, 0.02, 1.0])
def test_copies(cuda, R, epn, rank0, nranks, used):
    print(f"slots of ranks {rank0} + {nranks} of {R}, {epn} experts, {used} of them", flush=True)
    g = torch.Generator().manual_seed(R + epn + nranks)
    etc = _table(R, epn, used, g)
    nbytes = 1040
    local = torch.randint(0, 256, (R * epn, nbytes), dtype=torch.uint8, generator=g)
    want = torch.randint(0, 256, (R, epn, nbytes), dtype=torch.uint8, generator=g)
    src, got = local.to(cuda), want.to(cuda)
    there = etc >= 0
    there[:rank0] = False
    there[rank0 + nranks:] = False
    want[there] = local[etc[there].long()]
    etc = etc.to(cuda)
    arr_p, arr_i = C.c_void_p * 1, C.c_int64 * 1
    stride = arr_i(epn * nbytes)
    rc = _lib.lib().mep_prefetch_pull_ranks(1, arr_p(src.data_ptr()), stride, arr_p(got.data_ptr()), stride, arr_i(nbytes),
                                            etc.data_ptr(), rank0, nranks, epn, R, _lib.current_stream())
    _lib.check(rc, "mep_prefetch_pull_ranks")
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), want)
