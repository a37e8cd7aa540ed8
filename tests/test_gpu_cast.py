"""fp32 -> bf16 of several tensors' blocks (mep_cast_bf16): the bits of torch's conversion, for blocks
shorter than, equal to and longer than a span of 128 KiB, and nothing written between the blocks."""

import ctypes as C

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nranks,elems", [(1, (8,)), (3, (32768, 32776, 24)), (2, (5 * 32768 - 8, 4096)), (8, (3 * 32768 + 2048,) * 6)])
def test_cast(cuda, nranks, elems):
    print(f"cast nranks={nranks} elems={elems}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nranks + elems[0])
    src = [torch.randn(nranks, n, device=cuda, generator=g) for n in elems]
    for s in src:      # ties, a denormal, the ends of the range
        s[:, :8] = torch.tensor([1 + 2.0**-8, 1 + 3 * 2.0**-8, -1 - 2.0**-8, 1e-40, float("inf"), -float("inf"), 3.4e38, 0.0],
                                device=cuda)
        s[-1, -1] = float("nan")
    dst = [torch.full((nranks, 2 * n), 7.0, dtype=torch.bfloat16, device=cuda) for n in elems]
    k = len(elems)
    _lib.check(_lib.lib().mep_cast_bf16(k, (C.c_void_p * k)(*[t.data_ptr() for t in src]), (C.c_void_p * k)(*[t.data_ptr() for t in dst]),
                                        (C.c_int64 * k)(*elems), (C.c_int64 * k)(*[2 * n for n in elems]), nranks,
                                        _lib.current_stream()), "mep_cast_bf16")
    for s, d, n in zip(src, dst, elems):
        want = s.bfloat16()
        num = ~want.isnan()
        assert torch.equal(d[:, :n][num].view(torch.int16), want[num].view(torch.int16))
        assert d[-1, n - 1].isnan() and bool((d[:, n:] == 7.0).all())
