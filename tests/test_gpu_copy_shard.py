"""mep_copy_shard (a shard staged out of or into the communication buffers) is a byte copy:
exact, at the edges of its tile layout, with nothing written beyond either range."""

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu

BLOCK = 128 * 1024      # eight interleaved tiles; what is left is covered by tiles of 16 KiB


@pytest.mark.parametrize("nbytes,words", [
    (16, 0), (0, 1), (16, 1), (16 * 1024, 257), (16 * 1024 + 16, 3), (BLOCK, 0), (BLOCK - 16, 1000),
    (BLOCK + 16, 5), (5 * BLOCK + 3 * 16 * 1024 + 48, 4096), (600 * BLOCK, 70001)])
def test_copies_both_ranges_and_nothing_else(cuda, nbytes, words):
    print(f"copy_shard bytes={nbytes} words={words}", flush=True)
    pad = 4096
    src = torch.randint(0, 256, (nbytes + pad,), dtype=torch.uint8, device=cuda)
    src_w = torch.randint(-2**31, 2**31 - 1, (words + pad,), dtype=torch.int32, device=cuda)
    dst, dst_w = torch.full_like(src, 7), torch.full_like(src_w, 7)
    rc = _lib.lib().mep_copy_shard(dst.data_ptr(), src.data_ptr(), nbytes, dst_w.data_ptr(), src_w.data_ptr(), words,
                                   _lib.current_stream())
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(dst[:nbytes], src[:nbytes]) and bool((dst[nbytes:] == 7).all())
    assert torch.equal(dst_w[:words], src_w[:words]) and bool((dst_w[words:] == 7).all())
