"""What a Buffer's calls return is an ordinary tensor outside of inference mode, also of a world made inside."""

import pytest
import torch

from moonep_amd import Buffer, EmulatedWorld

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("made_inside", [False, True])
@pytest.mark.parametrize("copy", [False, True])
def test_outputs_and_inference_mode(cuda, made_inside, copy):
    S, H, K, E, R = 5, 256, 2, 8, 2
    with torch.inference_mode(made_inside):
        world = EmulatedWorld(S, H, K, E, R, 16)
        buf = Buffer(S, H, K, E, R, token_padding=16, rank=1, world=world)
    x = torch.randn(S, H, device=cuda).to(torch.bfloat16)
    w = torch.rand(S, K, device=cuda)
    topk = torch.tensor([[0, 5], [1, 4], [2, 7], [3, 6], [4, 0]], dtype=torch.int32, device=cuda)
    counts = torch.bincount(topk.flatten(), minlength=E).to(torch.int32).repeat(R, 1)
    modes = dict(zero_copy=not copy, router_weights_zero_copy=not copy)
    outs = []
    for inside in (False, True):
        with torch.inference_mode(inside):
            rows, slots, _, plan = buf.dispatch(x, w, topk, counts, **modes)
            out, back, _ = buf.combine(plan, rows, slots, **modes)
        assert out.is_inference() == inside and back.is_inference() == inside
        assert out.is_contiguous() and out.dtype == torch.bfloat16 and tuple(out.shape) == (S, H)
        assert back.is_contiguous() and back.dtype == torch.float32 and tuple(back.shape) == (S, K)
        assert torch.equal(back, w)
        outs.append(out.clone())
    assert torch.equal(*outs)
    assert not (outs[0] == 0).all()
