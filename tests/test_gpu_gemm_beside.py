"""The 256 x 256 GEMM kernel as several workgroups per CU: lists of tiles that are no multiple of what
the workgroups take, and its time beside a kernel that holds 32 of the compute units (what
``Buffer(num_sms=32)`` does to it).

Tolerance of the products: bf16 operands, fp32 sums, one rounding to bf16 (2^-9 relative): 5e-3 in
the 2-norm; the weight gradients stay in fp32: sums of n products in another order, 1e-5."""

import ctypes

import pytest
import torch

from moonep_amd import _lib

pytestmark = pytest.mark.gpu


def _ends(heights, cuda):
    return torch.tensor([128 * sum(heights[:i + 1]) for i in range(len(heights))], dtype=torch.int32, device=cuda)


# K steps of a tile: three tiles, one and one to a workgroup; row tiles of 256, short last ones, empty groups
@pytest.mark.parametrize("K", [43 * 64, 128 * 64, 200 * 64])
@pytest.mark.parametrize("heights", [(7, 0, 12, 1, 30, 3), (64,), (1,) * 40])
def test_row_tiles_over_several_workgroups(cuda, K, heights):
    N, G, M = 2304, len(heights), 128 * (sum(heights) + 1)
    print(f"K={K} heights={heights}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randn(M, K, device=cuda, generator=g).to(torch.bfloat16)
    B = torch.randn(G, N, K, device=cuda, generator=g).to(torch.bfloat16) * K ** -0.5
    scale = torch.rand(M, device=cuda, generator=g) + 0.1
    ends = _ends(heights, cuda)
    C = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=cuda)
    lib = _lib.lib()
    _lib.check(lib.mep_set_gemm_row_tile(256), "mep_set_gemm_row_tile")
    try:
        rc = lib.mep_grouped_gemm_nt(A.data_ptr(), B.data_ptr(), None, ends.data_ptr(), G, C.data_ptr(), scale.data_ptr(),
                                     M, N, K, 0, _lib.current_stream())
    finally:
        _lib.check(lib.mep_set_gemm_row_tile(0), "mep_set_gemm_row_tile")
    _lib.check(rc, "mep_grouped_gemm_nt")
    assert (C[int(ends[-1]):] == 7.0).all()
    beg = 0
    for i, end in enumerate(ends.tolist()):
        if end > beg:
            want = (A[beg:end].float() @ B[i].float().t()) * scale[beg:end, None]
            # row blocks on their own: a tile that was left out or taken twice shows
            for b in range(0, end - beg, 128):
                d = C[beg + b:beg + b + 128].float() - want[b:b + 128]
                assert float(d.norm() / want[b:b + 128].norm()) < 5e-3, (i, b)
        beg = end


@pytest.mark.parametrize("heights", [(40, 0, 3, 21, 1, 0), (2,) * 48])
def test_weight_gradient_over_several_workgroups(cuda, heights):
    Ma, Nb, G, M = 2048, 1792, len(heights), 128 * sum(heights)
    print(f"wgrad heights={heights}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(G)
    x1 = torch.randn(M, Ma, device=cuda, generator=g).to(torch.bfloat16)
    x2 = torch.randn(M, Nb, device=cuda, generator=g).to(torch.bfloat16)
    ends = _ends(heights, cuda)
    C = torch.full((G, Ma, Nb), 7.0, device=cuda)
    _lib.check(_lib.lib().mep_grouped_gemm_wgrad_tn(x1.data_ptr(), x2.data_ptr(), ends.data_ptr(), G, C.data_ptr(), Ma, Nb, M,
                                                    G // 2, _lib.current_stream()), "mep_grouped_gemm_wgrad_tn")
    beg = 0
    for i, end in enumerate(ends.tolist()):
        if end == beg:
            assert (C[i] == (7.0 if i >= G // 2 else 0.0)).all()
            continue
        want = x1[beg:end].double().t() @ x2[beg:end].double()
        d = (C[i] - want).view(Ma // 256, 256, Nb // 256, 256).square().sum((1, 3)).sqrt()
        n = want.view(Ma // 256, 256, Nb // 256, 256).square().sum((1, 3)).sqrt()
        assert float((d / n).max()) < 1e-5, i
        beg = end


@pytest.mark.parametrize("kind", ["forward", "weight gradient"])
def test_beside_a_kernel_that_holds_32_cus(cuda, kind):
    """224 of 256 CUs do the product in 8/7 of its time, a workgroup's share more or less; with one
    share of the tiles per CU the last 32 shares wait for the others: twice the time."""
    lib = _lib.lib()
    M, N, K, G = 32768, 4096, 4096, 16
    g = torch.Generator(device="cuda").manual_seed(1)
    A = torch.randn(M, K, device=cuda, generator=g).to(torch.bfloat16)
    ends = _ends((M // G // 128,) * G, cuda)
    if kind == "forward":
        B = torch.randn(G, N, K, device=cuda, generator=g).to(torch.bfloat16)
        C = torch.empty(M, N, dtype=torch.bfloat16, device=cuda)

        def product():
            _lib.check(lib.mep_grouped_gemm_nt(A.data_ptr(), B.data_ptr(), None, ends.data_ptr(), G, C.data_ptr(), None, M, N, K,
                                               0, _lib.current_stream()), "mep_grouped_gemm_nt")
    else:
        B = torch.randn(M, N // 2, device=cuda, generator=g).to(torch.bfloat16)
        C = torch.empty(G, K, N // 2, device=cuda)

        def product():
            _lib.check(lib.mep_grouped_gemm_wgrad_tn(A.data_ptr(), B.data_ptr(), ends.data_ptr(), G, C.data_ptr(), K, N // 2, M, G,
                                                     _lib.current_stream()), "mep_grouped_gemm_wgrad_tn")
    # one combine of many tokens: some 5 ms on 32 CUs
    S, H, R, NvS = 65536, 7168, 4, 8192
    shards = torch.randn(R, NvS, H, device=cuda, generator=g).to(torch.bfloat16)
    dst = torch.randint(0, R * NvS, (S * 8,), device=cuda, generator=g, dtype=torch.int32)
    out = torch.empty(S, H, dtype=torch.bfloat16, device=cuda)
    handle = ctypes.c_void_p()
    _lib.check(lib.mep_stream_create_limited(32, ctypes.byref(handle)), "mep_stream_create_limited")
    held = torch.cuda.ExternalStream(handle.value)
    times = {False: [], True: []}
    results = []
    try:
        # on streams of their own: a CU-masked stream waits for the null stream's work and the reverse.
        # Several, because some pairs of hardware queues take turns instead of running beside each
        # other (2.4 to 2.8 times the product's time, however its tiles are shared out).
        for main in [torch.cuda.Stream() for _ in range(6)]:
            with torch.cuda.stream(main):
                for beside in (False, True, True):
                    torch.cuda.synchronize()
                    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                    done = torch.cuda.Event()
                    if beside:
                        _lib.check(lib.mep_combine(shards.data_ptr(), NvS, None, 0, dst.data_ptr(), out.data_ptr(), None, S, H, 8,
                                                   R, NvS, _lib.COMBINE_TWO_LEVEL, handle.value), "mep_combine")
                        done.record(held)
                        torch.cuda._sleep(2_400_000)    # a millisecond: it has started
                    a.record()
                    product()
                    b.record()
                    b.synchronize()
                    if not (beside and done.query()):   # the product was alone at its end otherwise
                        times[beside].append(a.elapsed_time(b))
                    if len(results) < 2:
                        results.append(C.clone())
        torch.cuda.synchronize()
    finally:
        torch.cuda.synchronize()
        lib.mep_stream_destroy(handle)
    print(f"{kind}: " + " ".join(f"{t * 1e3:.0f}" for t in times[True]), flush=True)
    assert len(times[True]) >= 4, "the held CUs were free before the product ended"
    alone, beside = min(times[False][1:]), min(times[True])
    print(f"{kind}: {alone * 1e3:.0f} us alone, {beside * 1e3:.0f} us beside", flush=True)
    assert torch.equal(*results)
    assert beside < 1.4 * alone
