"""A call captured in the scratch that a larger eager call left on its stream
takes the split ranges that fit there, and gives the eager call's results."""
import pytest

from tests.gpu_util import TOL_BF16, TOL_F32, announce, host, need_gpu, rel_l2

pytestmark = pytest.mark.gpu

H = 4


def _decode(torch, bd, g, B, T, N, D):
    x = (torch.randn(B, H, N, generator=g, device="cuda") - 1.645).relu_()
    v = torch.randn(B, 1, D, generator=g, device="cuda")
    rho = torch.randn(B, H, N, D, generator=g, device="cuda")
    work = rho.clone()

    def call():
        work.copy_(rho)
        return bd.decode_step(x, v, work, position=9).readout, work
    return call


def _prefill(torch, bd, g, B, T, N, D):
    x = (torch.randn(B, H, T, N, generator=g, device="cuda", dtype=torch.bfloat16) - 1.645).relu_()
    v = torch.randn(B, 1, T, D, generator=g, device="cuda", dtype=torch.bfloat16)

    def call():
        out = bd.try_fused_recurrent_attention_rope(x, v, position=9)
        return out.context, out.rho
    return call


def _layer(torch, bd, g, B, T, N, D):
    w = bd.LowRankWeights.pack(torch.randn(1, H, D, N, generator=g, device="cuda") * 0.02,
                               torch.randn(1, H, D, N, generator=g, device="cuda") * 0.02,
                               torch.randn(H * N, D, generator=g, device="cuda") * 0.02)
    cur = torch.nn.functional.layer_norm(torch.randn(B, T, D, generator=g, device="cuda"), (D,))
    return lambda: (bd.lowrank_layer_forward(cur, w, position=9).next,)


def _vjp(torch, bd, g, B, T, N, D):
    x = (torch.randn(B, H, T, N, generator=g, device="cuda") - 1.645).relu_()
    v = torch.randn(B, 1, T, D, generator=g, device="cuda")
    go = torch.randn(B, H, T, D, generator=g, device="cuda")
    decay = torch.tensor([0.999, 0.99, 0.98, 0.97], device="cuda")

    def call():
        out = bd.dense_causal_attention_vjp(go, x, v, decay)
        return out.grad_query, out.grad_value, out.grad_decay
    return call


@pytest.mark.parametrize("make,N,D,big,small,tol", [
    (_decode, 8192, 64, (10, 1), (2, 1), TOL_F32),             # 40 streams of 4 ranges; 8 of 32
    (_prefill, 4096, 64, (9, 256), (4, 256), TOL_BF16),        # 36 streams of 2 gram ranges; 16 of 8
    (_prefill, 8192, 64, (6, 1024), (4, 1024), TOL_BF16),      # state-carry form: 240 tiles unsplit; 160 in 3 ranges
    (_layer, 8192, 64, (6, 1024), (4, 1024), TOL_BF16),        # the layer's gram: likewise
    (_layer, 8192, 64, (16, 17), (1, 255), TOL_BF16),          # decoder apart in 16 ranges; Y + decoder in 64
    (_vjp, 2048, 32, (12, 512), (8, 384), TOL_F32),            # 128-tiles unsplit; 64-tiles' sums, 2 ranges
])
def test_captured_in_a_larger_calls_scratch(make, N, D, big, small, tol):
    torch = need_gpu()
    import burn_dragon_amd as bd
    announce("captured in a larger call's scratch", make.__name__, N, D, big, small)
    g = torch.Generator(device="cuda").manual_seed(N + D)
    call = make(torch, bd, g, *small, N, D)
    want = [host(t) for t in call()]
    larger = make(torch, bd, g, *big, N, D)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        larger()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        out = call()
    for _ in range(3):
        for t in out:
            t.zero_()
        call()
        graph.replay()
        torch.cuda.synchronize()
        for t, w in zip(out, want):
            assert rel_l2(host(t), w) <= tol
    del graph
    bd.release_stream_scratch(st)


def test_backward_without_room_for_partials():
    # The gram's three ranges take 0.4 GB of partials: with less than that left
    # on the device it runs unsplit.
    torch = need_gpu()
    import burn_dragon_amd as bd
    announce("backward, memory short")
    B, T, N, D = 8, 1024, 4096, 64
    call = _vjp(torch, bd, torch.Generator(device="cuda").manual_seed(3), B, T, N, D)
    want = call()
    torch.cuda.synchronize()
    bd.release_stream_scratch()
    torch.cuda.empty_cache()
    S = B * H
    need = 4 * S * (2 * T * T + 4 * T * D)  # scores, their gradient's sums, four [T, D] buffers
    need += need // 4 + sum(t.numel() * 4 for t in want) + (200 << 20)
    hold = []
    try:
        free = torch.cuda.mem_get_info()[0]
        while free > need + (40 << 20):
            hold.append(torch.empty(min(free - need, 32 << 30), dtype=torch.uint8, device="cuda"))
            free = torch.cuda.mem_get_info()[0]
        assert free - need + (200 << 20) < 300 << 20  # less than the partials take
        out = call()
        torch.cuda.synchronize()
    finally:
        del hold
        bd.release_stream_scratch()
        torch.cuda.empty_cache()
    for t, w in zip(out, want):
        assert rel_l2(host(t), host(w)) <= TOL_F32
