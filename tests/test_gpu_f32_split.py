"""The fp32 path's products run as six bf16 part products each
(bdh_gemm_f32.h): tile, k-step and split edges of the forward and the
backward against the f64 oracle, and values that have no bf16 parts."""
import numpy as np
import pytest

from tests.gpu_util import announce, dev, host, need_gpu, rel_l2

pytestmark = pytest.mark.gpu

# A product rounds once per 16-deep step in each of two accumulators, and the
# products left out are below 2^-24: 64 bits away by at most about
# sqrt(K / 16) 2^-24 of the terms' norm, under 1.4e-6 for K <= 8192 and as
# much again for the chained products.
TOL = 3e-6


@pytest.mark.parametrize("B,H,Hv,T,N,D,rho,decay", [
    (1, 1, 1, 2, 2, 1, True, None),                # one partial k step, one column
    (1, 2, 1, 17, 14, 7, True, [0.9, 1.1]),        # k tail, rows not 16-byte aligned
    (2, 1, 1, 64, 30, 65, False, None),            # whole and ragged 64-row tiles
    (1, 2, 2, 129, 48, 129, True, [0.99, 0.98]),   # one row and column past a 128 tile
    (1, 1, 1, 257, 1026, 33, False, None),         # masked blocks, split k with a ragged range
    (16, 4, 1, 160, 64, 200, True, None),          # 128 tiles (over one a CU), ragged in both
    (1, 1, 1, 1030, 36, 12, True, [0.999]),        # the backward's second interval, three of the forward
    (2, 2, 1, 513, 130, 70, True, [0.99, 0.999]),  # two state intervals, the last short
    (16, 1, 1, 700, 1030, 72, False, None),        # two intervals, 128-row tiles, split k over both
    (1, 2, 1, 1030, 6, 1, True, [0.99, 0.9]),      # three intervals, one column: both strides of an operand are 1
    (2, 1, 1, 1030, 1, 3, True, None),             # three intervals, one row of the state
])
def test_edges_match_oracle(oracle, B, H, Hv, T, N, D, rho, decay):
    torch = need_gpu()
    import burn_dragon_amd as bd
    rng = np.random.default_rng(T * 31 + N)
    q = rng.standard_normal((B, H, T, N)).astype(np.float32)
    v = (rng.standard_normal((B, Hv, T, D)) / 16).astype(np.float32)
    r0 = (rng.standard_normal((B, H, N, D)) * 0.2).astype(np.float32) if rho else None
    d = np.asarray(decay, np.float32) if decay else None
    g = rng.standard_normal((B, H, T, D)).astype(np.float32)
    announce("f32 split edges", B, H, Hv, T, N, D, rho, decay)
    tq, tv, tg = dev(torch, q), dev(torch, v), dev(torch, g)
    tr, td = dev(torch, r0) if rho else None, dev(torch, d) if decay else None
    out = bd.try_fused_recurrent_attention(tq, tv, tr, td)
    grads = bd.recurrent_attention_vjp(tg, tq, tv, tr, td)
    torch.cuda.synchronize()
    ctx, rho1 = oracle.recurrent_f64(q, v, r0, d)
    assert rel_l2(host(out.context), ctx) <= TOL
    assert rel_l2(host(out.rho), rho1) <= TOL
    ref = oracle.attention_vjp_f64(q, v, g, d, r0, safe="recurrent")
    assert rel_l2(host(grads.grad_query), ref[0]) <= TOL
    assert rel_l2(host(grads.grad_value), ref[1]) <= TOL
    if rho:
        assert rel_l2(host(grads.grad_rho), ref[3]) <= TOL
    # The decay's gradient is one sum whose terms cancel: its error is held to
    # the terms' sizes (those of the whole sequence, no state).
    t = np.arange(T)
    gap = np.maximum(t[:, None] - t[None, :], 0)
    dd = np.ones(H) if d is None else d.astype(np.float64)
    size = np.abs((g @ np.broadcast_to(v, (B, H, T, D)).swapaxes(2, 3)) * (q @ q.swapaxes(2, 3)) * gap
                  * dd[:, None, None] ** np.maximum(gap - 1, 0)).sum((0, 2, 3))
    if rho:
        size += np.abs(g * (q @ r0) * t[:, None] * dd[:, None, None] ** np.maximum(t - 1, 0)[:, None]).sum((0, 2, 3))
    assert (np.abs(host(grads.grad_decay) - ref[2]) <= TOL * size).all()


@pytest.mark.parametrize("T,N,D", [(40, 32, 24), (200, 96, 160), (600, 32, 24)])
def test_values_without_bf16_parts(T, N, D):
    # An infinity, a NaN and a finite value above bf16's largest: every output
    # is what fp32 products give, infinite and NaN in the same places.
    torch = need_gpu()
    import burn_dragon_amd as bd
    rng = np.random.default_rng(T)
    q = np.abs(rng.standard_normal((1, 1, T, N))).astype(np.float32)
    v = np.abs(rng.standard_normal((1, 1, T, D))).astype(np.float32) * 1e-3
    q[0, 0, 5, 3] = np.inf
    v[0, 0, 9, 4] = np.nan
    v[0, 0, 11, 2] = 3.4e38
    q[0, 0, 20, :] = 0.0
    q[0, 0, 20, 7] = 3.4e38
    announce("f32 split, values without parts", T, N, D)
    out = bd.try_fused_recurrent_attention(dev(torch, q), dev(torch, v))
    torch.cuda.synchronize()
    q, v = q[0, 0].astype(np.float64), v[0, 0].astype(np.float64)
    with np.errstate(all="ignore"):
        s = (q[:, None, :] * q[None, :, :]).sum(-1).astype(np.float32).astype(np.float64)
        ctx = np.stack([(s[t, :t, None] * v[:t]).sum(0) for t in range(T)]).astype(np.float32)
        rho = (q[:, :, None] * v[:, None, :]).sum(0).astype(np.float32)
    assert np.isnan(rho).any() and np.isinf(rho).any() and np.isinf(ctx).any()
    # (A masked score is a 0 in the product with v: rows up to the NaN's may be NaN.)
    got = host(out.context)[0, 0]
    for rows in (slice(0, 5), slice(10, T)):
        cols = np.arange(D) != 4 if rows.start == 0 else slice(None)
        np.testing.assert_allclose(got[rows][:, cols], ctx[rows][:, cols], rtol=1e-5)
    np.testing.assert_allclose(host(out.rho)[0, 0], rho, rtol=1e-5)


@pytest.mark.parametrize("T,N,D", [(40, 32, 24), (300, 96, 160), (600, 160, 24)])
def test_operands_too_small_for_their_parts(oracle, T, N, D):
    # Operands near 2^-120, whose low part ends at bf16's smallest (2^-133) and
    # keeps 13 bits of 24: queries against large values (the state), and an
    # output gradient (every product of the backward but the scores).
    torch = need_gpu()
    import burn_dragon_amd as bd
    rng = np.random.default_rng(T)
    small, large = np.float32(2.0 ** -120), np.float32(2.0 ** 100)
    q = rng.standard_normal((1, 2, T, N)).astype(np.float32)
    v = rng.standard_normal((1, 1, T, D)).astype(np.float32)
    rho = rng.standard_normal((1, 2, N, D)).astype(np.float32)
    g = rng.standard_normal((1, 2, T, D)).astype(np.float32) * small
    announce("f32 split, small operands", T, N, D)
    out = bd.try_fused_recurrent_attention(dev(torch, q * small), dev(torch, v * large))
    grads = bd.recurrent_attention_vjp(dev(torch, g), dev(torch, q), dev(torch, v), dev(torch, rho))
    torch.cuda.synchronize()
    assert rel_l2(host(out.rho), oracle.recurrent_f64(q * small, v * large)[1]) <= TOL
    ref = oracle.attention_vjp_f64(q, v, g, None, rho, safe="recurrent")
    assert rel_l2(host(grads.grad_query), ref[0]) <= TOL
    assert rel_l2(host(grads.grad_value), ref[1]) <= TOL
    assert rel_l2(host(grads.grad_rho), ref[3]) <= TOL


@pytest.mark.parametrize("T,decay", [(4200, [0.999, 0.99, 0.9999, 0.9]), (4608, None)])
def test_groups_of_intervals(oracle, T, decay):
    # The scores of 128 streams fill a group with two intervals: nine of them
    # are five groups, the last a single (and, at T = 4200, a shorter) one.
    torch = need_gpu()
    import burn_dragon_amd as bd
    B, H, N, D = 32, 4, 32, 16
    g = torch.Generator(device="cuda").manual_seed(T)
    q = torch.randn(B, H, T, N, generator=g, device="cuda")
    v = torch.randn(B, 1, T, D, generator=g, device="cuda") / 16
    rho = torch.randn(B, H, N, D, generator=g, device="cuda") * 0.2
    d = dev(torch, np.asarray(decay, np.float32)) if decay else None
    announce("f32 groups of intervals", T, decay)
    out = bd.try_fused_recurrent_attention(q, v, rho.clone(), d)
    r = rho.clone()
    inplace = bd.try_fused_recurrent_attention(q, v, r, d, inplace=True)
    torch.cuda.synchronize()
    assert torch.equal(out.context, inplace.context) and torch.equal(out.rho, r)
    for b, h in ((0, 0), (13, 2), (31, 3)):
        ctx, rho1 = oracle.recurrent_f64(host(q[b, h])[None, None], host(v[b, 0])[None, None], host(rho[b, h])[None, None],
                                         np.asarray(decay[h:h + 1], np.float32) if decay else None)
        assert rel_l2(host(out.context[b, h]), ctx[0, 0]) <= TOL
        assert rel_l2(host(out.rho[b, h]), rho1[0, 0]) <= TOL


def test_groups_shrink_where_memory_is_short():
    # Eight intervals in one group hold 0.7 GB of states and scores: with less
    # than that left on the device the call runs in smaller groups.
    torch = need_gpu()
    import burn_dragon_amd as bd
    B, H, T, N, D = 4, 4, 4096, 4096, 256
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randn(B, H, T, N, generator=g, device="cuda")
    v = torch.randn(B, 1, T, D, generator=g, device="cuda") / 16
    announce("f32 groups, memory short")
    want = bd.try_fused_recurrent_attention(q, v)
    spare = bd.try_fused_recurrent_attention(q, v)  # its outputs' memory, kept for the next call
    torch.cuda.synchronize()
    bd.release_stream_scratch()
    del spare
    hold = []
    try:
        free = torch.cuda.mem_get_info()[0]
        while free > 400 << 20:
            hold.append(torch.empty(min(free - (300 << 20), 32 << 30), dtype=torch.uint8, device="cuda"))
            free = torch.cuda.mem_get_info()[0]
        out = bd.try_fused_recurrent_attention(q, v)
        torch.cuda.synchronize()
    finally:
        del hold
        bd.release_stream_scratch()
        torch.cuda.empty_cache()
    assert rel_l2(host(out.context), host(want.context)) <= TOL
    assert rel_l2(host(out.rho), host(want.rho)) <= TOL


@pytest.mark.parametrize("warm,T", [(256, 1500), (1024, 4096), (4096, 700)])
def test_captured_in_the_scratch_of_another_length(warm, T):
    # A capture takes the groups and split-K ranges that the stream's scratch has room for.
    torch = need_gpu()
    import burn_dragon_amd as bd
    B, H, N, D = 1, 4, 512, 64
    g = torch.Generator(device="cuda").manual_seed(T)
    q = torch.randn(B, H, max(warm, T), N, generator=g, device="cuda")
    v = torch.randn(B, 1, max(warm, T), D, generator=g, device="cuda") / 16
    qt, vt = q[:, :, :T].contiguous(), v[:, :, :T].contiguous()
    announce("f32 captured", warm, T)
    want = bd.try_fused_recurrent_attention(qt, vt)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(st):
        bd.try_fused_recurrent_attention(q[:, :, :warm].contiguous(), v[:, :, :warm].contiguous())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        out = bd.try_fused_recurrent_attention(qt, vt)
    assert out is not None
    for _ in range(3):
        out.context.zero_()
        out.rho.zero_()
        bd.try_fused_recurrent_attention(qt, vt)
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(host(out.context), host(want.context)) <= TOL
        assert rel_l2(host(out.rho), host(want.rho)) <= TOL
    del graph
    bd.release_stream_scratch(st)


@pytest.mark.parametrize("T", [300, 700])
@pytest.mark.parametrize("decay", [[0.7788, 0.5], [-0.7, 1.0], [1.02, 0.6]])
def test_state_of_neurons_long_silent(oracle, T, decay):
    # Neurons active at one token each: their rows of the state decay with the
    # tokens since, down to fp32's smallest normal number and beyond.  Every
    # value but the denormal ones keeps fp32's accuracy.
    torch = need_gpu()
    import burn_dragon_amd as bd
    N, D = 160, 70
    rng = np.random.default_rng(T)
    q = np.zeros((1, 2, T, N), np.float32)
    at = rng.integers(0, T, N)
    q[:, :, at, np.arange(N)] = rng.uniform(0.5, 2.0, (1, 2, N))
    v = rng.standard_normal((1, 1, T, D)).astype(np.float32)
    d = np.asarray(decay, np.float32)
    announce("f32 split, long silent neurons", T, decay)
    out = bd.try_fused_recurrent_attention(dev(torch, q), dev(torch, v), None, dev(torch, d))
    torch.cuda.synchronize()
    want = q.astype(np.float64).transpose(0, 1, 3, 2) * d.astype(np.float64)[:, None, None] ** (T - np.arange(T)) @ v
    got = out.rho.cpu().numpy()
    ok = np.abs(want) >= 2.0 ** -125
    # (Two powers of d, two products and a sum in fp32: 8 roundings of at most an ulp or so.)
    np.testing.assert_allclose(got[ok], want[ok], rtol=8 * 2.0 ** -23)
    assert np.all(np.abs(got[~ok]) <= 2.0 ** -124)


def test_decayed_sums_past_the_scaled_range(oracle):
    # The decayed operand is multiplied by 2^40: sums above 2^88 leave fp32's
    # range so scaled, and are computed again.
    torch = need_gpu()
    import burn_dragon_amd as bd
    B, H, T, N, D = 1, 2, 600, 96, 70
    rng = np.random.default_rng(5)
    q = rng.standard_normal((B, H, T, N)).astype(np.float32) * np.float32(2.0 ** 50)
    v = rng.standard_normal((B, 1, T, D)).astype(np.float32) * np.float32(2.0 ** 50)
    d = np.array([0.99, 0.9], np.float32)
    announce("f32 split, decayed sums past the scaled range")
    rho = bd.try_fused_recurrent_attention(dev(torch, q), dev(torch, v), None, dev(torch, d)).rho
    torch.cuda.synchronize()
    assert rel_l2(host(rho), oracle.recurrent_f64(q, v, None, d)[1]) <= TOL
