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
