"""Sequences whose length is no multiple of a tile: the layer's 128-token
tiles with missing rows (bdh_lowrank_layer_fwd), and a call of one interval
that continues a state, on both of its routes."""
import ctypes

import numpy as np
import pytest

from tests.gpu_util import TOL_BF16, announce, dev, host, need_gpu, rel_l2

pytestmark = pytest.mark.gpu


def _launches(bd, run):
    """run()'s result, and its launches of the prefill kernels and in all: a
    call of one interval makes (2, 4) in the state-carry form; in the other
    one launch of gram, readout and state units, (1, 4), or two in place,
    (2, 5)."""
    from burn_dragon_amd import _lib
    lib = _lib.load()
    bd.recurrent_profile_enable(True)
    bd.recurrent_profile_reset()
    assert lib.bdh_profile_kernel_timing(1) == _lib.BDH_OK
    try:
        out = run()
        ms, n = ctypes.c_double(), ctypes.c_int64()
        assert lib.bdh_profile_kernel_get(_lib.BDH_KERNEL_PREFILL, ctypes.byref(ms), ctypes.byref(n)) == _lib.BDH_OK
        return out, (n.value, bd.recurrent_profile_snapshot().launches)
    finally:
        lib.bdh_profile_kernel_timing(0)
        bd.recurrent_profile_enable(False)


# x: the wave-role GEMM X; yz: GEMM Y and the decoder in one launch.  Both take
# a sequence in tiles of 128 tokens, the other routes pack the rows.
@pytest.mark.parametrize("B,H,T,N,D,carried,yz", [
    (2, 2, 65, 256, 64, False, False),     # x: one tile a sequence, just over half filled
    (2, 2, 63, 256, 64, True, False),      # x: just under half
    (3, 1, 129, 512, 128, True, False),    # x: a second tile of one row
    (1, 2, 255, 512, 256, False, False),   # x: one row short of two tiles
    (5, 2, 200, 256, 192, True, False),    # x: ten tiles
    (5, 4, 20, 8192, 64, False, True),     # packed x: five row tiles for 100 rows
    (2, 4, 33, 2048, 64, False, True),     # a quarter filled
    (3, 2, 129, 4096, 128, True, True),    # a second tile of one row
    (1, 4, 255, 4096, 256, False, True),   # one row short of two tiles
    (20, 4, 100, 3328, 64, True, True),    # 20 tiles, ranges of unequal chunk counts
])
def test_layer_tiles_match_oracle(oracle, B, H, T, N, D, carried, yz):
    torch = need_gpu()
    import burn_dragon_amd as bd
    rng = np.random.default_rng(T * 3 + N)
    cur = oracle.layer_norm_f64(rng.standard_normal((B, T, D))).astype(np.float32)
    enc, encv = ((rng.standard_normal((H, D, N)) * 0.05).astype(np.float32) for _ in range(2))
    dec = (rng.standard_normal((H * N, D)) * 0.05).astype(np.float32)
    rho0 = (rng.standard_normal((B, H, N, D)) * 0.05).astype(np.float32) if carried else None
    w = bd.LowRankWeights.pack(dev(torch, enc[None]), dev(torch, encv[None]), dev(torch, dec))
    announce("layer tiles", B, H, T, N, D, carried, yz)
    # Scratch rows past the last token hold whatever was there: make it NaN.
    big = torch.full((B, T + 200, D), float("nan"), device="cuda")
    bd.lowrank_layer_forward(big, w, position=0)
    out, (_, n) = _launches(bd, lambda: bd.lowrank_layer_forward(
        dev(torch, cur), w, position=7, rho=dev(torch, rho0) if carried else None, want_rho=carried))
    torch.cuda.synchronize()
    # Rows to bf16, X, LayerNorm, Y and decoder, residual; the attention's v^T,
    # scores, context and, onto a state, the readout's sum.
    assert n == (5 if yz else 6) + (4 if carried else 3)
    nref, rref = oracle.lowrank_layer_f64(cur, oracle.round_bf16(enc), oracle.round_bf16(encv),
                                          oracle.round_bf16(dec), pos0=7, rho0=rho0)
    assert rel_l2(host(out.next), nref) <= TOL_BF16
    if carried:
        assert rel_l2(host(out.rho), rref) <= TOL_BF16


@pytest.mark.parametrize("B,T,N,D,rope,decay,inplace,carry", [
    (1, 130, 512, 96, 5, None, False, False),                    # few elements: gram, readout and state units
    (1, 130, 512, 96, None, [0.99, 0.98, 0.97, 0.96], True, False),
    (2, 390, 8192, 64, 5, None, False, False),                   # many, few columns: the same
    (2, 390, 8192, 64, 5, None, True, False),
    (2, 390, 8192, 64, None, [0.99, 0.98, 0.97, 0.96], False, False),
    (8, 390, 4096, 192, 5, None, False, False),                  # many, out of place: not enough beyond 320 tokens
    (8, 310, 5120, 192, 5, None, False, True),                   # enough below: the state-carry form
    (6, 390, 5632, 192, 5, None, False, True),                   # of 24 streams
    (4, 390, 8192, 192, 5, None, True, True),                    # in place
    (4, 390, 8192, 192, None, None, False, True),                # no rotation
    (4, 390, 8192, 192, None, [0.99, 0.98, 0.97, 0.96], False, False),
    (6, 390, 8192, 192, None, [0.99, 0.98, 0.97, 0.96], False, True),
    (6, 390, 8192, 224, None, [0.99, 0.98, 0.97, 0.96], False, False),
    (5, 410, 6400, 160, None, [0.99, 0.98, 0.97, 0.96], False, True),
    (4, 390, 8192, 192, 5, [0.99, 0.98, 0.97, 0.96], True, True),
])
def test_one_interval_onto_a_state(oracle, B, T, N, D, rope, decay, inplace, carry):
    torch = need_gpu()
    import burn_dragon_amd as bd
    H = 4
    rng = np.random.default_rng(N + T)
    x = oracle.round_bf16(np.maximum(rng.standard_normal((B, H, T, N), dtype=np.float32) - 1.645, 0))
    v = oracle.round_bf16(rng.standard_normal((B, 1, T, D), dtype=np.float32) / 16)
    rho0 = (rng.standard_normal((B, H, N, D)) * 0.2).astype(np.float32)
    d = np.array(decay, np.float32) if decay else None
    announce("one interval onto a state", B, T, N, D, rope, decay, inplace)
    tx, tv = dev(torch, x, torch.bfloat16), dev(torch, v, torch.bfloat16)
    tr, td = dev(torch, rho0), dev(torch, d) if decay else None
    kw = dict(inplace=inplace)
    out, n = _launches(bd, lambda: (
        bd.try_fused_recurrent_attention(tx, tv, tr, td, **kw) if rope is None else
        bd.try_fused_recurrent_attention_rope(tx, tv, tr, td, position=rope, **kw)))
    torch.cuda.synchronize()
    assert n == ((2, 4) if carry else (2, 5) if inplace else (1, 4))
    assert (out.rho.data_ptr() == tr.data_ptr()) == inplace
    if not inplace:
        assert np.array_equal(host(tr), rho0)
    for b, h in ((0, 0), (B - 1, 3)):
        q = x[b:b + 1, h:h + 1]
        q = q if rope is None else oracle.rope_rotate(q, pos0=rope)
        ctx, rho = oracle.recurrent_f64(q, v[b:b + 1], rho0[b:b + 1, h:h + 1], d[h:h + 1] if decay else None)
        assert rel_l2(host(out.context[b, h]), ctx[0, 0]) <= TOL_BF16
        assert rel_l2(host(out.rho[b, h]), rho[0, 0]) <= TOL_BF16
