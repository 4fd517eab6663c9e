"""A decode step whose streams are split into row ranges: the last range to
finish sums the partial readouts, in range order (the same bits as the
finalize launch of a step that also returns its active rows), step after
step, and in graph replays with other work between them."""
import numpy as np
import pytest

from tests.gpu_util import TOL_F32, announce, dev, host, need_gpu, rel_l2

pytestmark = pytest.mark.gpu


def _inputs(torch, B, H, N, D, seed):
    rng = np.random.default_rng(seed)
    x = np.maximum(rng.standard_normal((B, H, N)) - 1.645, 0).astype(np.float32)
    v = (rng.standard_normal((B, 1, D)) / 16).astype(np.float32)
    rho = (rng.standard_normal((B, H, N, D)) * 0.2).astype(np.float32)
    return dev(torch, x), dev(torch, v), dev(torch, rho)


@pytest.mark.parametrize("B,H,N,D", [
    (1, 4, 8192, 256),   # 32 ranges
    (1, 1, 514, 96),     # 4 ranges, the last ragged: the finalize launch in both forms
    (3, 4, 2050, 65),    # scalar columns, ranges not a multiple of 8 rows apart from the last
    (1, 1, 1026, 96),    # 8 ranges, the fewest summed in the step, the last ragged
    (1, 2, 4096, 600),   # three column blocks
    (32, 4, 1024, 64),   # 2 ranges on 128 streams, the most that are split: likewise
])
def test_combined_readout_is_the_finalized_one(oracle, B, H, N, D):
    # (Where both forms end in the finalize launch, the oracle's step is the other side.)
    torch = need_gpu()
    import burn_dragon_amd as bd
    announce("decode combine", B, H, N, D)
    x, v, rho = _inputs(torch, B, H, N, D, N)
    r1, r2 = rho.clone(), rho.clone()
    rho_ref = host(rho)
    a_ref, _, _ = oracle.decode_step_f32(host(x), host(v), rho_ref, 3)
    r3 = rho.clone()
    assert rel_l2(host(bd.decode_step(x, v, r3, position=3).readout), a_ref) <= TOL_F32
    assert rel_l2(host(r3), rho_ref) <= TOL_F32
    for step in range(6):
        a = bd.decode_step(x, v, r1, position=step).readout
        b = bd.decode_step(x, v, r2, position=step, want_active=True).readout
        torch.cuda.synchronize()
        assert torch.equal(a, b) and torch.equal(r1, r2), step


def test_replays_with_other_steps_between_them():
    torch = need_gpu()
    import burn_dragon_amd as bd
    announce("decode combine in a graph")
    x, v, rho = _inputs(torch, 1, 4, 8192, 256, 3)
    x2, v2, rho2 = _inputs(torch, 2, 4, 4096, 128, 4)
    out = torch.empty(1, 4, 256, device="cuda")
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        r = rho.clone()
        # The lists' form warms the stream; the form captured is the other one.
        bd.decode_step(x, v, r, position=0, want_active=True)
        r.copy_(rho)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            bd.decode_step(x, v, r, position=9, out=out)
        ref = rho.clone()
        for i in range(4):
            graph.replay()
            bd.decode_step(x2, v2, rho2, position=i)
            want = bd.decode_step(x, v, ref, position=9).readout
            torch.cuda.synchronize()
            assert torch.equal(out, want) and torch.equal(r, ref), i
        del graph
    bd.release_stream_scratch(st)


def test_overlapped_replays_spoil_no_later_step():
    # Two graphs captured on one stream share its buffers and must not overlap;
    # where they do all the same, every later replay is right again.
    torch = need_gpu()
    import burn_dragon_amd as bd
    announce("decode combine after overlapped replays")
    sizes = [(1, 4, 8192, 256), (2, 4, 4096, 128)]  # 32 ranges, 16
    st, other = torch.cuda.Stream(), torch.cuda.Stream()
    graphs = []
    for seed, (B, H, N, D) in enumerate(sizes):
        x, v, rho = _inputs(torch, B, H, N, D, seed)
        want = bd.decode_step(x, v, rho.clone(), position=9).readout
        out, r = torch.empty(B, H, D, device="cuda"), rho.clone()
        with torch.cuda.stream(st):
            bd.decode_step(x, v, r, position=9)
        torch.cuda.synchronize()
        graphs.append([x, v, rho, r, out, want])
    for c in graphs + graphs[:1]:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            bd.decode_step(c[0], c[1], c[3], position=9, out=c[4])
        c.append(g)
    for i in range(20):
        for a, b in ((graphs[0][6], graphs[1][6]), (graphs[0][6], graphs[0][7])):
            with torch.cuda.stream(st):
                a.replay()
            with torch.cuda.stream(other):
                b.replay()
            torch.cuda.synchronize()
        for c in graphs:
            c[3].copy_(c[2])
            c[4].zero_()
            c[6].replay()
            torch.cuda.synchronize()
            assert torch.equal(c[4], c[5]), i
    del graphs
    bd.release_stream_scratch(st)


def test_short_streams_are_captured_without_an_eager_call():
    # Fewer than 512 rows: the step takes no scratch, so a stream's first call may be a captured one.
    torch = need_gpu()
    import burn_dragon_amd as bd
    announce("decode of short streams captured cold")
    x, v, rho = _inputs(torch, 2, 4, 510, 64, 5)
    ref = rho.clone()
    want = bd.decode_step(x, v, ref, position=9).readout  # frequency table resident
    out = torch.empty(2, 4, 64, device="cuda")
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        r = rho.clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            bd.decode_step(x, v, r, position=9, out=out)
        for i in range(3):
            r.copy_(rho)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want) and torch.equal(r, ref), i
        del graph
    bd.release_stream_scratch(st)
