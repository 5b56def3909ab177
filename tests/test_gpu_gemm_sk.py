"""The prefill GEMM with evenly cut work (gemm_sk_int4.hip) at the edges of
its tiles and cuts: row counts around 32-row tiles and 128-row blocks, group
counts that leave half a step, column counts around a tile and its 16-byte
stores, every output form.  Bounds: fp32 outputs max abs 1e-4 as for every
exact route (a sum of K fp32 products of |x| ~ 1 and |q s| <= 0.2 rounds to
about 1e-6); fp16 outputs half a unit of the value (2^-11) beside that."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import cpu_threads, f16_dev, to_dev, to_np
from xinfer_amd import synth

pytestmark = pytest.mark.gpu

# (MT, M, N, K) and (MT, M, Ns, K): calls whose plan has MT row tiles and runs
# that end inside tiles, so that the second launch adds pieces
# (tests/test_plan_invariants.py asks the planner for each).  M <= 16: calls
# that small_batch sends here.
CUT_SWIGLU = [(1, 23, 200, 8192), (2, 64, 2000, 3456), (3, 96, 4000, 2176), (4, 250, 1500, 2176), (1, 12, 2400, 17408),
              (1, 13, 6500, 6272)]
CUT_FUSED = [(1, 23, (300, 48, 130), 5120), (2, 60, (4000, 700, 48), 3456), (3, 90, (4600, 1, 900, 48), 3200),
             (4, 250, (3000, 1, 300, 48), 2176), (1, 16, (9000, 100), 9088)]
CUT_STREAMS = [(4, 512, 136, 640), (1, 40, 640, 5120), (3, 300, 136, 2560)]  # many streams; two threads; a first call
CUT_GRAPH = [(1, 20, 2048, 3072), (1, 20, 3072, 2048), (3, 300, 136, 2560)]  # gate/up, down, other work


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    torch.cuda.synchronize()


def _inputs(M, N, K, seed):
    W, S = synth.packed_weights(seed, N, K), synth.scales(seed, N, K)
    return W, S, synth.activations(seed, M, K)


def _check16(y, ref):
    y = oracle.f16_to_f32(to_np(y)).astype(np.float64)
    assert np.isfinite(y).all()
    over = np.abs(y - ref) - (np.abs(ref) * 2.0 ** -11 + 1e-4)
    assert over.max() <= 0, over.max()


@pytest.mark.parametrize("M,N,K", [(17, 1, 128), (17, 130, 256), (32, 257, 384), (33, 128, 3456), (64, 600, 640),
                                   (65, 255, 1024), (96, 72, 2176), (97, 300, 128), (128, 1000, 896),
                                   (129, 264, 1152), (160, 48, 5120), (257, 520, 384), (512, 136, 640),
                                   (9, 9001, 9088), (16, 15632, 5248)])  # M <= 16: long K, many weights
def test_plain_forms(M, N, K):
    import torch
    from xinfer_amd import ops
    print("case plain", M, N, K, flush=True)
    W, S, Xb = _inputs(M, N, K, M + N)
    dW, dS, dX = to_dev(W), f16_dev(S), f16_dev(Xb)
    bias = np.linspace(-1, 1, N).astype(np.float32)
    ref = oracle.linear_int4(oracle.f16_to_f32(Xb), W, S, M, N, K, nthreads=cpu_threads())
    y32 = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    ops.linear_int4(y32, dX, dW, dS, to_dev(bias), M, N, K)
    assert np.abs(to_np(y32) - (ref + bias)).max() <= 1e-4
    # two bytes past a 16-byte boundary: element stores, nothing outside
    buf = torch.full((M * N + 8,), float("nan"), dtype=torch.float16, device="cuda")
    y = buf[1:1 + M * N].view(M, N)
    ops.linear_int4(y, dX, dW, dS, None, M, N, K)
    _check16(y, ref)
    assert torch.isnan(buf[0]) and torch.isnan(buf[1 + M * N:]).all()
    y2 = torch.empty((M, N), dtype=torch.float16, device="cuda")
    ops.linear_int4(y2, dX, dW, dS, None, M, N, K)
    if K % 1024 or N < 4096:  # the same kernel for both (the other GEMM takes launches that fill the chip)
        assert torch.equal(y, y2)
    r0 = torch.from_numpy(np.random.default_rng(M).normal(0, 1, (M, N))).half().cuda()
    r = r0.clone()
    ops.linear_int4_residual(r, dX, dW, dS, None, M, N, K)
    assert torch.equal(r, (y2.float() + r0.float()).half())


@pytest.mark.parametrize("M,N,K", [(17, 16, 128), (23, 1100, 640), (40, 129, 1024), (77, 264, 384), (130, 900, 896),
                                   (300, 257, 512)])
def test_swiglu(M, N, K):
    import torch
    from xinfer_amd import ops
    print("case swiglu", M, N, K, flush=True)
    W, S, Xb = _inputs(M, N, K, M + N)
    U, T, _ = _inputs(M, N, K, M + N + 1)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    ops.mlp_gate_up_swiglu_int4(y, f16_dev(Xb), to_dev(W), f16_dev(S), to_dev(U), f16_dev(T), M, N, K)
    _check16(y, oracle.swiglu_int4(oracle.f16_to_f32(Xb), W, S, U, T, M, N, K, nthreads=cpu_threads()))


def _cols(N, seed):
    """Columns that stand for a wide output: both ends and a hundred others."""
    c = np.random.default_rng(seed).integers(0, N, 100)
    return np.unique(np.concatenate([c, np.arange(min(N, 40)), np.arange(max(0, N - 40), N)]))


@pytest.mark.parametrize("mt,M,N,K", CUT_SWIGLU)
def test_swiglu_in_pieces(mt, M, N, K):
    """Also with the norm before it: the bits of norm and SwiGLU called apart."""
    import torch
    from xinfer_amd import ops
    print("case swiglu in pieces", M, N, K, flush=True)
    W, S = synth.packed_weights(M + N, N, K), synth.scales(M + N, N, K, 0.01)  # keeps SiLU(g) * u near 1 at long K
    U, T, Xb = synth.packed_weights(M, N, K), synth.scales(M, N, K, 0.01), synth.activations(M + N, M, K)
    g, u, x = (to_dev(W), f16_dev(S)), (to_dev(U), f16_dev(T)), f16_dev(Xb)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    ops.mlp_gate_up_swiglu_int4(y, x, *g, *u, M, N, K)
    assert torch.isfinite(y).all()
    c = _cols(N, M)
    ref = oracle.swiglu_int4(oracle.f16_to_f32(Xb), W[c], S[c], U[c], T[c], M, len(c), K, nthreads=cpu_threads())
    _check16(y[:, torch.from_numpy(c).cuda()], ref)
    nw = to_dev(np.random.default_rng(M).normal(1, 0.1, K).astype(np.float32))
    xn, a, b = torch.empty_like(x), torch.empty_like(y), torch.full_like(y, float("nan"))
    ops.rmsnorm(xn, x, nw, M, K, 1e-6)
    ops.mlp_gate_up_swiglu_int4(a, xn, *g, *u, M, N, K)
    ops.rmsnorm_mlp_gate_up_swiglu_int4(b, x, nw, 1e-6, *g, *u, M, N, K)
    assert torch.equal(a, b)


@pytest.mark.parametrize("mt,M,Ns,K", CUT_FUSED)
def test_fused_with_bias_in_pieces(mt, M, Ns, K):
    import torch
    from xinfer_amd import ops
    print("case fused in pieces", M, Ns, K, flush=True)
    Xb = synth.activations(M, M, K)
    x = f16_dev(Xb)
    descs, refs = [], []
    for i, N in enumerate(Ns):
        W, S = synth.packed_weights(M + i, N, K), synth.scales(M + i, N, K)
        bias = np.linspace(-1 - i, 1, N).astype(np.float32)
        y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        descs.append(ops.FusedProjectionDesc(y, to_dev(W), f16_dev(S), to_dev(bias), N))
        c = _cols(N, i)
        refs.append((c, oracle.linear_int4(oracle.f16_to_f32(Xb), W[c], S[c], M, len(c), K, nthreads=cpu_threads()) + bias[c]))
    ops.linear_int4_fused(x, descs, len(Ns), M, K)
    for d, (c, ref) in zip(descs, refs):
        assert torch.isfinite(d.Y).all()
        _check16(d.Y[:, torch.from_numpy(c).cuda()], ref)
    nw = to_dev(np.random.default_rng(M).normal(1, 0.1, K).astype(np.float32))
    xn = torch.empty_like(x)
    ops.rmsnorm(xn, x, nw, M, K, 1e-6)
    ops.linear_int4_fused(xn, descs, len(Ns), M, K)
    want = [d.Y.clone() for d in descs]
    for d in descs:
        d.Y.fill_(float("nan"))
    ops.rmsnorm_linear_int4_fused(x, nw, 1e-6, descs, len(Ns), M, K)
    for d, w in zip(descs, want):
        assert torch.equal(d.Y, w)


def test_more_rows_than_a_slab():
    """65536 rows go out in one slab, the 17 after them in another."""
    import torch
    from xinfer_amd import ops
    M, Ns, K = 65536 + 17, (16, 40), 128
    Xb = synth.activations(3, M, K)
    x, X = f16_dev(Xb), oracle.f16_to_f32(Xb)
    descs, refs = [], []
    for N in Ns:
        W, S = synth.packed_weights(N, N, K), synth.scales(N, N, K)
        y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        descs.append(ops.FusedProjectionDesc(y, to_dev(W), f16_dev(S), None, N))
        refs.append(oracle.linear_int4(X, W, S, M, N, K, nthreads=cpu_threads()))
    ops.linear_int4_fused(x, descs, 2, M, K)
    for d, ref in zip(descs, refs):
        _check16(d.Y, ref)
    d = descs[0]
    y32 = torch.full((M, d.N), float("nan"), device="cuda")
    ops.linear_int4(y32, x, d.W_int4, d.scales, None, M, d.N, K)
    assert np.abs(to_np(y32) - refs[0]).max() <= 1e-4
    r0 = torch.from_numpy(np.random.default_rng(1).normal(0, 1, (M, d.N))).half().cuda()
    r = r0.clone()
    ops.linear_int4_residual(r, x, d.W_int4, d.scales, None, M, d.N, K)
    assert torch.equal(r, (d.Y.float() + r0.float()).half())


def test_streams_past_the_areas():
    """Cut calls in flight on more streams than have areas for partial tiles,
    each on X of its own: every result within the bound of its own oracle
    values, and on the first streams, which have an area, also the bits that
    the same call gives on the current stream."""
    import ctypes
    import torch
    from xinfer_amd import _lib, ops
    _, M, N, K = CUT_STREAMS[0]  # whole tiles without an area
    W, S, _ = _inputs(M, N, K, 5)
    Xs = [synth.activations(100 + i, M, K) for i in range(36)]
    dW, dS, dXs = to_dev(W), f16_dev(S), [f16_dev(x) for x in Xs]
    refs = [oracle.linear_int4(oracle.f16_to_f32(x), W, S, M, N, K, nthreads=cpu_threads()) for x in Xs]
    solo = torch.full((36, M, N), float("nan"), device="cuda")
    for y, x in zip(solo, dXs):
        ops.linear_int4(y, x, dW, dS, None, M, N, K)
    # raw streams: torch hands out its 32 pooled ones over and over
    hip = ctypes.CDLL("libamdhip64.so")
    raw = []
    for _ in range(36):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        raw.append(h)
    ys = torch.full((3, 36, M, N), float("nan"), device="cuda")
    torch.cuda.synchronize()
    for r in range(3):  # a stream's calls differ from one to the next
        for i, h in enumerate(raw):
            j = (i + r) % 36
            ops.linear_int4(ys[r, i], dXs[j], dW, dS, None, M, N, K, stream=h.value)
    torch.cuda.synchronize()
    for h in raw:
        assert _lib.load_library().xinfer_stream_release(h) == 0
        assert hip.hipStreamDestroy(h) == 0
    for r in range(3):
        for i in range(36):
            j = (i + r) % 36
            assert np.abs(to_np(ys[r, i]) - refs[j]).max() <= 1e-4, (r, i)
            if i < 24:  # 32 areas, a few of them other tests' streams'
                assert torch.equal(ys[r, i], solo[j]), (r, i)


def test_threads_on_one_stream():
    """Two host threads with cut calls of different shapes on one stream: each
    result is what the call gives alone."""
    import threading
    import torch
    from xinfer_amd import ops
    calls = []
    for _, M, N, K in CUT_STREAMS[1:]:
        W, S, Xb = _inputs(M, N, K, M)
        calls.append((M, N, K, to_dev(W), f16_dev(S), f16_dev(Xb), torch.full((30, M, N), float("nan"), device="cuda")))
    solo = []
    for M, N, K, dW, dS, dX, ys in calls:
        solo.append(torch.empty((M, N), device="cuda"))
        ops.linear_int4(solo[-1], dX, dW, dS, None, M, N, K)
    stream = torch.cuda.current_stream().cuda_stream
    torch.cuda.synchronize()

    def work(M, N, K, dW, dS, dX, ys):
        for y in ys:
            ops.linear_int4(y, dX, dW, dS, None, M, N, K, stream=stream)

    threads = [threading.Thread(target=work, args=c) for c in calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for c, want in zip(calls, solo):
        for y in c[-1]:
            assert torch.equal(y, want)


def test_graph_replay():
    """A captured gate/up + down pair, both in pieces, replayed on its stream
    with other X each time and another call in pieces between the replays:
    every result bit-identical to the eager pass on another stream."""
    import torch
    from xinfer_amd import ops
    (_, M, N, K), (_, _, N2, K2), (_, m, n, k) = CUT_GRAPH
    assert (N2, K2) == (K, N)
    W, S, _ = _inputs(M, N, K, 9)
    U, T, _ = _inputs(M, N, K, 10)
    D, E, _ = _inputs(M, K, N, 11)
    O, P, Zb = _inputs(m, n, k, 12)
    g, u, d, o = (to_dev(W), f16_dev(S)), (to_dev(U), f16_dev(T)), (to_dev(D), f16_dev(E)), (to_dev(O), f16_dev(P))
    xs, z = [f16_dev(synth.activations(20 + i, M, K)) for i in range(5)], f16_dev(Zb)
    x = torch.empty_like(xs[0])
    act = torch.empty((M, N), dtype=torch.float16, device="cuda")
    out = torch.empty((M, K), dtype=torch.float16, device="cuda")
    other, want_other = torch.empty((m, n), device="cuda"), torch.empty((m, n), device="cuda")

    def step():
        ops.mlp_gate_up_swiglu_int4(act, x, *g, *u, M, N, K)
        ops.linear_int4(out, act, *d, None, M, K, N)

    want = []
    for xi in xs:
        x.copy_(xi)
        step()
        want.append((act.clone(), out.clone()))
    ops.linear_int4(want_other, z, *o, None, m, n, k)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        step()
    with torch.cuda.stream(stream):
        for xi, (wa, wo) in zip(xs, want):
            x.copy_(xi)
            out.zero_()
            act.zero_()
            other.zero_()
            ops.linear_int4(other, z, *o, None, m, n, k)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(act, wa) and torch.equal(out, wo)
            assert torch.equal(other, want_other)
