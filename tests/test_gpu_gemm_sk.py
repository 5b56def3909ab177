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


def test_streams_past_the_areas():
    """Cut calls in flight on more streams than have areas for partial tiles,
    each on X of its own: every result within the bound of its own oracle
    values, and on the first streams, which have an area, also the bits that
    the same call gives on the current stream."""
    import ctypes
    import torch
    from xinfer_amd import _lib, ops
    M, N, K = 512, 136, 640  # 20 runs over 4 tiles; 4 runs of whole tiles without an area
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
    shapes = [(40, 640, 5120), (300, 136, 2560)]
    calls = []
    for M, N, K in shapes:
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
    """A captured gate/up + down pair, replayed with other work in between:
    every replay bit-identical to the eager pass."""
    import torch
    from xinfer_amd import ops
    M, N, K = 50, 1024, 1536
    W, S, Xb = _inputs(M, N, K, 9)
    U, T, _ = _inputs(M, N, K, 10)
    D, E, _ = _inputs(M, K, N, 11)
    g, u, d = (to_dev(W), f16_dev(S)), (to_dev(U), f16_dev(T)), (to_dev(D), f16_dev(E))
    x = f16_dev(Xb)
    act = torch.empty((M, N), dtype=torch.float16, device="cuda")
    out = torch.empty((M, K), dtype=torch.float16, device="cuda")

    def step():
        ops.mlp_gate_up_swiglu_int4(act, x, *g, *u, M, N, K)
        ops.linear_int4(out, act, *d, None, M, K, N)

    step()
    torch.cuda.synchronize()
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(4):
        out.zero_()
        act.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        step()
        torch.cuda.synchronize()
