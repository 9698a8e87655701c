"""The allocation-free GEMM entry point (qmatmul_gemm_noalloc) against qmatmul_gemm, through the C ABI: two calls in a
row on the static scratch array, the second with a smaller input, each bit-identical to qmatmul_gemm's result (the
same kernels run on the same inputs; only where the workspace lives differs). Also: a shape beyond the scratch's
capacity is refused with QM_ERR_WORKSPACE, and a shape on the int8 path (no scratch) matches too."""
import numpy as np
import pytest

from arcinfer_amd import formats as F

pytestmark = pytest.mark.gpu


def _case(qm, dev, qtype, M, N, K, seed):
    import torch
    W = F.synth_weight(qtype, N, K, seed=seed)
    x = F.synth_activations(M, K, seed=seed + 1, outlier_frac=0.01)
    aq, asc, absum = qm.quantize_act(torch.from_numpy(x).to(dev))
    w = qm.QWeight(qtype, torch.from_numpy(W).to(dev), N, K)
    return w, aq, asc, absum


def test_noalloc_matches_gemm_twice(qm, dev):
    import torch
    for (M, N, K, seed) in [(512, 384, 2048, 1), (200, 256, 1024, 2)]:  # second call smaller than the first
        w, aq, asc, absum = _case(qm, dev, F.Q4_K, M, N, K, seed)
        ref = qm.gemm(w, aq, asc, absum)
        got = qm.gemm(w, aq, asc, absum, noalloc=True)
        torch.cuda.synchronize()
        assert torch.equal(got, ref), (M, N, K)
        # accumulate into an offset window, as qmatmul_gemm does
        C0 = torch.randn(M, N + 8, device=dev)
        C1 = C0.clone()
        qm.gemm(w, aq, asc, absum, C=C0, ldc=N + 8, c_off=3, accumulate=1)
        qm.gemm(w, aq, asc, absum, C=C1, ldc=N + 8, c_off=3, accumulate=1, noalloc=True)
        torch.cuda.synchronize()
        assert torch.equal(C0, C1)
        w.release()


def test_noalloc_int8_path_and_capacity(qm, dev):
    import torch
    w, aq, asc, absum = _case(qm, dev, F.IQ4_XS, 64, 256, 1024, 5)
    ref = qm.gemm(w, aq, asc, absum)
    got = qm.gemm(w, aq, asc, absum, noalloc=True)
    torch.cuda.synchronize()
    assert torch.equal(got, ref)
    w.release()
    # 4096 x 5120 needs 2 * 4096 * 5120 + 4 * 4096 * 160 bytes = 44.6 MB > 32 MiB: refused, nothing written
    M, N, K = 4096, 128, 5120
    w, aq, asc, absum = _case(qm, dev, F.Q4_K, M, N, K, 7)
    C = torch.full((M, N), 3.0, device=dev)
    with pytest.raises(qm.QMatmulError) as ei:
        qm.gemm(w, aq, asc, absum, C=C, ldc=N, noalloc=True)
    assert ei.value.status == 6  # QM_ERR_WORKSPACE
    torch.cuda.synchronize()
    assert bool(torch.all(C == 3.0))
    w.release()


def test_noalloc_calls_overlap(qm, dev):
    """Cut products (IQ4_XS, Q6_K) of two streams in turn without a wait between: each the result of the call by itself, and of
    qmatmul_gemm, though their partial results share one array; and two captured ones replayed together."""
    import torch
    M, K = 70, 8192
    cases = [_case(qm, dev, F.IQ4_XS, M, 272, K, 11), _case(qm, dev, F.Q6_K, M, 400, K, 13)]
    want = [qm.gemm(*c, M=M) for c in cases]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    out = [[torch.empty_like(w) for _ in range(20)] for w in want]
    torch.cuda.synchronize()
    for i in range(20):
        for c, o, s in zip(cases, out, streams):
            qm.gemm(*c, M=M, C=o[i], ldc=c[0].rows, noalloc=True, stream=s.cuda_stream)
    torch.cuda.synchronize()
    assert all(torch.equal(C, w) for o, w in zip(out, want) for C in o)
    uncut = [qm.gemm_ws(*c, None, M=M) for c in cases]
    graphs = [torch.cuda.CUDAGraph() for _ in cases]
    for g, c, o in zip(graphs, cases, out):
        with torch.cuda.graph(g):
            qm.gemm(*c, M=M, C=o[0], ldc=c[0].rows, noalloc=True)
    for _ in range(3):
        for o in out:
            o[0].zero_()
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o[0], u) for o, u in zip(out, uncut))
    for c in cases:
        c[0].release()


def test_gemm_beside_a_capture(qm, dev):
    """A call on one stream while the thread has a capture open on another: neither disturbs the other."""
    import torch
    w, aq, asc, absum = _case(qm, dev, F.IQ4_XS, 70, 272, 8192, 17)
    want, uncut = qm.gemm(w, aq, asc, absum, M=70), qm.gemm_ws(w, aq, asc, absum, None, M=70)
    side, C, D = torch.cuda.Stream(), torch.zeros_like(want), torch.zeros_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        qm.gemm(w, aq, asc, absum, M=70, C=C, ldc=272)
        qm.gemm(w, aq, asc, absum, M=70, C=D, ldc=272, stream=side.cuda_stream)
    for _ in range(2):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, uncut) and torch.equal(D, want)
    w.release()
