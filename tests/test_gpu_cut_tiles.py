"""Prompt products whose tiles are cut along K into pieces (partial tiles added by a second kernel): against the CPU oracle at
ragged tile edges, every accumulate mode, and the three entry points bit for bit the same where all have the room."""
import numpy as np
import pytest

import oracle
from arcinfer_amd import formats as F

from .test_gpu_parity import TOL_INT8_PATH, acts, assert_elementwise, rel_err, to_dev

pytestmark = pytest.mark.gpu

# (type, M, N, K): the f16, int8 and per-16 kernels; partial row and column tiles; superblocks that do not divide evenly over
# the pieces; 522 tiles, of which the last ten are cut, and 520 of the f16 kernel's (128 x 128), of which the last eight are
CASES = [(F.Q4_K, 130, 144, 2048), (F.Q4_K, 300, 272, 5888), (F.IQ4_XS, 70, 272, 8192), (F.IQ3_S, 64, 144, 17408),
         (F.Q6_K, 70, 272, 2304), (F.Q2_K, 129, 144, 4096), (F.IQ4_XS, 520, 7376, 4096), (F.Q6_K, 520, 7376, 2816),
         (F.Q4_K, 600, 13232, 2304)]


def f16_bytes(qtype, M, K):
    """Workspace of the f16 kernel's activations alone, to whole 256 bytes (0 for the types and sizes of the other kernels)."""
    if qtype not in (F.Q4_K, F.Q5_K, F.IQ3_S) or M < 128:
        return 0
    Mp = (M + 127) // 128 * 128
    return (2 * Mp * K + Mp * (K // 32) * (8 if qtype == F.Q5_K else 4) + 255) // 256 * 256


@pytest.mark.parametrize("qtype,M,N,K", CASES)
def test_cut_tiles(qm, dev, qtype, M, N, K):
    import torch
    W = F.synth_weight(qtype, N, K, seed=qtype + M)
    aq, asc, absum = acts(qm, F.synth_activations(M, K, seed=K, outlier_frac=0.01), dev, M_stride=M + 3)
    w = qm.QWeight(qtype, to_dev(W, dev), N, K)
    need = qm.gemm_workspace_size(w, M)
    assert need > f16_bytes(qtype, M, K)  # (room for partial tiles: the call is cut)
    C = qm.gemm(w, aq, asc, absum, M=M)
    ws = torch.empty((need,), dtype=torch.uint8, device=dev)
    assert torch.equal(C, qm.gemm_ws(w, aq, asc, absum, ws, M=M))
    assert torch.equal(C, qm.gemm(w, aq, asc, absum, M=M, noalloc=True))
    g = torch.randn((M, N + 8), device=dev)
    add = qm.gemm(w, aq, asc, absum, M=M, C=g.clone(), ldc=N + 8, c_off=5, accumulate=1)
    mul = qm.gemm(w, aq, asc, absum, M=M, C=g.clone(), ldc=N + 8, c_off=5, accumulate=2)
    torch.cuda.synchronize()
    stride = max(1, N // 256)
    ref = oracle.blockdot(qtype, W, K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=M, col_stride=stride)
    sel = np.arange(0, N, stride)
    got = C.cpu().numpy()[:, sel]
    ref = ref[:, sel] if ref.shape[1] == N else ref
    assert rel_err(got, ref) < TOL_INT8_PATH
    assert_elementwise(got, ref)
    assert torch.equal(add[:, 5:5 + N], g[:, 5:5 + N] + C)
    assert torch.allclose(mul[:, 5:5 + N], torch.nn.functional.silu(g[:, 5:5 + N]) * C, rtol=1e-5,
                          atol=1e-6 * C.abs().max().item())
    for t in (add, mul):
        assert torch.equal(t[:, :5], g[:, :5]) and torch.equal(t[:, 5 + N:], g[:, 5 + N:])


@pytest.mark.parametrize("qtype", [F.IQ4_XS, F.Q6_K])
def test_no_workspace_is_accepted(qm, dev, qtype):
    """The kernels that need no workspace run without one (uncut: equal up to the f32 order of the K pieces)."""
    import torch
    M, N, K = 70, 272, 8192
    w = qm.QWeight(qtype, to_dev(F.synth_weight(qtype, N, K, seed=1), dev), N, K)
    aq, asc, absum = acts(qm, F.synth_activations(M, K, seed=2), dev, M_stride=M)
    C = qm.gemm(w, aq, asc, absum, M=M)
    D = qm.gemm_ws(w, aq, asc, absum, None, M=M)
    torch.cuda.synchronize()
    assert rel_err(D.cpu().numpy(), C.cpu().numpy()) < 1e-5


def test_captured_call_matches(qm, dev):
    """Under stream capture the int8 kernels record no allocation; every replay gives the eager uncut result."""
    import torch
    M, N, K = 70, 272, 8192
    w = qm.QWeight(F.IQ4_XS, to_dev(F.synth_weight(F.IQ4_XS, N, K, seed=1), dev), N, K)
    aq, asc, absum = acts(qm, F.synth_activations(M, K, seed=2), dev, M_stride=M)
    want = qm.gemm_ws(w, aq, asc, absum, None, M=M)
    C = torch.empty((M, N), device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        qm.gemm(w, aq, asc, absum, M=M, C=C)
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)


@pytest.mark.parametrize("qtype", [F.Q5_K, F.IQ3_S])
@pytest.mark.parametrize("act32", [True, False])
@pytest.mark.parametrize("shape", [(500, 4624, 5376), (600, 13232, 3072)])
def test_f16_types(qm, dev, qtype, act32, shape):
    """Q5_K and IQ3_S products long enough for the f16 kernels (ragged rows and tokens; all tiles cut, and 512 whole with the last
    eight cut): f32 parity, block
    sums bit for bit, and the int8 kernels behind the same call without a workspace."""
    import torch
    M, N, K = shape
    W = F.synth_weight(qtype, N, K, seed=qtype)
    x = F.synth_activations(M, K, seed=K, outlier_frac=0.01)
    aq, asc, absum = qm.quantize_act(to_dev(x, dev), M_stride=M + 3, act32=act32)
    w = qm.QWeight(qtype, to_dev(W, dev), N, K)
    assert qm.gemm_workspace_size(w, M) > f16_bytes(qtype, M, K)  # (the f16 kernel, and cut)
    C = qm.gemm(w, aq, asc, absum, M=M, act32=act32)
    D = qm.gemm_ws(w, aq, asc, absum, None, M=M, act32=act32)
    torch.cuda.synchronize()
    stride = 37
    blockdot = oracle.blockdot if act32 else oracle.blockdot256
    ref = blockdot(qtype, W, K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=M, col_stride=stride)
    sel = np.arange(0, N, stride)
    ref = ref[:, sel] if ref.shape[1] == N else ref
    for got in (C, D):
        assert rel_err(got.cpu().numpy()[:, sel], ref) < TOL_INT8_PATH
        assert_elementwise(got.cpu().numpy()[:, sel], ref)
    if act32:
        R = 64  # (rows of the block sums; the kernel choice follows the whole product's shape, so the full matrix is run)
        isum = qm.gemm_blocksums(w, aq, M=M)[:, :R].cpu().numpy()
        _, risum, _ = oracle.blockdot(qtype, W[:R], K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=M, blocksums=True)
        assert np.array_equal(isum, risum)


def test_kept_workspaces_over_streams_and_threads(qm, dev):
    """More streams than kept workspaces, each with its own inputs, calls in turn and from threads: every result is the one of a
    call by itself; and again after the last weight (of this test) went and came back."""
    import threading

    import torch
    M, N, K, S = 130, 144, 2048, 11
    W = to_dev(F.synth_weight(F.Q4_K, N, K, seed=5), dev)
    xs = [acts(qm, F.synth_activations(M, K, seed=100 + i), dev, M_stride=M) for i in range(S)]
    for _ in range(2):
        w = qm.QWeight(F.Q4_K, W, N, K)
        want = [qm.gemm(w, *x, M=M) for x in xs]
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream() for _ in range(S)]
        out = [[torch.empty((M, N), device=dev) for _ in range(4)] for _ in range(S)]
        torch.cuda.synchronize()

        def calls(i):
            for C in out[i]:
                qm.gemm(w, *xs[i], M=M, C=C, ldc=N, stream=streams[i].cuda_stream)

        for i in range(S):
            calls(i)
        torch.cuda.synchronize()
        assert all(torch.equal(C, want[i]) for i in range(S) for C in out[i])
        for i in range(S):
            for C in out[i]:
                C.zero_()
        torch.cuda.synchronize()
        ts = [threading.Thread(target=calls, args=(i,)) for i in range(S)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        torch.cuda.synchronize()
        assert all(torch.equal(C, want[i]) for i in range(S) for C in out[i])
        w.release()


@pytest.mark.parametrize("qtype", [F.IQ4_XS, F.IQ4_NL])
@pytest.mark.parametrize("K,act32", [(256, True), (768, True), (1280, False)])
def test_four_row_tiles(qm, dev, qtype, K, act32):
    """Products of 1280 tiles of 128 x 128 and more (four row tiles per work-group for these types), the last row and column
    tile ragged, one superblock and odd numbers of them: parity on sampled columns, every accumulate mode, and block sums bit for
    bit on the first and last rows."""
    import torch
    M, N = 2047, 10256
    W = F.synth_weight(qtype, N, K, seed=qtype)
    x = F.synth_activations(M, K, seed=3, outlier_frac=0.01)
    aq, asc, absum = qm.quantize_act(to_dev(x, dev), M_stride=2048, act32=act32)
    w = qm.QWeight(qtype, to_dev(W, dev), N, K)
    C = qm.gemm(w, aq, asc, absum, M=M, act32=act32)
    g = torch.randn((M, N), device=dev)
    add = qm.gemm(w, aq, asc, absum, M=M, C=g.clone(), ldc=N, accumulate=1, act32=act32)
    mul = qm.gemm(w, aq, asc, absum, M=M, C=g.clone(), ldc=N, accumulate=2, act32=act32)
    assert torch.equal(add, g + C)
    assert torch.allclose(mul, torch.nn.functional.silu(g) * C, rtol=1e-5, atol=1e-6 * C.abs().max().item())
    C = C.cpu().numpy()
    isum = qm.gemm_blocksums(w, aq, M=M)
    a = (aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy())
    for r in (slice(0, 32), slice(N - 32, N)):
        if act32:
            ref, risum, _ = oracle.blockdot(qtype, W[r], K, *a, M=M, blocksums=True)
            assert np.array_equal(isum[:, r].cpu().numpy(), risum)
        else:
            ref = oracle.blockdot256(qtype, W[r], K, *a, M=M)
        assert rel_err(C[:, r], ref) < TOL_INT8_PATH
        assert_elementwise(C[:, r], ref)
