"""Products of 3 to 32 tokens (the few-token kernels behind qmatmul_gemv and qmatmul_gemm) against the CPU oracle: block sums
bit for bit from the instantiation that computes the product, f32 outputs within the parity bounds, where the route or a tile
can go wrong -- rows that end inside a 16-row tile, fewer quads than waves, a wave with one quad less than the others, token
counts at the edges of the 16-token tiles, and the sweep's first and last work-group shares."""
import numpy as np
import pytest

import oracle
from arcinfer_amd import formats as F

from .test_gpu_parity import GEMV_TYPES, TOL_INT8_PATH, acts, assert_elementwise, rel_err, to_dev

pytestmark = pytest.mark.gpu


def check(qm, dev, qtype, N, K, T, prompt):
    import torch
    W = F.synth_weight(qtype, N, K, seed=qtype + N + K)
    x = F.synth_activations(T, K, seed=N + K + T, outlier_frac=0.01)
    aq, asc, absum = acts(qm, x, dev, M_stride=(T + 15) // 16 * 16)
    w = qm.QWeight(qtype, to_dev(W, dev), N, K)
    base = torch.full((T, N + 24), 3.0, device=dev)
    C = base.clone()
    if prompt:
        qm.gemm(w, aq, asc, absum, M=T, C=C, ldc=N + 24, c_off=8, accumulate=1)
        isum, msum = qm.gemm_blocksums(w, aq, M=T), None
    else:
        qm.gemv(w, aq, asc, absum, T=T, C=C, ldc=N + 24, c_off=8, accumulate=1)
        isum, msum = qm.gemv_blocksums(w, aq, absum, T=T)
    torch.cuda.synchronize()
    ref, risum, rmsum = oracle.blockdot(qtype, W, K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=T,
                                        blocksums=True)
    assert np.array_equal(isum.cpu().numpy(), risum)
    if msum is not None:
        assert np.array_equal(msum.cpu().numpy(), rmsum)
    got = C[:, 8:8 + N].cpu().numpy()
    assert rel_err(got - 3.0, ref) < TOL_INT8_PATH
    # (3 + v rounds v to ulp(|3 + v|) / 2 <= 2^-23 max(3, |v|): below the element-wise floor of 1e-5 max|ref|)
    assert_elementwise(got, ref + 3.0)
    assert torch.equal(C[:, :8], base[:, :8]) and torch.equal(C[:, 8 + N:], base[:, 8 + N:])


@pytest.mark.parametrize("qtype", GEMV_TYPES)
@pytest.mark.parametrize("N,K,T", [(20, 256, 5), (40, 768, 8), (8200, 256, 5), (8200, 1280, 6), (33, 17408, 3)])
def test_decode(qm, dev, qtype, N, K, T):
    check(qm, dev, qtype, N, K, T, prompt=False)


@pytest.mark.parametrize("qtype", GEMV_TYPES)
@pytest.mark.parametrize("N,K,M", [(16, 256, 1), (48, 768, 16), (48, 1280, 17), (4112, 512, 9), (8208, 1280, 32), (8208, 2816, 16)])
def test_prompt(qm, dev, qtype, N, K, M):
    check(qm, dev, qtype, N, K, M, prompt=True)


@pytest.mark.parametrize("qtype", [F.IQ4_XS, F.Q5_K])
@pytest.mark.parametrize("N", [8208, 12304])
def test_sweep_five_quads_per_wave(qm, dev, qtype, N):
    check(qm, dev, qtype, N, 5120, 8, prompt=False)
    check(qm, dev, qtype, N, 4864, 23, prompt=True)


def test_prompt_fused_swiglu(qm, dev):
    """accumulate = 2: C = silu(C) * result."""
    import torch
    N, K, M = 64, 1024, 12
    W = F.synth_weight(F.IQ4_XS, N, K, seed=3)
    aq, asc, absum = acts(qm, F.synth_activations(M, K, seed=4), dev, M_stride=16)
    w = qm.QWeight(F.IQ4_XS, to_dev(W, dev), N, K)
    r = qm.gemm(w, aq, asc, absum, M=M)
    g = torch.linspace(-4, 4, M * N, device=dev).view(M, N)
    C = qm.gemm(w, aq, asc, absum, M=M, C=g.clone(), ldc=N, accumulate=2)
    torch.cuda.synchronize()
    assert torch.allclose(C, torch.nn.functional.silu(g) * r, rtol=1e-5, atol=1e-6 * r.abs().max().item())


@pytest.mark.parametrize("qtype", [F.Q8_0, F.Q4_K, F.Q6_K, F.IQ4_XS])
def test_long_rows_lose_no_precision(qm, dev, qtype):
    """Decode of 136 quads a row: root mean square of the error over that of the product. The GEMV these calls ran on before: 8.8e-8
    to 9.9e-8. Chains of four blocks and four quads in f32, then 64 bits and one rounding: 7e-8; the oracle's rounding of its
    double sums adds 3e-8 (in squares). One chain of 34 quads a wave: 1.27e-7."""
    N, K, T = 512, 17408, 5
    W = F.synth_weight(qtype, N, K, seed=qtype)
    aq, asc, absum = acts(qm, F.synth_activations(T, K, seed=9, outlier_frac=0.01), dev, M_stride=16)
    w = qm.QWeight(qtype, to_dev(W, dev), N, K)
    got = qm.gemv(w, aq, asc, absum, T=T).cpu().numpy().astype(np.float64)
    ref = oracle.blockdot(qtype, W, K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=T).astype(np.float64)
    assert np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2)) < 1e-7


@pytest.mark.parametrize("qtype", GEMV_TYPES)
@pytest.mark.parametrize("N,K,M", [(48, 768, 5), (4112, 1280, 16), (48, 1280, 17), (8208, 1280, 16), (8208, 1280, 32)])
def test_prompt_scales_per_256(qm, dev, qtype, N, K, M):
    """Per-256 activation scales (one scale row per eight blocks), on each of the kernels and both token tiles."""
    W = F.synth_weight(qtype, N, K, seed=qtype + N)
    aq, asc, absum = qm.quantize_act(to_dev(F.synth_activations(M, K, seed=M, outlier_frac=0.01), dev), M_stride=M, act32=False)
    w = qm.QWeight(qtype, to_dev(W, dev), N, K)
    got = qm.gemm(w, aq, asc, absum, M=M, act32=False).cpu().numpy()
    ref = oracle.blockdot256(qtype, W, K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=M)
    assert rel_err(got, ref) < TOL_INT8_PATH
    assert_elementwise(got, ref)
