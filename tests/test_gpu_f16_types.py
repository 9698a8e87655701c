"""Precision of the f16-pipe GEMM of Q5_K, whose shorter products take the int8 kernels: on inputs where a rounded operand or sum
shows, its error against the oracle (sums in double) is no larger than the int8 kernel's on the same call."""
import numpy as np
import pytest

import oracle
from arcinfer_amd import formats as F

from .test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu


def _zero_mean(N, K, seed):
    """Q5_K rows whose min term is the mean of their values (mn = sc, dmin = 15.5 d): with activations of one sign the products
    and the min terms are each about sqrt(K) times the result."""
    W = F.synth_weight(F.Q5_K, N, K, seed=seed).reshape(-1, F.SB_BYTES[F.Q5_K])
    W[:, 8:12] = W[:, 4:8]  # (scales and mins: the low six bits, then both high parts from one nibble)
    lo = np.random.default_rng(seed).integers(0, 16, size=(len(W), 4), dtype=np.uint8)
    W[:, 12:16] = lo | (lo << 4)
    d = W[:, 0:2].copy().view(np.float16).astype(np.float32)
    W[:, 2:4] = (15.5 * d).astype(np.float16).view(np.uint8)
    return W.reshape(N, -1)


def _largest(N, K, seed):
    """Q5_K rows of the largest values (31) and the largest scales (63): superblock sums past 2^24."""
    W = F.synth_weight(F.Q5_K, N, K, seed=seed).reshape(-1, F.SB_BYTES[F.Q5_K])
    W[:, 4:16] = 0xFF
    W[:, 16:] = 0xFF
    return W.reshape(N, -1)


@pytest.mark.parametrize("act32", [True, False])
@pytest.mark.parametrize("rows", [_zero_mean, _largest])
def test_q5_k_error_is_the_int8_kernels(qm, dev, rows, act32):
    import torch
    M, N, K = 500, 4624, 5376
    W = rows(N, K, seed=3)
    x = 1.0 + 0.1 * F.synth_activations(M, K, seed=4)
    aq, asc, absum = qm.quantize_act(to_dev(x, dev), M_stride=M, act32=act32)
    w = qm.QWeight(F.Q5_K, to_dev(W, dev), N, K)
    assert qm.gemm_workspace_size(w, M) > 2 * M * K  # (the f16 kernel)
    C = qm.gemm(w, aq, asc, absum, M=M, act32=act32)
    D = qm.gemm_ws(w, aq, asc, absum, None, M=M, act32=act32)  # (the int8 kernel)
    torch.cuda.synchronize()
    blockdot = oracle.blockdot if act32 else oracle.blockdot256
    sel = np.arange(0, N, 37)
    ref = blockdot(F.Q5_K, W[sel], K, aq.cpu().numpy(), asc.cpu().numpy(), absum.cpu().numpy(), M=M)
    rms = [float(np.sqrt(np.mean((t.cpu().numpy()[:, sel] - ref.astype(np.float64)) ** 2) / np.mean(ref.astype(np.float64) ** 2)))
           for t in (C, D)]
    print("relative error: f16 %.3g, int8 %.3g" % tuple(rms))
    assert rms[0] <= rms[1]
