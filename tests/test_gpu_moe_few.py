"""MoE layers small enough for the fine-grained expert kernels, against the CPU oracle at the edges of their tiles."""
import numpy as np
import pytest

from arcinfer_amd import formats as F

from .test_gpu_moe import _moe_setup, moe_check, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("types", [(F.IQ4_XS, F.IQ4_XS, F.Q6_K), (F.Q6_K, F.Q6_K, F.Q8_0), (F.Q3_K, F.Q3_K, F.IQ2_S),
                                   (F.Q8_0, F.Q8_0, F.IQ3_S), (F.IQ2_XXS, F.IQ2_XXS, F.Q4_0)])
@pytest.mark.parametrize("E,Fd", [(768, 256), (256, 512)])  # (quads of gate / up: an uneven share per wave, fewer than waves)
def test_slot_tile_edges(qm, dev, types, E, Fd):
    """Experts of 1, 16, 17, 0, 32 and 33 slots: one and two token tiles, no slots, a second slot tile."""
    import torch
    NE, NU, sizes = 6, 1, [1, 16, 17, 0, 32, 33]
    T = sum(sizes)
    s = _moe_setup(qm, dev, NE, E, Fd, T, NU, types[0], seed=77, types=types)
    lg = np.full((T, NE), -5.0, dtype=np.float32)
    lg[np.arange(T), np.repeat(np.arange(NE), sizes)] = 5.0
    s["lg"], s["lgt"] = lg, to_dev(lg, dev)
    qm.moe_grouped(s["g"], s["u"], s["d"], NE, s["lgt"], NU, s["aq"], s["asc"], s["out"], s["ws"])
    torch.cuda.synchronize()
    moe_check(qm, s, types, NE, E, Fd, T, NU)


@pytest.mark.parametrize("types,E,Fd", [
    ((F.Q8_0, F.Q8_0, F.IQ4_XS), 256, 512),    # gate and up on the prompt kernels, down on the fine-grained one
    ((F.IQ4_XS, F.IQ3_S, F.IQ2_XXS), 256, 256),  # gate and up of two types, one launch each
    ((F.IQ4_XS, F.IQ4_XS, F.Q8_0), 512, 1024),  # the other way round
])
def test_one_product_of_the_two(qm, dev, types, E, Fd):
    NE, NU, T = 32, 2, 35
    s = _moe_setup(qm, dev, NE, E, Fd, T, NU, types[0], seed=5, types=types)
    qm.moe_grouped(s["g"], s["u"], s["d"], NE, s["lgt"], NU, s["aq"], s["asc"], s["out"], s["ws"])
    moe_check(qm, s, types, NE, E, Fd, T, NU)
