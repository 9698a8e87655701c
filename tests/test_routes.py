"""The dispatch rules of the dense and expert products (host code of the built library, no GPU): at shapes where each side was measured, the
call takes the faster one. Times in microseconds, whole call, one MI355X."""
import ctypes

import pytest

from arcinfer_amd import formats as F
from arcinfer_amd import qmatmul


class Split(ctypes.Structure):
    _fields_ = [("start", ctypes.c_int), ("splits", ctypes.c_int), ("bytes", ctypes.c_size_t), ("halves", ctypes.c_bool),
                ("us", ctypes.c_float)]


@pytest.fixture(scope="module")
def rules():
    lib = qmatmul.load_library()
    split = lib._ZN2qm14gemm_split_forEiiiib
    split.restype, split.argtypes = Split, [ctypes.c_int] * 4 + [ctypes.c_bool]
    f16 = lib._ZN2qm18f16_gemm_supportedEiiii
    f16.restype, f16.argtypes = ctypes.c_bool, [ctypes.c_int] * 4
    return split, f16


def deal(rules, qtype, M, N, K):
    split, f16 = rules
    use = f16(qtype, M, N, K)
    s = split(qtype, M, N, K, use)
    return ("f16 " if use else "") + ("cut %d" % s.splits if s.splits > 1 else "halves" if s.halves else "whole")


@pytest.mark.parametrize("qtype,M,N,K,want", [
    # cut tiles against K halves of the int8 kernel
    (F.IQ2_XXS, 341, 3776, 4096, "halves"),   # 36.6 against 41.4 cut in four
    (F.IQ2_XXS, 393, 3360, 3072, "halves"),   # 30.5, 36.4
    (F.IQ3_S, 71, 10896, 3072, "halves"),     # 32.8, 37.9
    (F.IQ1_S, 93, 8896, 2560, "halves"),      # 28.9, 33.0 in five
    (F.IQ2_XXS, 74, 6896, 9216, "halves"),    # 48.9, 53.0 in two
    (F.Q8_0, 384, 4352, 15616, "halves"),     # 101, 109 in five
    (F.Q8_0, 384, 4352, 12544, "halves"),     # 84, 93
    (F.Q8_0, 70, 5632, 10496, "cut 5") ,      # 46.2 in halves, 39.4
    (F.Q4_K, 120, 5888, 13056, "cut 5"),      # 68.8 in halves, 55.4
    (F.IQ4_XS, 339, 2048, 9472, "cut 5"),     # 50.1 in halves, 41.3
    (F.IQ4_XS, 1115, 5584, 8704, "cut 3"),    # 792 tiles, whole 238, 216
    # whole tiles against halves: more than one tile per CU
    (F.IQ4_XS, 142, 15312, 3072, "halves"),   # 46.6 against 48.5 whole: a nearly empty token tile's halves cost little
    (F.IQ3_S, 133, 14368, 3072, "halves"),    # 52.0, 54.1
    (F.Q5_K, 777, 4096, 4096, "whole"),       # 93 in halves, 75
    (F.Q8_0, 1005, 3328, 2304, "whole"),      # 52.8 in halves, 34.6
    # the f16 kernel against int8
    (F.Q5_K, 1167, 13120, 1792, "whole"),     # 142, 146 on f16: a third round of six tiles
    (F.Q5_K, 333, 5120, 17408, "f16 cut 4"),  # 157 on int8, 143
    (F.Q5_K, 2048, 17408, 5120, "f16 whole"), # 773, 697
    (F.IQ3_S, 512, 5120, 5120, "f16 cut 3"),  # 78, 73
])
def test_prompt_products(rules, qtype, M, N, K, want):
    assert deal(rules, qtype, M, N, K) == want


@pytest.mark.parametrize("qtype,slots,NE,E,Fd,want", [
    # gate and up on the fine-grained kernels (whole layer, prompt kernels' time against theirs)
    (F.IQ4_XS, 330, 8, 2048, 512, True),    # 91, 57
    (F.Q6_K, 118, 8, 1792, 256, True),      # 107, 48
    (F.IQ4_XS, 268, 128, 2048, 256, True),  # 78, 59
    (F.Q6_K, 222, 64, 4096, 512, False),    # 155, 183
    (F.IQ2_XXS, 318, 64, 2048, 512, False), # 84, 86
    (F.IQ2_XXS, 1812, 8, 2048, 512, False), # 78, 87
    (F.IQ2_S, 72, 64, 2816, 512, True),     # 110, 71
    (F.Q8_0, 96, 32, 2048, 512, False),     # 67, 73
    (F.Q8_0, 108, 64, 2048, 512, False),    # 68, 81
    (F.Q8_0, 198, 64, 4096, 256, False),    # 87, 93
    (F.Q8_0, 660, 64, 1024, 256, False),    # 61, 63
])
def test_expert_gate_up(qtype, slots, NE, E, Fd, want):
    few = qmatmul.load_library()._ZN2qm7moe_fewEiiiii
    few.restype = ctypes.c_bool
    assert few(qtype, slots, NE, E, Fd) == want


@pytest.mark.parametrize("qtype,slots,NE,E,Fd,want", [
    (F.IQ4_XS, 160, 32, 1024, 512, True),    # 66, 52
    (F.IQ3_S, 164, 8, 1280, 1024, True),     # 72, 65
    (F.IQ4_XS, 1302, 32, 4096, 512, False),  # 137, 144
    (F.Q8_0, 220, 32, 2048, 1024, False),    # 90, 111
    (F.Q8_0, 752, 128, 2048, 256, False),    # 98, 126
    (F.Q8_0, 624, 64, 2048, 512, False),     # 90, 116
    (F.Q6_K, 384, 64, 2048, 512, False),     # 94, 106
    (F.Q6_K, 542, 32, 2048, 768, False),     # 140, 149
])
def test_expert_down(qtype, slots, NE, E, Fd, want):
    few = qmatmul.load_library()._ZN2qm12moe_few_downEiiiii
    few.restype = ctypes.c_bool
    assert few(qtype, slots, NE, E, Fd) == want


@pytest.mark.parametrize("qtype,M,N,K,want", [
    # prompts of up to 32 tokens on the few-token kernels (the prompt kernel's time against theirs)
    (F.Q8_0, 12, 6016, 5376, True),     # 19.1, 11.2
    (F.Q8_0, 30, 11376, 3072, True),    # 14.6, 11.9
    (F.Q8_0, 9, 10400, 4864, True),     # 17.8, 14.0
    (F.Q8_0, 9, 22672, 7424, True),     # 41.9, 35.8
    (F.Q8_0, 28, 13296, 3584, False),   # 16.5, 19.3
    (F.Q8_0, 20, 15504, 3584, False),   # 16.7, 18.9
    (F.Q8_0, 4, 15600, 4608, False),    # 17.8, 19.7
    (F.Q8_0, 9, 9792, 8192, False),     # 25.0, 33.8
    (F.Q8_0, 5, 12640, 11264, False),   # 32.8, 43.1
    (F.Q8_0, 31, 4560, 4096, False),    # 15.3, 17.6
    (F.IQ4_XS, 13, 9952, 7168, True),
    (F.Q6_K, 32, 17408, 17408, True),
])
def test_few_token_prompts(qtype, M, N, K, want):
    takes = qmatmul.load_library()._ZN2qm16skinny_supportedEibiii
    takes.restype, takes.argtypes = ctypes.c_bool, [ctypes.c_int, ctypes.c_bool] + [ctypes.c_int] * 3
    assert takes(qtype, True, M, N, K) == want
