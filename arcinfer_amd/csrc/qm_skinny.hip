// Few-token products: routes a weight type to its instantiation (qm_skinny_*.hip; kernels in qm_skinny_impl.h).
#include "qm_launch.h"

namespace qm {

template <int TYPE> hipError_t skinny_dispatch(const SkinnyArgs& a, hipStream_t s);
template <int TYPE> bool skinny_takes(bool prompt, int M, int rows, int K);

bool skinny_supported(int type, bool prompt, int M, int rows, int K) {
  switch (type) {
    case T_Q8_0: return skinny_takes<T_Q8_0>(prompt, M, rows, K);
    case T_Q4_0: return skinny_takes<T_Q4_0>(prompt, M, rows, K);
    case T_Q4_K: return skinny_takes<T_Q4_K>(prompt, M, rows, K);
    case T_Q5_K: return skinny_takes<T_Q5_K>(prompt, M, rows, K);
    case T_Q6_K: return skinny_takes<T_Q6_K>(prompt, M, rows, K);
    case T_Q3_K: return skinny_takes<T_Q3_K>(prompt, M, rows, K);
    case T_IQ4_XS: return skinny_takes<T_IQ4_XS>(prompt, M, rows, K);
    case T_IQ4_NL: return skinny_takes<T_IQ4_NL>(prompt, M, rows, K);
    case T_IQ3_S: return skinny_takes<T_IQ3_S>(prompt, M, rows, K);
    case T_IQ3_XXS: return skinny_takes<T_IQ3_XXS>(prompt, M, rows, K);
    case T_IQ2_XXS: return skinny_takes<T_IQ2_XXS>(prompt, M, rows, K);
    case T_IQ2_XS: return skinny_takes<T_IQ2_XS>(prompt, M, rows, K);
    case T_IQ2_S: return skinny_takes<T_IQ2_S>(prompt, M, rows, K);
    case T_Q2_0: return skinny_takes<T_Q2_0>(prompt, M, rows, K);
    case T_Q2_K: return skinny_takes<T_Q2_K>(prompt, M, rows, K);
    case T_IQ1_S: return skinny_takes<T_IQ1_S>(prompt, M, rows, K);
    case T_IQ1_M: return skinny_takes<T_IQ1_M>(prompt, M, rows, K);
    default: return false;
  }
}

hipError_t launch_skinny(int type, const SkinnyArgs& a, hipStream_t s) {
  switch (type) {
    case T_Q8_0: return skinny_dispatch<T_Q8_0>(a, s);
    case T_Q4_0: return skinny_dispatch<T_Q4_0>(a, s);
    case T_Q4_K: return skinny_dispatch<T_Q4_K>(a, s);
    case T_Q5_K: return skinny_dispatch<T_Q5_K>(a, s);
    case T_Q6_K: return skinny_dispatch<T_Q6_K>(a, s);
    case T_Q3_K: return skinny_dispatch<T_Q3_K>(a, s);
    case T_IQ4_XS: return skinny_dispatch<T_IQ4_XS>(a, s);
    case T_IQ4_NL: return skinny_dispatch<T_IQ4_NL>(a, s);
    case T_IQ3_S: return skinny_dispatch<T_IQ3_S>(a, s);
    case T_IQ3_XXS: return skinny_dispatch<T_IQ3_XXS>(a, s);
    case T_IQ2_XXS: return skinny_dispatch<T_IQ2_XXS>(a, s);
    case T_IQ2_XS: return skinny_dispatch<T_IQ2_XS>(a, s);
    case T_IQ2_S: return skinny_dispatch<T_IQ2_S>(a, s);
    case T_Q2_0: return skinny_dispatch<T_Q2_0>(a, s);
    case T_Q2_K: return skinny_dispatch<T_Q2_K>(a, s);
    case T_IQ1_S: return skinny_dispatch<T_IQ1_S>(a, s);
    case T_IQ1_M: return skinny_dispatch<T_IQ1_M>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace qm
