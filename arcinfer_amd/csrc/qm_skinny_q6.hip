// Few-token product instantiations for Q6_K, Q3_K; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_Q6_K>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q6_K>(bool, int, int, int);
template hipError_t skinny_dispatch<T_Q3_K>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q3_K>(bool, int, int, int);
}  // namespace qm
