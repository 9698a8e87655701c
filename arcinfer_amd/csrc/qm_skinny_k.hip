// Few-token product instantiations for Q4_K, Q5_K; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_Q4_K>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q4_K>(bool, int, int, int);
template hipError_t skinny_dispatch<T_Q5_K>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q5_K>(bool, int, int, int);
}  // namespace qm
