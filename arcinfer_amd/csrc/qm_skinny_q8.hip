// Few-token product instantiations for Q8_0, Q4_0; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_Q8_0>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q8_0>(bool, int, int, int);
template hipError_t skinny_dispatch<T_Q4_0>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q4_0>(bool, int, int, int);
}  // namespace qm
