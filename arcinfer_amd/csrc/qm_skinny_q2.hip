// Few-token product instantiations for Q2_K; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_Q2_K>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q2_K>(bool, int, int, int);
}  // namespace qm
