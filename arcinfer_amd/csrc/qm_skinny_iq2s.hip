// Few-token product instantiations for IQ2_S, Q2_0; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_IQ2_S>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ2_S>(bool, int, int, int);
template hipError_t skinny_dispatch<T_Q2_0>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_Q2_0>(bool, int, int, int);
}  // namespace qm
