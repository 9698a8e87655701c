// Few-token product instantiations for IQ1_S, IQ1_M; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_IQ1_S>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ1_S>(bool, int, int, int);
template hipError_t skinny_dispatch<T_IQ1_M>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ1_M>(bool, int, int, int);
}  // namespace qm
