// Few-token product instantiations for IQ4_XS, IQ4_NL; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_IQ4_XS>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ4_XS>(bool, int, int, int);
template hipError_t skinny_dispatch<T_IQ4_NL>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ4_NL>(bool, int, int, int);
}  // namespace qm
