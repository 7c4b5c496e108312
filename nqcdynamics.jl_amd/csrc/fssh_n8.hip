// fssh_n8.hip -- the five- to eight-state instantiations of the n-state FSSH / Ehrenfest kernel
// (fssh_n.hip), compiled as a translation unit of their own.
#include "fssh_n_kern.h"

namespace nqcd {

NQCD_NS_KERNELS(5)
NQCD_NS_KERNELS(6)
NQCD_NS_KERNELS(7)
NQCD_NS_KERNELS(8)

NsKernelPtr ns_kernel_hi(int NM, int precision, bool five) {
    switch (NM) {
    case 5: return NQCD_NS_PICK(5, precision, five);
    case 6: return NQCD_NS_PICK(6, precision, five);
    case 7: return NQCD_NS_PICK(7, precision, five);
    case 8: return NQCD_NS_PICK(8, precision, five);
    default: return nullptr;
    }
}

}  // namespace nqcd
