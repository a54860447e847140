// Generated by gen_eri.py -- do not edit.
#include "../eri_kernels.h"

EriKernel polyeri_kernel_2010(int mode) {
    switch (mode) {
    case 0: return k_eri<2, 0, 1, 0, 0>;
    case 1: return k_eri<2, 0, 1, 0, 1>;
    case 2: return k_eri<2, 0, 1, 0, 2>;
    case 3: return k_eri<2, 0, 1, 0, 3>;
    case 4: return k_eri<2, 0, 1, 0, 4>;
    case 5: return k_eri_seg<2, 0, 1, 0, false, true>;
    case 6: return k_eri_seg<2, 0, 1, 0, true, true>;
    case 7: return k_eri_seg<2, 0, 1, 0, true, false>;
    }
    return nullptr;
}
