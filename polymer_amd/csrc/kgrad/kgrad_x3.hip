// Two-electron gradient kernels of bra pair class 3 (kgrad.h).
#include "../kgrad.h"

void polyeri_grad_row_launch_3(const GradArgs& gq, int Y, int x0, int y0, unsigned grid, size_t lds, double* d,
                               hipStream_t s) {
    grad_class_row<3>(Y, GradLaunch{gq, x0, y0, grid, lds, d, s});
}

void polyeri_grad_row_host_3(const GradArgs& gq, int Y, int x0, int y0, double* grad) {
    const RysTabs rt = host_tabs();
    grad_class_row<3>(Y, GradHostRun{gq, rt, x0, y0, grad});
}
