// FP64 instances of the VMC kernels (the parity mode).
#include "kern_launch.hpp"
namespace rbmgpu {
RBM_INSTANTIATE(double)
bool sx_ofree_ok(int real_size, int N, int M, int64_t ld, int npf) {
    const int w = sx_waves(ld);
    // (16-wave blocks have no instance for N >= 32, kOfWide none for the Pfaffian block)
    const int mode = of_mode(N, M);
    if ((w != 4 && mode != kOfN32) || (mode == kOfWide && npf > 0)) return false;
    return of_ok(real_size, N, M, (int)ld, npf, w);
}
}
