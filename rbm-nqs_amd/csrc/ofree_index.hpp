// ofree_index.hpp -- what k_sx_ofree (kern_impl.hpp) reads where: the rule on
// the machines it takes, its LDS, and the places of a lane's entries.  Plain
// C++, so that the ranges can be checked without a device
// (tests/test_ofree_index.py).
#pragma once
#include <stddef.h>
#ifdef __HIPCC__
#define RBM_HD __host__ __device__
#else
#define RBM_HD
#endif

namespace rbmgpu {

// rows per step: 4, or 2 where the accumulators leave no registers for more
// (blocks of 16 waves: 128 per lane; FP64 rows of over 1024 entries); rsize:
// bytes of a real
RBM_HD constexpr int of_rows(int rsize, int waves, int ld) {
    return waves == 16 || (rsize == 8 && ld > 1024) ? 2 : 4;
}
constexpr int kOfMaxN = 62;  // bit 62 of a masked state word is 0
// MODE: spins in both halves of the state word, in the low half, B32
constexpr int kOfWide = 0, kOfN32 = 1, kOfB32 = 2;
RBM_HD inline int of_mode(int N, int M) { return N > 32 ? kOfWide : N == 32 && M % 32 == 0 ? kOfB32 : kOfN32; }
RBM_HD inline int of_pad(int ld) { return (ld + 127) / 128 * 128; }
RBM_HD inline int of_xs(int ld, int npf) { return of_pad(ld) + (npf + 1) / 2 * 2; }
// LDS: x and the waves' rows, then two rows of sums
RBM_HD inline size_t of_lds(int rsize, int ld, int M, int npf, int waves) {
    const size_t loop = (size_t)of_xs(ld, npf) + (size_t)waves * of_rows(rsize, waves, ld) * (M + 1);
    return (loop > 2 * (size_t)ld ? loop : 2 * (size_t)ld) * 2 * rsize;
}
// basic RBMs whose pairs never straddle two units (even N and M), the biases
// within the first pair, at least two of the 4-wave blocks' LDS per CU
RBM_HD inline bool of_ok(int rsize, int N, int M, int ld, int npf, int waves) {
    return N <= kOfMaxN && N % 2 == 0 && M % 2 == 0 && N + M <= 128 &&
           of_lds(rsize, ld, M, npf, waves) <= (waves == 16 ? 163840 : 81920);
}

// A staged row holds the M tanh values and 1 at place M.  Pair 0 of a lane: the
// places e0, e1 of its entries and the spin ej of their signs (ej, ej + 1; 62:
// +1); pair 1: its unit u1 and spin j1.  Lanes past the last parameter read
// place M (times x = 0: what they read has to be finite).
struct OfLane {
    int e0, e1, ej, u1, j1;
};
RBM_HD inline OfLane of_lane(int lane, int N, int M) {
    const int q0 = 2 * lane - N - M, u0 = q0 / N, u1 = (q0 + 128) / N;
    OfLane o;
    o.e0 = q0 >= 0 ? (u0 < M ? u0 : M) : 2 * lane < N ? M : 2 * lane - N;
    o.e1 = q0 >= 0 ? o.e0 : 2 * lane < N ? M : 2 * lane - N + 1;
    o.ej = q0 >= 0 ? q0 - u0 * N : 2 * lane < N ? 2 * lane : 62;
    o.u1 = u1 < M ? u1 : M;
    o.j1 = (q0 + 128) % N;
    return o;
}
// from pair to pair 128 entries on: du = 128 / N units and dj = 128 % N spins
RBM_HD inline void of_next(int& u, int& j, int du, int dj, int N, int M) {
    u = u + du < M ? u + du : M;
    j += dj;
    if (j >= N) {
        j -= N;
        u = u + 1 < M ? u + 1 : M;
    }
}

}  // namespace rbmgpu
