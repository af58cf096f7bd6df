// kern_logpsi.hip -- log psi of given states (rbm_base.cpp:294-304,
// rbm_symmetry.cpp:138-147) without the Pfaffian factor, for rbmgpu_eval_logpsi.
//
// theta is a product of the +-1 spins (states x sites) with the weights (sites
// x units, gathered through the symmetry permutations), so it runs on
// v_mfma_f64_16x16x4_f64 / v_mfma_f32_16x16x4_f32: a block takes 16 states (the
// rows of a tile), its 4 waves the tiles of 16 units.  A group of lanes per
// state (k_eval) walks the sites one by one through dependent LDS reads.
//
// sum_h ln cosh theta_h: with E = exp(-2|x|), cosh(x + iy) = e^|x| p,
// p = ((1 + E) cos y, sgn(x) (1 - E) sin y) / 2, so the lane multiplies the p
// of its units and takes one logarithm and one arctangent per state instead of
// one per unit (and none of the logarithms' ln 2 cancels).  The sum of the
// principal arguments (what the sum of logarithms gives) is the argument of the
// product plus 2 pi per wrap, which the half planes of the two factors and of
// the product tell.  The product and the sums are FP64 in both precisions:
// against sums in 80 bits the error is 0.4 of k_eval's at weights of 0.05 and
// the same at 0.3 and 1.
//
// Bound by the exponentials and sines (some 200 FP64 operations per unit; VALU
// issue in 0.64 of the cycles).  Kitaev 6x6 symmetric alpha = 4 (288 units),
// 65 536 states, FP64: 1706 us by k_eval, 397 us; 37 states of Kitaev 4x4 basic
// alpha = 2 in FP32: the kernel 26 -> 9 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kern_api.hpp"

namespace rbmgpu {

template <typename R>
struct Tile;  // accumulator, product and the tile row of register r
template <>
struct Tile<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static __device__ acc mma(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ int row(int r, int g) { return 4 * r + g; }
};
template <>
struct Tile<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static __device__ acc mma(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ int row(int r, int g) { return 4 * g + r; }
};

// exp(-2a) - 1 for a >= 0, without cancellation
__device__ inline double em1_2(double a) { return ::expm1(-2 * a); }
__device__ inline float em1_2(float a) { return ::expm1f(-2 * a); }
__device__ inline void sc(double y, double& s, double& c) { ::sincos(y, &s, &c); }
__device__ inline void sc(float y, float& s, float& c) { ::sincosf(y, &s, &c); }

// the argument of (re, im) lies in (0, pi]
__device__ inline bool upper(double re, double im) { return im > 0 || (im == 0 && re < 0 && !signbit(im)); }

template <typename R>
__global__ void __launch_bounds__(64 * kLpWaves) k_logpsi(LogpsiArgs<R> a) {
    extern __shared__ __align__(16) char smem[];
    __shared__ double red[kLpWaves][16][2];
    static_assert(sizeof(red) == kLpStatic, "counted in the LDS budget");
    const int N = a.N, H = a.H, na = a.na, ns = a.ns;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    cplx<R>* Wl = reinterpret_cast<cplx<R>*>(smem);
    uint8_t* P = reinterpret_cast<uint8_t*>(Wl + (a.w_lds ? N * na : 0));
    if (a.w_lds)
        for (int i = threadIdx.x; i < N * na; i += 64 * kLpWaves) Wl[i] = a.W[i];
    if (ns > 1)
        for (int i = threadIdx.x; i < ns * N; i += 64 * kLpWaves) P[i] = a.perm[i];
    __syncthreads();
    const int tiles = (H + 15) / 16, steps = (N + 3) / 4;
    for (int64_t k0 = (int64_t)blockIdx.x * 16; k0 < a.n; k0 += (int64_t)gridDim.x * 16) {
        // the state of row n
        const int64_t ks = min(k0 + n, a.n - 1);
        const uint64_t w0 = a.states[ks * a.nw], w1 = a.nw > 1 ? a.states[ks * a.nw + 1] : 0;
        double pr[4], pi[4], lre[4];  // the product and sum |x| in FP64 in both precisions
        int wrap[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            pr[r] = 1;
            pi[r] = 0;
            lre[r] = 0;
            wrap[r] = 0;
        }
        for (int c = wv; c < tiles; c += kLpWaves) {
            const int u = 16 * c + n, uu = min(u, H - 1), al = uu % na, s = uu / na;
            const uint8_t* Ps = P + s * N;
            const cplx<R> hb = a.hb[al];
            typename Tile<R>::acc ur{hb.re, hb.re, hb.re, hb.re}, ui{hb.im, hb.im, hb.im, hb.im};
            for (int q = 0; q < steps; q++) {
                const int f = 4 * q + g, fc = min(f, N - 1);
                const int e = (ns > 1 ? (int)Ps[fc] : fc) * na + al;
                cplx<R> w = a.w_lds ? Wl[e] : a.W[e];
                if (f >= N) w = {0, 0};
                const R sg = (((f < 64 ? w0 : w1) >> (f & 63)) & 1) ? (R)-1 : (R)1;
                ur = Tile<R>::mma(sg, w.re, ur);
                ui = Tile<R>::mma(sg, w.im, ui);
            }
            if (u < H) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const R x = ur[r], ax = M<R>::fabs(x), em = em1_2(ax);
                    R sn, cs;
                    sc((R)ui[r], sn, cs);
                    const double qr = (1 + 0.5 * (double)em) * (double)cs;
                    const double qi = 0.5 * (double)M<R>::copysign(em, x) * (double)sn;  // em <= 0
                    const double nr = pr[r] * qr - pi[r] * qi, ni = pr[r] * qi + pi[r] * qr;
                    // both arguments in (0, pi] (or [-pi, 0)) and their sum past pi (-pi)
                    const bool both_neg = pr[r] < 0 && qr < 0;
                    if (upper(pr[r], pi[r]) && upper(qr, qi) && (both_neg || !upper(nr, ni))) wrap[r]++;
                    if (upper(pr[r], -pi[r]) && upper(qr, -qi) && (both_neg || !upper(nr, -ni))) wrap[r]--;
                    pr[r] = nr;
                    pi[r] = ni;
                    lre[r] += (double)ax;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const double re = group_sum<16>(lre[r] + 0.5 * ::log(pr[r] * pr[r] + pi[r] * pi[r]));
            const double im = group_sum<16>(::atan2(pi[r], pr[r]) + 6.283185307179586477 * wrap[r]);
            if (n == r) {
                red[wv][Tile<R>::row(r, g)][0] = re;
                red[wv][Tile<R>::row(r, g)][1] = im;
            }
        }
        // sum_f sigma_f c_f of row n over the lanes g
        double br = 0, bi = 0;
        if (wv == 0) {
            for (int f = g; f < N; f += 4) {
                const double sg = (((f < 64 ? w0 : w1) >> (f & 63)) & 1) ? -1.0 : 1.0;
                br += sg * (double)a.lb[f].re;
                bi += sg * (double)a.lb[f].im;
            }
            br += partner<16>(br);
            bi += partner<16>(bi);
            br += partner<32>(br);
            bi += partner<32>(bi);
        }
        __syncthreads();
        if (wv == 0 && g == 0 && k0 + n < a.n) {
            for (int v = 0; v < kLpWaves; v++) {
                br += red[v][n][0];
                bi += red[v][n][1];
            }
            a.logpsi[2 * (k0 + n)] = br;
            a.logpsi[2 * (k0 + n) + 1] = bi;
        }
        __syncthreads();
    }
}

template <typename R>
hipError_t launch_logpsi(LogpsiArgs<R> a, int n_cu, hipStream_t st) {
    if (a.n < 1 || a.N < 1 || a.H < 1 || a.nw > 2) return hipErrorInvalidValue;
    const size_t wb = (size_t)a.N * a.na * sizeof(cplx<R>), pb = a.ns > 1 ? (size_t)a.ns * a.N : 0;
    if (!logpsi_tables_fit(a.ns, a.N)) return hipErrorInvalidValue;
    a.w_lds = wb + pb <= kLpTables;  // else from memory (caches)
    const size_t lds = (a.w_lds ? wb : 0) + pb;
    const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(8, 163840 / (int64_t)(lds + kLpStatic)));
    const int64_t blocks = std::min<int64_t>((a.n + 15) / 16, per_cu * n_cu);
    hipLaunchKernelGGL(k_logpsi<R>, dim3((unsigned)blocks), dim3(64 * kLpWaves), lds, st, a);
    return hipGetLastError();
}
template hipError_t launch_logpsi<float>(LogpsiArgs<float>, int, hipStream_t);
template hipError_t launch_logpsi<double>(LogpsiArgs<double>, int, hipStream_t);

}  // namespace rbmgpu
