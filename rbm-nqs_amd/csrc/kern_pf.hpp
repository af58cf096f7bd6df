// kern_pf.hpp -- the Pfaffian factor of the wave function (pfaffian.cpp)
// for one Markov chain per wavefront, N <= 32 spins.
//
// Register layout.  Lane l holds row i = l & 31 of the inverse of the skew
// matrix A(sigma), columns 16h .. 16h + 15 with h = l >> 5: v[q] =
// inv(i, 16h + q).  Rows i >= N are zero.
//
// Per-wave LDS scratch, one region reused: the real or imaginary parts of a
// fresh FP64 inverse (N x (N + 1) doubles) while it is transposed, the
// Pfaffian derivative's sums, and for flip sets of more than two sites D (8 x
// 32) for the Delta-a rows and G (16 x 16) for the small 2m x 2m matrix.  Where
// log Pf is asked for (k_eval), the whole matrix (N x N complex double,
// column-major X[j*N + i]).
//
// Cross-lane traffic stays in registers: the 16 lanes of a DPP row read the
// value of lane q of their row by a row broadcast, rows and halves exchange by
// v_permlane16_swap / v_permlane32_swap, wave-uniform entries come by
// v_readlane.  The sampler was bound by the latency of the LDS round trips and
// fences of these exchanges, at one wavefront per SIMD (20 KB of scratch per
// wave); Kitaev 4x4 + Pfaffian, 8192 chains x 8 samples, FP32: 119.6 ms before,
// 49.1 ms now, VALU issue in 0.83 of the cycles, with the same sums in the same
// order (the chains are the same state for state).
//
// Ratio and update follow pfaffian.cpp:299-397 (Sherman-Morrison-Woodbury):
// for flips f_0..f_{m-1}, B = [Delta-a columns | unit columns e_{f_k}],
// Cinv' = Cinv0 + (G - G^T) / 2 with G = B^T inv B, ratio = sign Pf(Cinv'),
// and on acceptance inv += t2 - t2^T with t2 = (inv B) C (inv B)^T / 2,
// C = antisym(Cinv'^-1).
#pragma once
#include <type_traits>

#include "dev_common.hpp"

namespace rbmgpu {

constexpr int kPfMaxN = 32;
constexpr int kPfMaxM = 8;  // flips per ratio

// cross-lane LDS ordering within one wavefront
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// bytes of a wave's scratch; full: with room for pf_logpf's matrix
template <typename R>
__host__ __device__ inline size_t pf_scratch(int N, int rows, int full) {
    size_t b = (size_t)(8 * 32 + 16 * 16) * sizeof(cplx<R>) + 64;  // D, G, flip list
    const size_t t = (size_t)N * (N + 1) * sizeof(double), d = 4 * (size_t)rows * sizeof(cplx<R>);
    const size_t m = full ? (size_t)N * N * sizeof(cplx<double>) : 0;
    b = b > t ? b : t;
    b = b > d ? b : d;
    b = b > m ? b : m;
    return (b + 15) & ~(size_t)15;
}

template <typename R>
struct PfLds {
    const int16_t* bs;   // N x N, bs[i*N + j] = index-map entry b(i, j)
    const cplx<R>* fs;   // rows x 4: fs[r*4 + c]
    int N, rows;
    // this wave's scratch, by use
    cplx<R>* X;          // derivative sums
    double* Xr;          // N x (N + 1): one part of a matrix, entry (i, j) at j (N + 1) + i
    cplx<double>* Xd;    // N x N (scratch with room for it)
    cplx<R>* D;          // 8 x 32
    cplx<R>* G;          // 16 x 16, after D
    int* F;              // 16 ints after G: the flip list of the current ratio
};

__device__ inline int bit2(const uint64_t* st, int i) { return (int)((st[i >> 6] >> (i & 63)) & 1); }

// A_ij for spin bits si, sj (pfaffian.cpp:123-137)
template <typename R>
__device__ inline cplx<R> pf_a(const PfLds<R>& l, int i, int j, int si, int sj) {
    if (i == j) return {0, 0};
    int bb = l.bs[i * l.N + j];
    int sp = i > j ? (si << 1) | sj : (sj << 1) | si;
    cplx<R> v = l.fs[(abs(bb) - 1) * 4 + sp];
    return bb < 0 ? cplx<R>{-v.re, -v.im} : v;
}

template <typename R>
__device__ inline cplx<R> cdiv(cplx<R> a, cplx<R> b) {
    R d = 1 / (b.re * b.re + b.im * b.im);
    return {(a.re * b.re + a.im * b.im) * d, (a.im * b.re - a.re * b.im) * d};
}

// a b with the roundings of each part spelled out: an incremental inverse in
// FP32 is sensitive to the last bit (chains leave each other within an epoch),
// so the products here are not left to the compiler's choice of which product
// an FMA takes, and the order of their factors matters: pmul(a, b) and pmul(b,
// a) differ in the imaginary part
template <typename R>
__device__ inline cplx<R> pmul(cplx<R> a, cplx<R> b) {
    if constexpr (sizeof(R) == 4)
        return {__builtin_fmaf(a.re, b.re, -(a.im * b.im)), __builtin_fmaf(a.im, b.re, a.re * b.im)};
    else return {__builtin_fma(a.re, b.re, -(a.im * b.im)), __builtin_fma(a.im, b.re, a.re * b.im)};
}

// -a b; the real part rounds the product of the real parts
template <typename R>
__device__ inline cplx<R> pmuln(cplx<R> a, cplx<R> b) {
    if constexpr (sizeof(R) == 4)
        return {__builtin_fmaf(a.im, b.im, -(a.re * b.re)), -__builtin_fmaf(a.im, b.re, a.re * b.im)};
    else return {__builtin_fma(a.im, b.im, -(a.re * b.re)), -__builtin_fma(a.im, b.re, a.re * b.im)};
}

// 1 / a
template <typename R>
__device__ inline cplx<R> pinv(cplx<R> a) {
    R d;
    if constexpr (sizeof(R) == 4) d = 1 / __builtin_fmaf(a.re, a.re, a.im * a.im);
    else d = 1 / __builtin_fma(a.re, a.re, a.im * a.im);
    return {a.re * d, -a.im * d};
}

template <typename R>
__device__ inline cplx<R> shfl_c(cplx<R> v, int src) {
    return {__shfl(v.re, src), __shfl(v.im, src)};
}

// both halves of a value's 16-lane row pairs / 32-lane halves: (even row or
// low half, odd row or high half), the same in both partners
template <typename T>
struct Two {
    T lo, hi;
};
__device__ inline Two<uint32_t> swap16(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {r[0], r[1]};
}
__device__ inline Two<uint32_t> swap32(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {r[0], r[1]};
}
template <bool W32>
__device__ inline Two<float> swp(float v) {
    const Two<uint32_t> r = W32 ? swap32(__float_as_uint(v)) : swap16(__float_as_uint(v));
    return {__uint_as_float(r.lo), __uint_as_float(r.hi)};
}
template <bool W32>
__device__ inline Two<double> swp(double v) {
    const Two<uint32_t> a = W32 ? swap32((uint32_t)__double2loint(v)) : swap16((uint32_t)__double2loint(v));
    const Two<uint32_t> b = W32 ? swap32((uint32_t)__double2hiint(v)) : swap16((uint32_t)__double2hiint(v));
    return {__hiloint2double((int)b.lo, (int)a.lo), __hiloint2double((int)b.hi, (int)a.hi)};
}
template <bool W32, typename R>
__device__ inline Two<cplx<R>> swp(cplx<R> v) {
    const Two<R> a = swp<W32>(v.re), b = swp<W32>(v.im);
    return {{a.lo, b.lo}, {a.hi, b.hi}};
}
// lane n of each 16-lane row to the whole row
template <int n>
__device__ inline float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + n, 0xF, 0xF, false));
}
template <int n>
__device__ inline double row_bcast(double v) {
    return __longlong_as_double(__builtin_amdgcn_update_dpp(0LL, __double_as_longlong(v), 0x150 + n, 0xF, 0xF, false));
}
template <int n, typename R>
__device__ inline cplx<R> row_bcast(cplx<R> v) {
    return {row_bcast<n>(v.re), row_bcast<n>(v.im)};
}
// f(integral_constant<I>) .. f(integral_constant<n - 1>)
template <int I, int n, typename F>
__device__ __attribute__((always_inline)) inline void unroll_n(F&& f) {
    if constexpr (I < n) {
        f(std::integral_constant<int, I>{});
        unroll_n<I + 1, n>(f);
    }
}
// lane src (wave-uniform) of v as a wave-uniform value
__device__ inline float lane_of(float v, int src) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
__device__ inline double lane_of(double v, int src) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src),
                            __builtin_amdgcn_readlane(__double2loint(v), src));
}
template <typename R>
__device__ inline cplx<R> lane_of(cplx<R> v, int src) {
    return {lane_of(v.re, src), lane_of(v.im, src)};
}
// group_csum<32> with the last step by v_permlane16_swap: the same sums
template <typename R>
__device__ inline cplx<R> csum32(cplx<R> v) {
    v = group_csum<16>(v);
    const Two<cplx<R>> t = swp<false>(v);
    return t.lo + t.hi;
}

// wave argmax of key over lanes (ties: smaller lane); returns the lane
__device__ inline int wave_argmax(double key, int lane) {
    int best = lane;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        double k2 = __shfl_xor(key, o);
        int b2 = __shfl_xor(best, o);
        if (k2 > key || (k2 == key && b2 < best)) {
            key = k2;
            best = b2;
        }
    }
    return __builtin_amdgcn_readfirstlane(best);
}

// Xd = A(sigma) (column-major), all N x N entries, in FP64
template <typename R>
__device__ inline void pf_build(const PfLds<R>& l, const uint64_t* st, int lane) {
    const int N = l.N;
    for (int e = lane; e < N * N; e += 64) {
        int i = e % N, j = e / N;
        cplx<R> a = pf_a(l, i, j, bit2(st, i), bit2(st, j));
        l.Xd[e] = {(double)a.re, (double)a.im};
    }
    wave_sync();
}

// fresh FP64 inverse of A(sigma), antisymmetrised (pfaffian.cpp:284-297), into
// v: Gauss-Jordan with partial pivoting in registers, lane l holding row i = l
// & 31, columns 16h .. 16h + 15.  Rows stay in their lanes; pos is the row's
// place under the row swaps (ties between pivots go to the smaller place), the
// columns are unscrambled and the matrix transposed through LDS at the end, one
// part at a time.  Returns false if singular.
template <typename R>
__device__ inline bool pf_fresh(const PfLds<R>& l, const uint64_t* st, int lane, cplx<R> (&v)[16]) {
    const int N = l.N, i = lane & 31, h = lane >> 5;
    cplx<double> x[16];
    const int si = i < N ? bit2(st, i) : 0;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int j = 16 * h + q;
        x[q] = {0, 0};
        if (i < N && j < N) {
            const cplx<R> a = pf_a(l, i, j, si, bit2(st, j));
            x[q] = {(double)a.re, (double)a.im};
        }
    }
    bool ok = true;
    int pos = i, ip = i;  // ip: lane c holds the place swapped with place c
    for (int hc = 0; hc < 2; hc++)
        unroll_n<0, 16>([&](auto qc) __attribute__((always_inline)) {
            constexpr int q0 = decltype(qc)::value;
            const int c = 16 * hc + q0;
            if (c >= N) return;
            // column c of the lane's row, in both halves
            const Two<cplx<double>> t = swp<true>(x[q0]);
            const cplx<double> col = hc ? t.hi : t.lo;
            // pivot: the largest |X(row, c)|^2 at places >= c, the smallest place among equals
            double key = -1;
            if (i < N && pos >= c) key = col.re * col.re + col.im * col.im;
            double best = key;
            best = fmax(best, partner<1>(best));
            best = fmax(best, partner<2>(best));
            best = fmax(best, partner<4>(best));
            best = fmax(best, partner<8>(best));
            {
                const Two<double> m = swp<false>(best);
                best = fmax(m.lo, m.hi);
            }
            int p = i < N && pos >= c && (key == best || !(best == best)) ? pos : 64;
            p = min(p, partner<1>(p));
            p = min(p, partner<2>(p));
            p = min(p, partner<4>(p));
            p = min(p, partner<8>(p));
            {
                const Two<uint32_t> m = swap16((uint32_t)p);
                p = min((int)m.lo, (int)m.hi);
            }
            p = __builtin_amdgcn_readfirstlane(p < 64 ? p : c);
            const int prow = __builtin_ctzll(__ballot(pos == p));  // lane of the pivot row (low half)
            if (lane == c) ip = p;
            if (pos == c) pos = p;
            else if (i == prow) pos = c;
            const cplx<double> piv = lane_of(col, prow);
            if (piv.re == 0 && piv.im == 0) ok = false;
            const cplx<double> inv = cdiv(cplx<double>{1, 0}, piv);
            // the pivot row (with 1 at column c) times 1 / piv, then subtracted
            // from every other row (with 0 at column c)
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const cplx<double> r0 = lane_of(x[q], prow), r1 = lane_of(x[q], prow + 32);
                cplx<double> row = h ? r1 : r0;
                const bool at = q == q0 && h == hc;
                if (at) row = {1, 0};
                row = row * inv;
                const cplx<double> xq = at ? cplx<double>{0, 0} : x[q];
                x[q] = i == prow ? row : xq - col * row;
            }
        });
    // where column k (lane k) ends: swaps in reverse pivot order
    int loc = i;
    for (int c = N - 1; c >= 0; c--) {
        const int p = __builtin_amdgcn_readlane(ip, c);
        loc = loc == p ? c : loc == c ? p : loc;
    }
#pragma unroll
    for (int part = 0; part < 2; part++) {
        wave_sync();
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int c0 = __builtin_amdgcn_readlane(loc, q), c1 = __builtin_amdgcn_readlane(loc, 16 + q);
            if (i < N && 16 * h + q < N) l.Xr[(h ? c1 : c0) * (N + 1) + pos] = part ? x[q].im : x[q].re;
        }
        wave_sync();
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int j = 16 * h + q;
            R r = 0;
            if (i < N && j < N) r = (R)(0.5 * (l.Xr[j * (N + 1) + i] - l.Xr[i * (N + 1) + j]));
            if (part) v[q].im = r;
            else v[q].re = r;
        }
    }
    wave_sync();
    return ok;
}

// log Pf(A(sigma)) by Parlett-Reid on X (pfaffian10 of pfaffian.cpp:284-297;
// own restatement); returns (-inf, 0) for a singular or odd matrix
template <typename R>
__device__ inline cplx<double> pf_logpf(const PfLds<R>& l, const uint64_t* st, int lane) {
    pf_build(l, st, lane);
    const int N = l.N;
    cplx<double>* X = l.Xd;
    if (N & 1) return {-INFINITY, 0};
    double lre = 0, lim = 0;
    for (int k = 0; k + 1 < N; k += 2) {
        double key = -1;
        if (lane > k && lane < N) {
            cplx<double> x = X[lane * N + k];  // X(k, lane)
            key = (double)x.re * x.re + (double)x.im * x.im;
        }
        int kp = wave_argmax(key, lane);
        if (kp != k + 1) {
            if (lane < N) {  // rows k+1 <-> kp
                cplx<double> a = X[lane * N + k + 1], b = X[lane * N + kp];
                X[lane * N + k + 1] = b;
                X[lane * N + kp] = a;
            }
            wave_sync();
            if (lane < N) {  // columns k+1 <-> kp
                cplx<double> a = X[(k + 1) * N + lane], b = X[kp * N + lane];
                X[(k + 1) * N + lane] = b;
                X[kp * N + lane] = a;
            }
            wave_sync();
            lim += M_PI;  // sign flip
        }
        cplx<double> a = X[(k + 1) * N + k];
        if (a.re == 0 && a.im == 0) return {-INFINITY, 0};
        lre += 0.5 * ::log((double)a.re * a.re + (double)a.im * a.im);
        lim += ::atan2((double)a.im, (double)a.re);
        int n2 = N - k - 2;
        for (int e = lane; e < n2 * n2; e += 64) {
            int i = k + 2 + e % n2, j = k + 2 + e / n2;
            cplx<double> up = X[i * N + k + 1] * X[j * N + k] - X[i * N + k] * X[j * N + k + 1];
            X[j * N + i] = X[j * N + i] + cdiv(up, a);
        }
        wave_sync();
    }
    return {lre, lim};
}

// Pfaffian of the 2m x 2m skew matrix G (row-major, stride 16), m > 2 (the
// closed forms of one and two flips are pf_ratio2's), by Parlett-Reid in one
// lane (uniform result)
template <typename R>
__device__ inline cplx<R> small_pf(cplx<R>* G, int m, int lane) {
    cplx<R> pf{1, 0};
    if (lane == 0) {
        const int n = 2 * m;
        for (int k = 0; k + 1 < n; k += 2) {
            int kp = k + 1;
            R best = norm2(G[k * 16 + k + 1]);
            for (int i = k + 2; i < n; i++)
                if (norm2(G[k * 16 + i]) > best) best = norm2(G[k * 16 + i]), kp = i;
            if (kp != k + 1) {
                for (int i = 0; i < n; i++) {
                    cplx<R> t = G[i * 16 + k + 1];
                    G[i * 16 + k + 1] = G[i * 16 + kp];
                    G[i * 16 + kp] = t;
                }
                for (int i = 0; i < n; i++) {
                    cplx<R> t = G[(k + 1) * 16 + i];
                    G[(k + 1) * 16 + i] = G[kp * 16 + i];
                    G[kp * 16 + i] = t;
                }
                pf = cplx<R>{-pf.re, -pf.im};
            }
            cplx<R> a = G[k * 16 + k + 1];
            pf = pf * a;
            if (a.re == 0 && a.im == 0) break;
            for (int i = k + 2; i < n; i++)
                for (int j = k + 2; j < n; j++)
                    G[i * 16 + j] = G[i * 16 + j] +
                                    cdiv(G[(k + 1) * 16 + i] * G[k * 16 + j] - G[k * 16 + i] * G[(k + 1) * 16 + j], a);
        }
    }
    return shfl_c(pf, 0);
}

// The Woodbury pieces of one flip set.  KEEP keeps the columns of inv B of
// this lane's row (m <= 2) for a following accept.
template <typename R, bool KEEP>
struct PfProp {
    cplx<R> ib[KEEP ? 4 : 1];
    cplx<R> g[KEEP ? 6 : 1];  // upper triangle 01, 02, 03, 12, 13, 23 of Cinv' (m = 1: 01)
    int m;
};

// v[f & 15] of the half f >> 4, in both halves (f wave-uniform)
template <typename R>
__device__ inline cplx<R> pf_column(const cplx<R> (&v)[16], int f) {
    cplx<R> sel = v[0];
#pragma unroll
    for (int q = 1; q < 16; q++)
        if (q == (f & 15)) sel = v[q];
    const Two<cplx<R>> t = swp<true>(sel);
    return (f >> 4) ? t.hi : t.lo;
}
// value of lane (i, h) -> value of index 16 h + (lane & 15)
template <typename R>
__device__ inline cplx<R> to_half(cplx<R> v, int h) {
    const Two<cplx<R>> t = swp<false>(v);
    return h ? t.hi : t.lo;
}

// pf_ratio for one or two flipped sites f0 (, f1; -1: one), wave-uniform: the
// entries of G = B^T inv B that Cinv' reads, each formed as pf_ratio forms it
template <typename R, bool KEEP>
__device__ inline cplx<R> pf_ratio2(const PfLds<R>& l, const cplx<R> (&v)[16], const uint64_t* st, int f0, int f1,
                                    int lane, PfProp<R, KEEP>& pp) {
    const int N = l.N, i = lane & 31, h = lane >> 5;
    const bool two = f1 >= 0;
    const int s0 = bit2(st, f0), s1 = two ? bit2(st, f1) : 0;
    const int si = i < N ? bit2(st, i) : 0, sn = si ^ (i == f0 || i == f1);
    // Delta-a rows a(i, f; flipped) - a(i, f)
    cplx<R> d0{0, 0}, d1{0, 0};
    if (i < N && i != f0) d0 = pf_a(l, i, f0, sn, s0 ^ 1) - pf_a(l, i, f0, si, s0);
    if (two && i < N && i != f1) d1 = pf_a(l, i, f1, sn, s1 ^ 1) - pf_a(l, i, f1, si, s1);
    // columns inv Delta-a and inv e_f
    auto mv = [&](cplx<R> d) __attribute__((always_inline)) {
        const cplx<R> e = to_half(d, h);
        cplx<R> s{0, 0};
        unroll_n<0, 16>([&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value;
            s = s + pmul(v[q], row_bcast<q>(e));
        });
        const Two<cplx<R>> t = swp<true>(s);
        return t.lo + t.hi;
    };
    auto half = [](cplx<R> a, cplx<R> b) { return cplx<R>{(R)0.5 * (a.re - b.re), (R)0.5 * (a.im - b.im)}; };
    pp.m = two ? 2 : 1;
    const cplx<R> c0 = mv(d0);
    if (!two) {
        const cplx<R> e0 = pf_column(v, f0);
        cplx<R> g01 = half(csum32(pmul(e0, d0)), lane_of(c0, f0));
        g01.re -= 1;
        if constexpr (KEEP) {
            pp.ib[0] = c0;
            pp.ib[1] = e0;
            pp.ib[2] = pp.ib[3] = {0, 0};
            pp.g[0] = g01;
        }
        return {-g01.re, -g01.im};
    }
    const cplx<R> c1 = mv(d1);
    const cplx<R> e0 = pf_column(v, f0), e1 = pf_column(v, f1);
    cplx<R> g01 = half(csum32(pmul(c1, d0)), csum32(pmul(c0, d1)));
    cplx<R> g02 = half(csum32(pmul(e0, d0)), lane_of(c0, f0)), g03 = half(csum32(pmul(e1, d0)), lane_of(c0, f1));
    cplx<R> g12 = half(csum32(pmul(e0, d1)), lane_of(c1, f0)), g13 = half(csum32(pmul(e1, d1)), lane_of(c1, f1));
    const cplx<R> g23 = half(lane_of(e1, f0), lane_of(e0, f1));
    g02.re -= 1;
    g13.re -= 1;
    // pair entry Cinv0(1, 0) = a(f1, f0) - a(f1, f0; both flipped)
    g01 = g01 - (pf_a(l, f1, f0, s1, s0) - pf_a(l, f1, f0, s1 ^ 1, s0 ^ 1));
    if constexpr (KEEP) {
        pp.ib[0] = c0;
        pp.ib[1] = c1;
        pp.ib[2] = e0;
        pp.ib[3] = e1;
        pp.g[0] = g01;
        pp.g[1] = g02;
        pp.g[2] = g03;
        pp.g[3] = g12;
        pp.g[4] = g13;
        pp.g[5] = g23;
    }
    const cplx<R> pf = pmul(g01, g23) - pmul(g02, g13) + pmul(g03, g12);
    return {-pf.re, -pf.im};
}

// Pf(A(sigma')) / Pf(A(sigma)) for sigma' = sigma with the sites fl[i]
// (bit i of mask set, i < 8) flipped, in increasing i (uniform over the
// wave).  One or two sites by pf_ratio2, more through D and G in LDS.
template <typename R>
__device__ inline cplx<R> pf_ratio(const PfLds<R>& l, const cplx<R> (&v)[16], const uint64_t* st, const int* fl,
                                   int mask, int lane) {
    constexpr int NS = 8;  // flip slots
    const int N = l.N, i = lane & 31, h = lane >> 5;
    const int m = __builtin_popcount(mask);
    if (m <= 2) {
        int f0 = -1, f1 = -1;
#pragma unroll
        for (int t = 0; t < NS; t++)
            if ((mask >> t) & 1) {
                if (f0 < 0) f0 = fl[t];
                else f1 = fl[t];
            }
        PfProp<R, false> pp;
        return pf_ratio2<R, false>(l, v, st, __builtin_amdgcn_readfirstlane(f0), __builtin_amdgcn_readfirstlane(f1),
                                   lane, pp);
    }
    // compacted flip list (uniform) -> F
    if (lane == 0) {
        int k = 0;
#pragma unroll
        for (int t = 0; t < NS; t++)
            if ((mask >> t) & 1) l.F[k++] = fl[t];
    }
    wave_sync();
    int si = i < N ? bit2(st, i) : 0, fli = 0;
    for (int k = 0; k < m; k++) fli |= l.F[k] == i;
    // Delta-a rows: D[k][i] = a(i, f_k; flipped) - a(i, f_k)
    for (int k = 0; k < m; k++) {
        int f = l.F[k], sf = bit2(st, f);
        cplx<R> d{0, 0};
        if (i < N && i != f) d = pf_a(l, i, f, si ^ fli, sf ^ 1) - pf_a(l, i, f, si, sf);
        if (h == 0) l.D[k * 32 + i] = d;
    }
    wave_sync();
    // G = B^T inv B: column b < m is inv Delta-a_b, column m + b is inv e_{f_b}
    for (int b = 0; b < 2 * m; b++) {
        cplx<R> col;
        if (b < m) {
            cplx<R> s{0, 0};
#pragma unroll
            for (int q = 0; q < 16; q++) s = s + v[q] * l.D[b * 32 + 16 * h + q];
            col = {s.re + partner<32>(s.re), s.im + partner<32>(s.im)};
        } else {
            int f = l.F[b - m];
            cplx<R> sel{0, 0};
#pragma unroll
            for (int q = 0; q < 16; q++)
                if (q == (f & 15)) sel = v[q];
            cplx<R> oth{partner<32>(sel.re), partner<32>(sel.im)};
            col = (f >> 4) == h ? sel : oth;
        }
        for (int a = 0; a < m; a++) {
            // rows a < m: sum_i Delta-a_a(i) col(i); rows m + a: col(f_a)
            cplx<R> x = group_csum<32>(l.D[a * 32 + i] * col);
            int fa = __builtin_amdgcn_readfirstlane(l.F[a]);
            cplx<R> r{__shfl(col.re, fa), __shfl(col.im, fa)};
            if (lane == 0) {
                l.G[a * 16 + b] = x;
                l.G[(m + a) * 16 + b] = r;
            }
        }
    }
    wave_sync();
    // Cinv' = Cinv0 + (G - G^T) / 2: unit entries and the antisymmetric part
    const int n = 2 * m, nE = n * n;
    constexpr int NU = (2 * NS * 2 * NS + 63) / 64;
    cplx<R> g[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
        int e = lane + 64 * u;
        cplx<R> val{0, 0};
        if (e < nE) {
            int a = e / n, b = e % n;
            cplx<R> gab = l.G[a * 16 + b], gba = l.G[b * 16 + a];
            val = {(R)0.5 * (gab.re - gba.re), (R)0.5 * (gab.im - gba.im)};
            if (a >= m && b == a - m) val.re += 1;
            if (b >= m && a == b - m) val.re -= 1;
        }
        g[u] = val;
    }
    wave_sync();
#pragma unroll
    for (int u = 0; u < NU; u++) {
        int e = lane + 64 * u;
        if (e < nE) l.G[(e / n) * 16 + e % n] = g[u];
    }
    wave_sync();
    // pair entries Cinv0(k, q) = a(f_k, f_q) - a(f_k, f_q; both flipped), k > q
    if (lane == 0)
        for (int k = 1; k < m; k++)
            for (int q = 0; q < k; q++) {
                int fk = l.F[k], fq = l.F[q], sk = bit2(st, fk), sq = bit2(st, fq);
                cplx<R> c0 = pf_a(l, fk, fq, sk, sq) - pf_a(l, fk, fq, sk ^ 1, sq ^ 1);
                l.G[k * 16 + q] = l.G[k * 16 + q] + c0;
                l.G[q * 16 + k] = l.G[q * 16 + k] - c0;
            }
    wave_sync();
    cplx<R> pf = small_pf(l.G, m, lane);
    wave_sync();
    bool neg = ((m * (m + 1) / 2) & 1) != 0;
    return neg ? cplx<R>{-pf.re, -pf.im} : pf;
}

// accept the flip set of the last pf_ratio2<R, true>, whose Cinv' is in
// pp.g.  C = antisym(Cinv'^-1 / 2) = Cinv'^-1 for the skew Cinv', by
// the closed forms of the 2 x 2 and 4 x 4 skew inverses:
//   [[0, x], [-x, 0]]^-1 = [[0, -1/x], [1/x, 0]],
//   A^-1 = (1/Pf A) [[0, -a23, a13, -a12], [a23, 0, -a03, a02],
//                    [-a13, a03, 0, -a01], [a12, -a02, a01, 0]].
template <typename R>
__device__ inline void pf_accept(const PfLds<R>& l, cplx<R> (&v)[16], const PfProp<R, true>& pp, int lane) {
    const int m = pp.m, n = 2 * m, h = lane >> 5;
    // upper triangle c01, c02, c03, c12, c13, c23 of C
    cplx<R> c01, c02{0, 0}, c03{0, 0}, c12{0, 0}, c13{0, 0}, c23{0, 0};
    if (m == 1) {
        const cplx<R> ip = pinv(pp.g[0]);
        c01 = {-ip.re, -ip.im};
    } else {
        cplx<R> a01 = pp.g[0], a02 = pp.g[1], a03 = pp.g[2], a12 = pp.g[3], a13 = pp.g[4], a23 = pp.g[5];
        const cplx<R> ip = pinv(pmul(a01, a23) - pmul(a02, a13) + pmul(a03, a12));
        // times 1 / Pf; the products' rounding differs between the precisions
        auto by = [&](cplx<R> a) { return sizeof(R) == 4 ? pmul(ip, a) : pmul(a, ip); };
        auto byn = [&](cplx<R> a) { return cplx<R>{pmuln(a, ip).re, sizeof(R) == 4 ? pmuln(a, ip).im : -pmul(ip, a).im}; };
        c01 = byn(a23);
        c02 = by(a13);
        c03 = byn(a12);
        c12 = byn(a03);
        c13 = by(a02);
        c23 = byn(a01);
    }
    auto neg = [](cplx<R> x) { return cplx<R>{-x.re, -x.im}; };
    // t1 = (inv B) C for this lane's row
    cplx<R> t1[4];
    const cplx<R>(&ib)[4] = pp.ib;
    t1[0] = neg(pmul(ib[1], c01)) - pmul(c02, ib[2]) - pmul(c03, ib[3]);
    t1[1] = pmul(ib[0], c01) - pmul(c12, ib[2]) - pmul(c13, ib[3]);
    t1[2] = pmul(c02, ib[0]) + pmul(c12, ib[1]) - pmul(c23, ib[3]);
    t1[3] = pmul(c03, ib[0]) + pmul(c13, ib[1]) + pmul(c23, ib[2]);
    // inv(i, j) += (1/2) sum_b [t1(i, b) invB(j, b) - t1(j, b) invB(i, b)], the
    // rows j = 16 h + q of inv B and t1 by row broadcasts
    cplx<R> eb[4], et[4];
#pragma unroll
    for (int b = 0; b < 4; b++)
        if (b < n) {
            eb[b] = to_half(pp.ib[b], h);
            et[b] = to_half(t1[b], h);
        }
    auto update = [&](auto nc) __attribute__((always_inline)) {
        constexpr int nb = decltype(nc)::value;
        unroll_n<0, 16>([&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value;
            cplx<R> s{0, 0};
#pragma unroll
            for (int b = 0; b < nb; b++) {
                const cplx<R> tj = row_bcast<q>(et[b]);
                s = s + pmul(t1[b], row_bcast<q>(eb[b]));
                if (b < 3) {
                    const cplx<R> u = pmuln(ib[b], tj);
                    s = {s.re + u.re, s.im + u.im};
                } else s = s - pmul(ib[b], tj);
            }
            v[q] = v[q] + cplx<R>{(R)0.5 * s.re, (R)0.5 * s.im};
        });
    };
    if (m == 1) update(std::integral_constant<int, 2>{});
    else update(std::integral_constant<int, 4>{});
}

// d ln Pf / d fs (pfaffian.cpp:399-415) summed into out[n_pf] (this wave's
// accumulators in X, then written by the lanes)
template <typename R>
__device__ inline void pf_derivative(const PfLds<R>& l, const cplx<R> (&v)[16], const uint64_t* st, int lane,
                                     cplx<R>* out) {
    const int N = l.N, i = lane & 31, h = lane >> 5, npf = 4 * l.rows;
    wave_sync();
    for (int e = lane; e < npf; e += 64) l.X[e] = {0, 0};
    wave_sync();
    if (i < N) {
        int si = bit2(st, i);
#pragma unroll
        for (int q = 0; q < 16; q++) {
            int j = 16 * h + q;
            if (j < i) {
                int bb = l.bs[i * N + j];
                int idx = (abs(bb) - 1) + ((si << 1) | bit2(st, j)) * l.rows;
                cplx<R> x = v[q];
                if (bb > 0) x = {-x.re, -x.im};
                atomicAdd(&l.X[idx].re, x.re);
                atomicAdd(&l.X[idx].im, x.im);
            }
        }
    }
    wave_sync();
    for (int e = lane; e < npf; e += 64) out[e] = l.X[e];
    wave_sync();
}

}  // namespace rbmgpu
