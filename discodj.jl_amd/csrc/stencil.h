// Cell assignment and mass-assignment weights of the particle kernels (pm.jl:49-74): g = mod(x, L) / L * N with
// Julia's float mod, base cell floor(g) for even orders and round-half-even(g) for odd ones, weights of
// |g - cell|, every operation rounded as the reference rounds it (the library is built without contraction).
#pragma once

#include <hip/hip_runtime.h>

namespace dj {

// Julia's float mod(x, L) for L > 0.  On [-L, 2L) it is computed without fmod: there fmod returns x,
// x - L (exact, Sterbenz) or x (for -L < x < 0, then shifted by L), and every branch below gives
// the same bits as the general rule (rem, then + L for a negative remainder, +0 for a zero one).
// The three in-range cases are computed with the same operations and selected without branches;
// only positions outside [-L, 2L) take the general path.
template <typename T> __device__ __noinline__ T tjmod_general(T x, T L) {
    T r = fmod(x, L);
    if (r == (T)0) return copysign(r, L);
    if ((r > (T)0) != (L > (T)0)) return r + L;
    return r;
}
template <typename T> __device__ __forceinline__ T tjmod(T x, T L) {
    T r = x + (T)0;            // [0, L): + 0 turns -0 into +0, as copysign(0, L) does
    if (x >= L) r = x - L;     // [L, 2L)
    if (x < (T)0) r = x + L;   // [-L, 0)
    if (__builtin_expect(x < -L || x >= (T)2 * L, 0)) r = tjmod_general(x, L);
    return r;
}
// a mod n for a in [-n, 2n)
__device__ __forceinline__ int wrapn(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }
template <int W, typename T> __device__ __forceinline__ int twbase(T g) {
    return (W % 2 == 0) ? (int)floor(g) : (int)rint(g);
}
template <int W> __device__ __forceinline__ constexpr int twlo() { return W == 2 ? 0 : -1; }
__device__ __forceinline__ int timod(int a, int n) {
    int r = a % n;
    return r < 0 ? r + n : r;
}
// 1-D assignment weights (pm.jl:49-51).  Every piece is evaluated with the reference's operations
// and the applicable one selected, so the code has no branches and the values are the same bits.
template <int W, typename T> __device__ __forceinline__ T twk(T d) {
    if constexpr (W == 2) {
        const T a = (T)1 - d;
        return d > (T)1 ? (T)0 : a;
    } else if constexpr (W == 3) {
        const T t = (T)1.5 - d;
        const T outer = (T)0.5 * (t * t), inner = (T)0.75 - d * d;
        return d > (T)1.5 ? (T)0 : (d > (T)0.5 ? outer : inner);
    } else {
        const T t = (T)2 - d;
        const T outer = t * t * t / (T)6;
        const T inner = ((T)4 - (T)6 * (d * d) + (T)3 * (d * d * d)) / (T)6;
        return d > (T)2 ? (T)0 : (d > (T)1 ? outer : inner);
    }
}

// The weight of stencil cell o (0 <= o < W) at d = |g - (b + lo + o)|, b the base cell of g.  Each
// cell's d stays in one piece of the window, so only that piece is evaluated: TSC (b = round(g),
// |g - b| <= 1/2) has d <= 1/2 at the centre (inner piece) and 1/2 <= d <= 3/2 at the sides (outer
// piece; at d = 1/2 both pieces give 1/2 and at d = 3/2 the outer one gives the reference's 0); CIC
// (b = floor(g)) has d <= 1, where the weight is 1 - d.  The values are the same bits as twk's.
template <int W, typename T> __device__ __forceinline__ T twk_at(int o, T d) {
    if constexpr (W == 3) {
        if (o == 1) return (T)0.75 - d * d;
        const T t = (T)1.5 - d;
        return (T)0.5 * (t * t);
    } else if constexpr (W == 2) {
        return (T)1 - d;
    } else {
        return twk<W>(d);
    }
}

}  // namespace dj
