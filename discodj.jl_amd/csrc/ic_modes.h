// Mode indexing of the IC pipeline's spectra (x-halved B layout B[kz + N (kx + H ky)]) and the amplitude
// phi(k) / w(k) of the white noise.
#pragma once

#include <hip/hip_runtime.h>

#include "dj_complex.h"

namespace dj {

struct BIdx {
    int kx, ky, kz;
};
__device__ __forceinline__ BIdx bidx(size_t e, int N) {
    const int H = N / 2 + 1;
    BIdx r;
    r.kz = (int)(e % N);
    size_t t = e / N;
    r.kx = (int)(t % H);
    r.ky = (int)(t / H);
    return r;
}
__device__ __forceinline__ int sgn_full(int m, int N) { return m < N / 2 ? m : m - N; }

// k along an axis of N modes with the Nyquist entry zeroed (nlpt_core.jl:49-67)
__device__ __forceinline__ double k_axis(int m, int N, double dk) {
    return m == N / 2 ? 0.0 : (double)sgn_full(m, N) * dk;
}

// phi(k) / w(k) = -sqrt(P(k) (n/L)^3) / k^2 (grf.jl:118-144, 190-216; P interpolated as np.interp, clamped; 0 at
// k = 0) depends on the squared length of the integer mode alone: a table over it, filled once per call
// (ic_amplitude_entry), serves every mode of the spectrum
inline size_t ic_amplitudes(int n) { return 3 * (size_t)(n / 2) * (n / 2) + 1; }
struct IcAmplitude {
    const double *tab;
    __device__ double operator()(const BIdx &b, int N) const {
        const int y = b.ky <= N / 2 ? b.ky : N - b.ky, z = b.kz <= N / 2 ? b.kz : N - b.kz;
        return tab[b.kx * b.kx + y * y + z * z];
    }
};
__device__ inline double ic_amplitude_entry(size_t m2, int N, double L, const double *kt, const double *pt, int ntab) {
    const double dk = 2 * M_PI / L, k2 = (double)m2 * (dk * dk);
    if (k2 == 0) return 0.0;
    const double k = sqrt(k2);
    double P;
    if (k <= kt[0]) P = pt[0];
    else if (k >= kt[ntab - 1]) P = pt[ntab - 1];
    else {
        int lo = 0, hi = ntab - 1;  // kt[lo] < k <= kt[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (kt[mid] < k) lo = mid; else hi = mid;
        }
        const double t = (k - kt[hi - 1]) / (kt[hi] - kt[hi - 1]);
        P = pt[hi - 1] * (1 - t) + pt[hi] * t;
    }
    const double rb = (double)N / L;
    return -sqrt(P * (rb * rb * rb)) / k2;
}

}  // namespace dj
