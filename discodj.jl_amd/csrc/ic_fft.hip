// The transforms of the IC pipeline and of its reverse, in FP64, between spectra on the particle grid (n) and
// real fields on it or on the de-aliased grid (ext = 3 n / 2).
//
// Every field here is a scalar spectrum times at most two factors i k_a: psi_c = c2r(-(i k_c) S), and the six
// distinct second derivatives A_ik = A_ki = c2r_ext(k_i k_k pad(phi)) of phi (nlpt_fast.jl:27-64 forms nine).
// A factor i k_a commutes with the transforms along the other axes, so it is applied by the pass along axis a,
// and the fields share their passes: for the A_ik one z pass writes three spectra (k_z^0, k_z^1, k_z^2), their
// y passes write six, and one x pass forms the source mu from the six real lines that its workgroup holds
// (all ICs at n = 256: 8.2 ms with nine stored fields of three passes each over the whole padded spectrum,
// 3.4 so).  The reverse runs the same tree backwards, each pass adding the spectra that the forward split.
//
// A pad has non-zero modes only for |k| < n/2: the spectra between the passes are stored without the rest.
//   line spectra  S[z + N line], line = kx + HX ky': HX = n/2 (pad) or n/2 + 1, ky' the n grid's index
//   after y       Y[y + N (kx + HX z)]
// The y and z passes are bound by HBM traffic, the x passes of the de-aliased grid by their transforms (VALU 46 %,
// LDS 29 % of the time); a workgroup's tile, line groups and block order are those of the mesh
// transforms (fft_shape.h).
#include <hip/hip_runtime.h>

#include "dj_internal.h"
#include "fft_shape.h"
#include "ic_modes.h"

namespace dj {

namespace {

using cd = cx<double>;
struct IcOut {
    cd *p[6];
};
struct IcIn {
    const cd *p[6];
};
// the power of k_x in the spectra of A11, A22, A33, A12, A13, A23
__device__ __forceinline__ int second_power(int f) { return f == 0 ? 2 : f == 3 || f == 4 ? 1 : 0; }

// The thread's index, opaque to the compiler: what a round of a kernel's loop derives from it (indexes, twiddles) is
// computed in that round.  Taken out of the loop as invariant it costs up to 150 registers, and with them all but
// one workgroup of a CU (the x pass of mu at n = 256, then with the fields
// stored: 2.4 ms against 1.6).  The x kernels keep the twiddles in LDS: through the caches, four twiddle loads to one of
// data, that pass took 1.15 ms, 1.01 so, and the x passes of its reverse 2.3, 1.75.
__device__ __forceinline__ int round_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// all lines of a workgroup's y/z tile, between workgroup barriers
template <int N, int DIR> __device__ __forceinline__ void yz_lines(cd *lds, const cd *t, int tid) {
    using EF = typename FftShape<double, N>::PY::EF;
    __syncthreads();
    if constexpr (EF::wave_ok()) EF::template run_wave<DIR, 1>(lds, t, tid);
    else EF::template run<DIR, 1>(lds, t, tid);
    __syncthreads();
}
// all packed real lines of a workgroup's x tile
template <int N, int DIR> __device__ __forceinline__ void x_lines(cd *lds, const cd *t, int tid) {
    using EX = typename FftShape<double, N>::P::EX;
    __syncthreads();
    if constexpr (EX::wave_ok()) EX::template run_wave<DIR, 2>(lds, t, tid);
    else EX::template run<DIR, 2>(lds, t, tid);
    __syncthreads();
}
__device__ __forceinline__ double power(double k, int r) { return r == 0 ? 1.0 : r == 1 ? k : k * k; }

// the n-grid index of mode m of an N grid whose modes are those of the n grid padded with zeros (-1: a zero)
template <int N, int n> __device__ __forceinline__ int band(int m) {
    if constexpr (N == n) return m;
    else return m < n / 2 ? m : (m > N - n / 2 ? m - N + n : -1);
}

// Inverse z pass: out[p] = inverse z of k_z^p src(line, kz), p < NOUT
template <int N, int NOUT, typename SRC>
__global__ __launch_bounds__((FftShape<double, N>::NTY), 2) void k_ic_zi(SRC src, IcOut out, const cd *__restrict__ tw,
                                                                     double dk) {
    using S = FftShape<double, N>;
    using EF = typename S::PY::EF;
    constexpr int NT = S::NTY, TOTAL = S::B * N, CNT = (TOTAL + NT - 1) / NT;
    __shared__ cd lds[EF::LDS_ELEMS];
    __shared__ cd twl[S::TWL ? N : 1];
    const cd *t = stage_twiddles<double, N, S::TWL>(tw, twl, threadIdx.x, NT);
    const size_t l0 = (size_t)blockIdx.x * S::B;
    cd v[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = threadIdx.x + c * NT;
        if (TOTAL % NT == 0 || i < TOTAL) v[c] = src(l0 + i / N, i % N);
    }
#pragma unroll 1
    for (int p = 0; p < NOUT; p++) {
        const int tid = round_tid();
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL)
                lds[EF::idx(i / N, i % N)] = v[c];
            v[c] = scale(v[c], k_axis(i % N, N, dk));
        }
        yz_lines<N, +1>(lds, t, tid);
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL) out.p[p][l0 * N + i] = lds[EF::idx(i / N, i % N)];
        }
        __syncthreads();
    }
}

// Inverse y pass of the line spectra in (HX kx values, the modes of an n grid along y): out[q] = inverse y of
// k_y^q in, q < NOUT
template <int N, int n, int HX, int NOUT>
__global__ __launch_bounds__((FftShape<double, N>::NTY), 2) void k_ic_yi(const cd *__restrict__ in, IcOut out,
                                                                     const cd *__restrict__ tw, double dk) {
    using S = FftShape<double, N>;
    using EF = typename S::PY::EF;
    constexpr int B = S::B, NT = S::NTY, TOTAL = B * N, CNT = (TOTAL + NT - 1) / NT;
    __shared__ cd lds[EF::LDS_ELEMS];
    __shared__ cd twl[S::TWL ? N : 1];
    const cd *t = stage_twiddles<double, N, S::TWL>(tw, twl, threadIdx.x, NT);
    const int lb = xcd_block(blockIdx.x, gridDim.x), zb = lb % (N / B), kx = lb / (N / B);
    cd v[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = threadIdx.x + c * NT, ky = band<N, n>(i / B);
        v[c] = cd{0, 0};
        if ((TOTAL % NT == 0 || i < TOTAL) && ky >= 0)
            v[c] = in[(size_t)(zb * B + i % B) + (size_t)N * ((size_t)kx + (size_t)HX * ky)];
    }
#pragma unroll 1
    for (int q = 0; q < NOUT; q++) {
        const int tid = round_tid();
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL)
                lds[EF::idx(i % B, i / B)] = v[c];
            v[c] = scale(v[c], k_axis(i / B, N, dk));
        }
        yz_lines<N, +1>(lds, t, tid);
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL)
                out.p[q][(size_t)(i % N) + (size_t)N * ((size_t)kx + (size_t)HX * (zb * B + i / N))] =
                    lds[EF::idx(i / N, i % N)];
        }
        __syncthreads();
    }
}

// the workgroup's lines of an after-y spectrum, times k_x^r, ready for the packed real inverse in lds
template <int N, int HX>
__device__ __forceinline__ void x_load(const cd *__restrict__ in, cd *lds, const cd *tw, int yb, int z, int r, double dk,
                                       int tid) {
    using P = typename FftShape<double, N>::P;
    constexpr int B = FftShape<double, N>::B, NT = FftShape<double, N>::NT, NC = N / 2, TOTAL = B * (NC / 2 + 1);
    cd va[P::XI_CNT], vb[P::XI_CNT];
#pragma unroll
    for (int c = 0; c < P::XI_CNT; c++) {
        const int i = tid + c * NT;
        va[c] = vb[c] = cd{0, 0};
        if (!(TOTAL % NT == 0 || i < TOTAL)) continue;
        const int k = i / B, m = NC - k;
        const size_t row = (size_t)(yb * B + i % B) + (size_t)N * ((size_t)HX * z);
        if (k < HX) va[c] = scale(in[row + (size_t)N * k], power(k_axis(k, N, dk), r));
        if (m < HX) vb[c] = scale(in[row + (size_t)N * m], power(k_axis(m, N, dk), r));
    }
    P::xi_pre(lds, tw, tid, va, vb);
}

// Inverse x pass: the real field out = s c2r_x(k_x^r in)
template <int N, int HX, typename T>
__global__ __launch_bounds__((FftShape<double, N>::NT), 4) void k_ic_xi(const cd *__restrict__ in, int r, double s, T *__restrict__ out,
                                               const cd *__restrict__ tw, double dk) {
    using S = FftShape<double, N>;
    using EX = typename S::P::EX;
    constexpr int B = S::B, NC = N / 2, TOTAL = B * NC;
    __shared__ cd lds[EX::LDS_ELEMS];
    __shared__ cd twl[N];
    const cd *t = stage_twiddles<double, N, true>(tw, twl, threadIdx.x, S::NT);
    __syncthreads();
    const int lb = xcd_block(blockIdx.x, gridDim.x), yb = lb % (N / B), z = lb / (N / B);
    const int tid = threadIdx.x;
    x_load<N, HX>(in, lds, t, yb, z, r, dk, tid);
    x_lines<N, +1>(lds, t, tid);
    const size_t base = (size_t)N * N * z + (size_t)N * yb * B;
    for (int i = threadIdx.x; i < TOTAL; i += S::NT) {
        const cd v = lds[EX::idx(i / NC, i % NC)];
        *(cx<T> *)(out + (base + 2 * (size_t)i)) = cx<T>{(T)(v.x * s), (T)(v.y * s)};
    }
}

// Inverse x pass of the six spectra of A11, A22, A33, A12, A13, A23 (k_x powers 2, 0, 0, 1, 1, 0; each field s times
// its transform) and the 2LPT source from them, mu = (A11 A22 + A11 A33 + A22 A33 - A12^2 - A13^2 - A23^2) smu.
// The fields are not stored (at n = 256 that took 0.35 ms): the reverse forms them again from the kept spectra,
// which it reads in less time than the fields, in the pass that needs them.
template <int N, int HX>
__global__ __launch_bounds__((FftShape<double, N>::NT), 3) void k_ic_xi_mu(IcIn in, double s, double smu,
                                                                              double *__restrict__ mu,
                                                                              const cd *__restrict__ tw, double dk) {
    using S = FftShape<double, N>;
    using EX = typename S::P::EX;
    constexpr int B = S::B, NC = N / 2, TOTAL = B * NC, CNT = (TOTAL + S::NT - 1) / S::NT;
    __shared__ cd lds[EX::LDS_ELEMS];
    __shared__ cd twl[N];
    const cd *t = stage_twiddles<double, N, true>(tw, twl, threadIdx.x, S::NT);
    __syncthreads();
    const int lb = xcd_block(blockIdx.x, gridDim.x), yb = lb % (N / B), z = lb / (N / B);
    const size_t base = (size_t)N * N * z + (size_t)N * yb * B;
    // one field's code six times over (unrolled it takes twice the registers): g = A11, A11 + A22 meets the next
    // diagonal field in m
    cd g[CNT], m[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) g[c] = m[c] = cd{0, 0};
#pragma unroll 1
    for (int f = 0; f < 6; f++) {
        const int tid = round_tid();
        x_load<N, HX>(in.p[f], lds, t, yb, z, second_power(f), dk, tid);
        x_lines<N, +1>(lds, t, tid);
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * S::NT;
            if (!(TOTAL % S::NT == 0 || i < TOTAL)) continue;
            const cd v = scale(lds[EX::idx(i / NC, i % NC)], s);
            if (f < 3) {
                m[c] = cd{m[c].x + g[c].x * v.x, m[c].y + g[c].y * v.y};
                g[c] = g[c] + v;
            } else {
                m[c] = cd{m[c].x - v.x * v.x, m[c].y - v.y * v.y};
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = threadIdx.x + c * S::NT;
        if (TOTAL % S::NT == 0 || i < TOTAL) *(cd *)(mu + (base + 2 * (size_t)i)) = scale(m[c], smu);
    }
}

// the lines in lds after the packed real forward, unpacked and times k_x^r, to an after-y spectrum
template <int N, int HX>
__device__ __forceinline__ void x_store(const cd *lds, cd *out, const cd *tw, int yb, int z, int r, double dk, int tid) {
    using S = FftShape<double, N>;
    using EX = typename S::P::EX;
    constexpr int B = S::B, NC = N / 2;
    for (int i = tid; i < B * HX; i += S::NT) {
        const int kx = i / B, l = i % B;
        const cd z1 = lds[EX::idx(l, kx == NC ? 0 : kx)], z2 = conj(lds[EX::idx(l, kx == 0 ? 0 : NC - kx)]);
        const cd e = scale(z1 + z2, 0.5), d = z1 - z2, o = {d.y * 0.5, -d.x * 0.5};
        out[(size_t)(yb * B + l) + (size_t)N * ((size_t)kx + (size_t)HX * z)] =
            scale(e + cmul(o, tw[kx]), power(k_axis(kx, N, dk), r));
    }
}

// Forward x pass of NF real fields (src(f, g): the values g, g + 1 of field f as a complex), times k_x^r[f], the
// first HX modes stored
struct IcPowers {
    int r[3];
};
template <int N, int HX, int NF, typename SRC>
__global__ __launch_bounds__((FftShape<double, N>::NT), 4) void k_ic_xf(SRC src, IcOut out, IcPowers pw, const cd *__restrict__ tw, double dk) {
    using S = FftShape<double, N>;
    using EX = typename S::P::EX;
    constexpr int B = S::B, NC = N / 2, TOTAL = B * NC, CNT = (TOTAL + S::NT - 1) / S::NT;
    __shared__ cd lds[EX::LDS_ELEMS];
    __shared__ cd twl[N];
    const cd *t = stage_twiddles<double, N, true>(tw, twl, threadIdx.x, S::NT);
    __syncthreads();
    const int lb = xcd_block(blockIdx.x, gridDim.x), yb = lb % (N / B), z = lb / (N / B);
    const size_t base = (size_t)N * N * z + (size_t)N * yb * B;
#pragma unroll 1
    for (int f = 0; f < NF; f++) {
        const int tid = round_tid();
        cd v[CNT];
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * S::NT;
            if (TOTAL % S::NT == 0 || i < TOTAL) v[c] = src(f, base + 2 * (size_t)i);
        }
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * S::NT;
            if (TOTAL % S::NT == 0 || i < TOTAL) lds[EX::idx(i / NC, i % NC)] = v[c];
        }
        x_lines<N, -1>(lds, t, tid);
        x_store<N, HX>(lds, out.p[f], t, yb, z, pw.r[f], dk, tid);
        __syncthreads();
    }
}

// The cotangents of three A_ik through mu, between their spectra in and out (in place when equal: a workgroup's
// rows are its own): inverse x of the three (s times their transforms), mubar (A_jj + A_kk) each (DIAG: in =
// A11, A22, A33) or -2 mubar A_ik (in = A12, A13, A23), forward x
template <int N, int HX, bool DIAG>
__global__ __launch_bounds__((FftShape<double, N>::NT), DIAG ? 2 : 3) void k_ic_x_adj(IcIn in, IcOut out, double s,
                                                                          const double *__restrict__ mub,
                                                                          const cd *__restrict__ tw, double dk) {
    using S = FftShape<double, N>;
    using EX = typename S::P::EX;
    constexpr int B = S::B, NC = N / 2, TOTAL = B * NC, CNT = (TOTAL + S::NT - 1) / S::NT;
    __shared__ cd lds[EX::LDS_ELEMS];
    __shared__ cd twl[N];
    const cd *t = stage_twiddles<double, N, true>(tw, twl, threadIdx.x, S::NT);
    __syncthreads();
    const int lb = xcd_block(blockIdx.x, gridDim.x), yb = lb % (N / B), z = lb / (N / B);
    const size_t base = (size_t)N * N * z + (size_t)N * yb * B;
    constexpr int F0 = DIAG ? 0 : 3;
    cd a[3][DIAG ? CNT : 1], m[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = threadIdx.x + c * S::NT;
        if (TOTAL % S::NT == 0 || i < TOTAL) m[c] = *(const cd *)(mub + (base + 2 * (size_t)i));
    }
    if constexpr (DIAG) {
#pragma unroll 1
        for (int f = 0; f < 3; f++) {  // a = the fields, the last one in a[2]
            const int tid = round_tid();
            x_load<N, HX>(in.p[f], lds, t, yb, z, second_power(F0 + f), dk, tid);
            x_lines<N, +1>(lds, t, tid);
#pragma unroll
            for (int c = 0; c < CNT; c++) {
                const int i = tid + c * S::NT;
                a[0][c] = a[1][c];
                a[1][c] = a[2][c];
                if (TOTAL % S::NT == 0 || i < TOTAL) a[2][c] = scale(lds[EX::idx(i / NC, i % NC)], s);
            }
            __syncthreads();
        }
    }
#pragma unroll 1
    for (int f = 0; f < 3; f++) {
        const int tid = round_tid();
        if constexpr (!DIAG) {
            x_load<N, HX>(in.p[f], lds, t, yb, z, second_power(F0 + f), dk, tid);
            x_lines<N, +1>(lds, t, tid);
        }
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * S::NT;
            if (!(TOTAL % S::NT == 0 || i < TOTAL)) continue;
            cd &v = lds[EX::idx(i / NC, i % NC)];
            if constexpr (DIAG) {
                const cd x = a[0][c];
                v = cd{m[c].x * (a[1][c].x + a[2][c].x), m[c].y * (a[1][c].y + a[2][c].y)};
                a[0][c] = a[1][c];
                a[1][c] = a[2][c];
                a[2][c] = x;
            } else {
                const cd x = scale(v, s);
                v = cd{-2.0 * (m[c].x * x.x), -2.0 * (m[c].y * x.y)};
            }
        }
        x_lines<N, -1>(lds, t, tid);
        x_store<N, HX>(lds, out.p[f], t, yb, z, second_power(F0 + f), dk, tid);
        __syncthreads();
    }
}

// Forward y pass: out = sum_q k_y^q (forward y of in[q]), q < NIN, the modes of an n grid stored
template <int N, int n, int HX, int NIN>
__global__ __launch_bounds__((FftShape<double, N>::NTY), 2) void k_ic_yf(IcIn in, cd *__restrict__ out,
                                                                     const cd *__restrict__ tw, double dk) {
    using S = FftShape<double, N>;
    using EF = typename S::PY::EF;
    constexpr int B = S::B, NT = S::NTY, TOTAL = B * N, CNT = (TOTAL + NT - 1) / NT;
    __shared__ cd lds[EF::LDS_ELEMS];
    __shared__ cd twl[S::TWL ? N : 1];
    const cd *t = stage_twiddles<double, N, S::TWL>(tw, twl, threadIdx.x, NT);
    const int lb = xcd_block(blockIdx.x, gridDim.x), zb = lb % (N / B), kx = lb / (N / B);
    cd acc[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) acc[c] = cd{0, 0};
#pragma unroll 1
    for (int q = NIN - 1; q >= 0; q--) {  // acc = acc k_y + in[q]
        const int tid = round_tid();
        cd v[CNT];
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL)
                v[c] = in.p[q][(size_t)(i % N) + (size_t)N * ((size_t)kx + (size_t)HX * (zb * B + i / N))];
        }
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL) lds[EF::idx(i / N, i % N)] = v[c];
        }
        yz_lines<N, -1>(lds, t, tid);
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (!(TOTAL % NT == 0 || i < TOTAL)) continue;
            acc[c] = scale(acc[c], k_axis(i / B, N, dk)) + lds[EF::idx(i % B, i / B)];
        }
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = threadIdx.x + c * NT, ky = band<N, n>(i / B);
        if ((TOTAL % NT == 0 || i < TOTAL) && ky >= 0)
            out[(size_t)(zb * B + i % B) + (size_t)N * ((size_t)kx + (size_t)HX * ky)] = acc[c];
    }
}

// Forward z pass: dst(line, kz, sum_p k_z^p (forward z of in[p])), p < NIN
template <int N, int NIN, typename DST>
__global__ __launch_bounds__((FftShape<double, N>::NTY), 2) void k_ic_zf(IcIn in, DST dst, const cd *__restrict__ tw,
                                                                     double dk) {
    using S = FftShape<double, N>;
    using EF = typename S::PY::EF;
    constexpr int NT = S::NTY, TOTAL = S::B * N, CNT = (TOTAL + NT - 1) / NT;
    __shared__ cd lds[EF::LDS_ELEMS];
    __shared__ cd twl[S::TWL ? N : 1];
    const cd *t = stage_twiddles<double, N, S::TWL>(tw, twl, threadIdx.x, NT);
    const size_t l0 = (size_t)blockIdx.x * S::B;
    cd acc[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) acc[c] = cd{0, 0};
#pragma unroll 1
    for (int p = NIN - 1; p >= 0; p--) {  // acc = acc k_z + in[p]
        const int tid = round_tid();
        cd v[CNT];
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL) v[c] = in.p[p][l0 * N + i];
        }
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (TOTAL % NT == 0 || i < TOTAL) lds[EF::idx(i / N, i % N)] = v[c];
        }
        yz_lines<N, -1>(lds, t, tid);
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int i = tid + c * NT;
            if (!(TOTAL % NT == 0 || i < TOTAL)) continue;
            acc[c] = scale(acc[c], k_axis(i % N, N, dk)) + lds[EF::idx(i / N, i % N)];
        }
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = threadIdx.x + c * NT;
        if (TOTAL % NT == 0 || i < TOTAL) dst(l0 + i / N, i % N, acc[c]);
    }
}

// ------------------------------------------------------------------------ sources and destinations
template <int n> __device__ __forceinline__ BIdx grid_mode(size_t line, int kz) {
    constexpr int H = n / 2 + 1;
    return BIdx{(int)(line % H), (int)(line / H), kz};
}
template <int n> __device__ __forceinline__ size_t grid_at(const BIdx &b) {
    return (size_t)b.kz + (size_t)n * ((size_t)b.kx + (size_t)(n / 2 + 1) * b.ky);
}
template <int n> __device__ __forceinline__ double k_squared(const BIdx &b, double dk) {
    const double kx = b.kx * dk, ky = sgn_full(b.ky, n) * dk, kz = sgn_full(b.kz, n) * dk;
    return (kx * kx + ky * ky) + kz * kz;
}
// a padded line's mode on the n grid; false where the pad is zero (the Nyquist planes are dropped, nlpt_core.jl:126-177)
template <int n> __device__ __forceinline__ bool pad_mode(size_t line, int z, BIdx &b) {
    constexpr int h = n / 2;
    b = BIdx{(int)(line % h), (int)(line / h), band<3 * n / 2, n>(z)};
    return b.ky != h && b.kz >= 0;
}

// phi(k) from the transform of the white noise
template <int n> struct PhiDst {
    cd *F;
    IcAmplitude amp;
    __device__ void operator()(size_t line, int kz, cd v) const {
        const BIdx b = grid_mode<n>(line, kz);
        F[grid_at<n>(b)] = scale(v, amp(b, n));
    }
};
// the transpose, F amp / w, as the source of the white noise's cotangent (w: 1 at kx = 0 and n/2, else 2)
template <int n> struct PhiAdjSrc {
    const cd *F;
    IcAmplitude amp;
    __device__ cd operator()(size_t line, int kz) const {
        const BIdx b = grid_mode<n>(line, kz);
        return scale(F[grid_at<n>(b)], amp(b, n) * (b.kx == 0 || b.kx == n / 2 ? 1.0 : 0.5));
    }
};
// the padded spectrum s F (ADJ: divided by the half-spectrum weight as well)
template <int n, bool ADJ> struct PadSrc {
    const cd *F;
    double s;
    __device__ cd operator()(size_t line, int z) const {
        BIdx b;
        if (!pad_mode<n>(line, z, b)) return cd{0, 0};
        return scale(F[grid_at<n>(b)], ADJ && b.kx ? 0.5 * s : s);
    }
};
// -i (c1 F + c2 G): the scalar spectrum of a displacement c1 psi1 + c2 psi2 (G = fL / k^2; no G on the Nyquist planes)
template <int n> struct CombineSrc {
    const cd *F, *G;
    double c1, c2;
    __device__ cd operator()(size_t line, int kz) const {
        const BIdx b = grid_mode<n>(line, kz);
        cd v = scale(F[grid_at<n>(b)], c1);
        if (G && b.kx != n / 2 && b.ky != n / 2 && b.kz != n / 2) v = v + scale(G[grid_at<n>(b)], c2);
        return cd{v.y, -v.x};
    }
};
// G = crop(fL) s / k^2 (0 at k = 0)
template <int n> struct SourceDst {
    cd *G;
    double s, dk;
    __device__ void operator()(size_t line, int z, cd v) const {
        BIdx b;
        if (!pad_mode<n>(line, z, b)) return;
        const double k2 = k_squared<n>(b, dk);
        G[grid_at<n>(b)] = k2 == 0 ? cd{0, 0} : scale(v, s / k2);
    }
};
// cotangents of F and G from a displacement's cotangent spectrum v: i w s v times c1, and times c2 / k^2; the first
// assigns, the second adds
template <int n, bool ADD> struct CombineAdjDst {
    cd *Fb, *Gb;
    double s, c1, c2, dk;
    __device__ void operator()(size_t line, int kz, cd v) const {
        const BIdx b = grid_mode<n>(line, kz);
        const double w = b.kx == 0 || b.kx == n / 2 ? s : 2.0 * s;
        const cd u = {-(w * v.y), w * v.x};
        const size_t e = grid_at<n>(b);
        const cd f = scale(u, c1);
        Fb[e] = ADD ? Fb[e] + f : f;
        if (Gb) {
            const double k2 = k_squared<n>(b, dk);
            const cd g = k2 == 0 ? cd{0, 0} : scale(u, c2 / k2);
            Gb[e] = ADD ? Gb[e] + g : g;
        }
    }
};
// Fb += crop(v) w s
template <int n> struct PadAdjDst {
    cd *Fb;
    double s;
    __device__ void operator()(size_t line, int z, cd v) const {
        BIdx b;
        if (!pad_mode<n>(line, z, b)) return;
        const size_t e = grid_at<n>(b);
        Fb[e] = Fb[e] + scale(v, b.kx ? 2.0 * s : s);
    }
};
// real fields: particle components of either precision; one field
template <typename T> struct ComponentsSrc {
    const T *p;
    size_t stride;
    __device__ cd operator()(int f, size_t g) const {
        const cx<T> v = *(const cx<T> *)(p + (stride * f + g));
        return cd{(double)v.x, (double)v.y};
    }
};
struct FieldSrc {
    const double *p;
    __device__ cd operator()(int, size_t g) const { return *(const cd *)(p + g); }
};
// order-2 factor of mu: ((3-2)/2 - 2) / ((2 + 3/2)(2 - 1)) = -3/7
constexpr double IC_MU2 = ((3.0 - 2) / 2 - 2.0) / ((2 + 1.5) * 1.0);

template <int n>
struct IcN {
    static constexpr int ext = 3 * n / 2, h = n / 2, H = n / 2 + 1;
    static constexpr bool has_second = n == 16 || n == 32 || n == 64 || n == 128 || n == 256 || n == 512;
    using S = FftShape<double, n>;

    // z, y and x passes of the n grid
    template <int NOUT, typename SRC> static void zi(const IcWork &w, const SRC &src, IcOut o, double dk, hipStream_t st) {
        k_ic_zi<n, NOUT><<<n * H / S::B, S::NTY, 0, st>>>(src, o, (const cd *)w.twn, dk);
    }
    template <typename T>
    static void displacement(const IcWork &w, double L, double c1, double c2, bool two, T *out, hipStream_t st) {
        const double dk = 2 * M_PI / L, s = 1.0 / ((double)n * n * n);
        const size_t M = (size_t)n * n * n;
        cd *const *Z = (cd *const *)w.Z, *const *Y = (cd *const *)w.W;
        const cd *tw = (const cd *)w.twn;
        zi<2>(w, CombineSrc<n>{(const cd *)w.F, two ? (const cd *)w.G : nullptr, c1, c2}, IcOut{{Z[0], Z[1]}}, dk, st);
        constexpr int by = n / S::B * H, bx = n / S::B * n, NX = S::NT;
        k_ic_yi<n, n, H, 2><<<by, S::NTY, 0, st>>>(Z[0], IcOut{{Y[0], Y[1]}}, tw, dk);
        k_ic_yi<n, n, H, 1><<<by, S::NTY, 0, st>>>(Z[1], IcOut{{Y[2]}}, tw, dk);
        for (int c = 0; c < 3; c++)
            k_ic_xi<n, H, T><<<bx, NX, 0, st>>>(Y[c], c == 0 ? 1 : 0, s, out + c * M, tw, dk);
    }
    template <typename T, bool ADD>
    static void displacement_adj(const IcWork &w, double L, const T *in, double c1, double c2, bool two, hipStream_t st) {
        const double dk = 2 * M_PI / L, s = 1.0 / ((double)n * n * n);
        const size_t M = (size_t)n * n * n;
        cd *const *Z = (cd *const *)w.Z, *const *Y = (cd *const *)w.W;
        const cd *tw = (const cd *)w.twn;
        constexpr int by = n / S::B * H, bx = n / S::B * n, NX = S::NT;
        k_ic_xf<n, H, 3><<<bx, NX, 0, st>>>(ComponentsSrc<T>{in, M}, IcOut{{Y[0], Y[1], Y[2]}}, IcPowers{{1, 0, 0}}, tw,
                                             dk);
        k_ic_yf<n, n, H, 2><<<by, S::NTY, 0, st>>>(IcIn{{Y[0], Y[1]}}, Z[0], tw, dk);
        k_ic_yf<n, n, H, 1><<<by, S::NTY, 0, st>>>(IcIn{{Y[2]}}, Z[1], tw, dk);
        k_ic_zf<n, 2><<<n * H / S::B, S::NTY, 0, st>>>(
            IcIn{{Z[0], Z[1]}},
            CombineAdjDst<n, ADD>{(cd *)w.Fb, two ? (cd *)w.G : nullptr, s, c1, c2, dk}, tw, dk);
    }

    // the spectra of the six A_ik after their y passes, in w.A (A11, A22, A33, A12, A13, A23)
    static void second(const IcWork &w, double L, hipStream_t st) {
        if constexpr (has_second) {
            using E = FftShape<double, ext>;
            const double dk = 2 * M_PI / L, pad = 27.0 / 8.0;  // (ext / n)^3
            cd *const *Z = (cd *const *)w.Z, *const *A = (cd *const *)w.A;
            const cd *tw = (const cd *)w.twe;
            k_ic_zi<ext, 3><<<n * h / E::B, E::NTY, 0, st>>>(PadSrc<n, false>{(const cd *)w.F, pad},
                                                           IcOut{{Z[0], Z[1], Z[2]}}, tw, dk);
            constexpr int by = ext / E::B * h;
            static_assert(ext % E::B == 0 && (n * h) % E::B == 0, "whole groups of lines");
            k_ic_yi<ext, n, h, 3><<<by, E::NTY, 0, st>>>(Z[0], IcOut{{A[0], A[3], A[1]}}, tw, dk);
            k_ic_yi<ext, n, h, 2><<<by, E::NTY, 0, st>>>(Z[1], IcOut{{A[4], A[5]}}, tw, dk);
            k_ic_yi<ext, n, h, 1><<<by, E::NTY, 0, st>>>(Z[2], IcOut{{A[2]}}, tw, dk);
        }
    }

    static void phi(const IcWork &w, double L, hipStream_t st) {
        const IcAmplitude amp{(const double *)w.amp};
        k_ic_zf<n, 1><<<n * H / S::B, S::NTY, 0, st>>>(IcIn{{(const cd *)w.Z[0]}}, PhiDst<n>{(cd *)w.F, amp},
                                                      (const cd *)w.twn, 2 * M_PI / L);
    }
    static void source(const IcWork &w, double L, hipStream_t st) {
        if constexpr (has_second) {
            using E = FftShape<double, ext>;
            const double dk = 2 * M_PI / L, s = 1.0 / ((double)ext * ext * ext), crop = 8.0 / 27.0;  // (n / ext)^3
            cd *const *Z = (cd *const *)w.Z, *const *Y = (cd *const *)w.W, *const *A = (cd *const *)w.A;
            const cd *tw = (const cd *)w.twe;
            constexpr int bx = ext / E::B * ext, by = ext / E::B * h, NX = E::NT;
            k_ic_xi_mu<ext, h><<<bx, NX, 0, st>>>(IcIn{{A[0], A[1], A[2], A[3], A[4], A[5]}}, s, IC_MU2, (double *)w.mu,
                                                  tw, dk);
            k_ic_xf<ext, h, 1><<<bx, NX, 0, st>>>(FieldSrc{(const double *)w.mu}, IcOut{{Y[0]}}, IcPowers{{0}}, tw, dk);
            k_ic_yf<ext, n, h, 1><<<by, E::NTY, 0, st>>>(IcIn{{Y[0]}}, Z[0], tw, dk);
            k_ic_zf<ext, 1><<<n * h / E::B, E::NTY, 0, st>>>(IcIn{{Z[0]}}, SourceDst<n>{(cd *)w.G, crop, dk}, tw, dk);
        }
    }
    template <typename T> static void combine(const IcWork &w, double L, double D, bool two, T *psi, T *pi, hipStream_t st) {
        displacement<T>(w, L, D, D * D, two, psi, st);
        displacement<T>(w, L, 1.0, 2 * D, two, pi, st);
    }
    static void combine_any(const IcWork &w, double L, double D, bool two, int prec, void *psi, void *pi, hipStream_t st) {
        if (prec == 64) combine(w, L, D, two, (double *)psi, (double *)pi, st);
        else combine(w, L, D, two, (float *)psi, (float *)pi, st);
    }
    template <typename T>
    static void combine_adj(const IcWork &w, double L, double D, bool two, const T *psibar, const T *pibar, hipStream_t st) {
        displacement_adj<T, false>(w, L, psibar, D, D * D, two, st);
        displacement_adj<T, true>(w, L, pibar, 1.0, 2 * D, two, st);
    }
    static void combine_adj_any(const IcWork &w, double L, double D, bool two, int prec, const void *psibar,
                                const void *pibar, hipStream_t st) {
        if (prec == 64) combine_adj(w, L, D, two, (const double *)psibar, (const double *)pibar, st);
        else combine_adj(w, L, D, two, (const float *)psibar, (const float *)pibar, st);
    }
    static void mu_adj(const IcWork &w, double L, hipStream_t st) {
        if constexpr (has_second) {
            using E = FftShape<double, ext>;
            const double dk = 2 * M_PI / L, crop = 8.0 / 27.0;
            cd *const *Z = (cd *const *)w.Z, *const *Y = (cd *const *)w.W;
            const cd *tw = (const cd *)w.twe;
            constexpr int bx = ext / E::B * ext, by = ext / E::B * h;
            // fL = crop(r2c_ext(-3/7 mu)) crop, G = fL / k^2:  mubar = -3/7 c2r_ext(pad(fLbar) crop / w)
            k_ic_zi<ext, 1><<<n * h / E::B, E::NTY, 0, st>>>(PadSrc<n, true>{(const cd *)w.G, crop}, IcOut{{Z[0]}}, tw, dk);
            k_ic_yi<ext, n, h, 1><<<by, E::NTY, 0, st>>>(Z[0], IcOut{{Y[0]}}, tw, dk);
            k_ic_xi<ext, h, double><<<bx, E::NT, 0, st>>>(Y[0], 0, IC_MU2, (double *)w.mu, tw, dk);
        }
    }
    static void source_adj(const IcWork &w, double L, hipStream_t st) {
        if constexpr (has_second) {
            using E = FftShape<double, ext>;
            const double dk = 2 * M_PI / L, s = 1.0 / ((double)ext * ext * ext), pad = 27.0 / 8.0;
            cd *const *Z = (cd *const *)w.Z, *const *Y = (cd *const *)w.W, *const *A = (cd *const *)w.A;
            const cd *tw = (const cd *)w.twe;
            constexpr int bx = ext / E::B * ext, by = ext / E::B * h, bz = n * h / E::B, NX = E::NT;
            const double *mub = (const double *)w.mu;
            k_ic_x_adj<ext, h, true><<<bx, NX, 0, st>>>(IcIn{{A[0], A[1], A[2]}}, IcOut{{Y[0], Y[1], Y[2]}}, s, mub, tw, dk);
            k_ic_x_adj<ext, h, false><<<bx, NX, 0, st>>>(IcIn{{A[3], A[4], A[5]}}, IcOut{{Y[3], Y[4], Y[5]}}, s, mub, tw, dk);
            k_ic_yf<ext, n, h, 3><<<by, E::NTY, 0, st>>>(IcIn{{Y[0], Y[3], Y[1]}}, Z[0], tw, dk);
            k_ic_yf<ext, n, h, 2><<<by, E::NTY, 0, st>>>(IcIn{{Y[4], Y[5]}}, Z[1], tw, dk);
            k_ic_yf<ext, n, h, 1><<<by, E::NTY, 0, st>>>(IcIn{{Y[2]}}, Z[2], tw, dk);
            k_ic_zf<ext, 3><<<bz, E::NTY, 0, st>>>(IcIn{{Z[0], Z[1], Z[2]}}, PadAdjDst<n>{(cd *)w.Fb, pad * s}, tw, dk);
        }
    }
    static void phi_adj(const IcWork &w, double L, hipStream_t st) {
        const IcAmplitude amp{(const double *)w.amp};
        zi<1>(w, PhiAdjSrc<n>{(const cd *)w.Fb, amp}, IcOut{{(cd *)w.Z[0]}}, 2 * M_PI / L, st);
    }
};

}  // namespace

bool ic_passes(int n, IcPasses &o) {
#define CASE(m)                                      \
    case m:                                          \
        o.phi = IcN<m>::phi;                         \
        o.second = IcN<m>::second;                   \
        o.source = IcN<m>::source;                   \
        o.combine = IcN<m>::combine_any;             \
        o.combine_adj = IcN<m>::combine_adj_any;     \
        o.mu_adj = IcN<m>::mu_adj;                   \
        o.source_adj = IcN<m>::source_adj;           \
        o.phi_adj = IcN<m>::phi_adj;                 \
        o.has_second = IcN<m>::has_second;           \
        return true;
    switch (n) {
        CASE(16) CASE(24) CASE(32) CASE(48) CASE(64) CASE(96) CASE(128) CASE(192) CASE(256) CASE(384)
        CASE(512) CASE(768) CASE(1024)
    }
#undef CASE
    return false;
}

}  // namespace dj
