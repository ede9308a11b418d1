// Sheet resampling (n_resample > 1): n_resample^3 - 1 extra point sets per interlacing pass, each the
// particle sheet displaced by a Lagrangian offset d (grid cells), deposited into the same density
// (NR/src/nbody/pm.jl:189-234 and 430-464).
//
//   psi_c = mod(Xs_c - q_c + L/2, L) - L/2                     (wrap, per component)
//   Fourier: npsi_c = brfft(rfft(psi_c) * px py pz / n^3)      (p_a = exp(2 pi i m_a d_a / n))
//   linear:  npsi_c = periodic trilinear interpolation of psi_c at (i + dx, j + dy, k + dz)
//   Xr_c = mod(q_c + npsi_c + d_c L / n + L, L), deposited like the particles
//
// The reference halves the slowest axis (z) of its real transforms, and once the phase factors break
// the Hermitian symmetry of the half spectrum the inverse depends on that choice.  The library's FFT
// passes halve the contiguous axis, so the Fourier path works on the transposed field psiT[z + n (y + n x)]:
// its halved axis is the reference's z, with the half-axis frequencies m / n (Nyquist +1/2), and the
// inverse is then the reference's.
#include <hip/hip_runtime.h>

#include "dj_complex.h"
#include "dj_internal.h"
#include "stencil.h"

namespace dj {

// psi_c of particle (i, j, k) at X_s = (psi + q) + s_c, into the natural or the transposed layout (the latter
// through a 32 x 32 tile in LDS: written straight, every lane's store is a line of its own, 182 us for 256^3
// in FP32)
template <typename T>
__device__ __forceinline__ T rs_wrapped(const T *psi, const T *q1, size_t p, int ic, T sc, T L) {
    const T qc = q1[ic], xs = (psi[p] + qc) + sc;
    return tjmod(xs - qc + L / (T)2, L) - L / (T)2;
}
template <typename T>
__global__ __launch_bounds__(256) void k_rs_wrap(const T *__restrict__ psi, const T *__restrict__ q1, int n, int c, T sc,
                                                 T L, T *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n, p = (size_t)i + N * ((size_t)j + N * k);
    out[p] = rs_wrapped(psi + (size_t)c * N * N * N, q1, p, c == 0 ? i : c == 1 ? j : k, sc, L);
}
template <typename T>
__global__ __launch_bounds__(256) void k_rs_wrap_t(const T *__restrict__ psi, const T *__restrict__ q1, int n, int c, T sc,
                                                   T L, T *__restrict__ out) {
    __shared__ T sh[32][33];
    const int i0 = blockIdx.x * 32, j = blockIdx.y, k0 = blockIdx.z * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const size_t N = (size_t)n;
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + tx, k = k0 + r;
        if (i < n && k < n)
            sh[r][tx] = rs_wrapped(psi + (size_t)c * N * N * N, q1, (size_t)i + N * ((size_t)j + N * k),
                                   c == 0 ? i : c == 1 ? j : k, sc, L);
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + r, k = k0 + tx;
        if (i < n && k < n) out[(size_t)k + N * ((size_t)j + N * i)] = sh[tx][r];
    }
}

// the phase of offset d on the transposed field's half spectrum, library layout B[w + n (h + H v)]:
// w = the reference's x (full axis), h = its z (half axis), v = its y (full axis)
template <typename T>
__global__ __launch_bounds__(256) void k_rs_phase(const cx<T> *__restrict__ in, cx<T> *__restrict__ out, int n,
                                                  const cx<T> *__restrict__ px, const cx<T> *__restrict__ py,
                                                  const cx<T> *__restrict__ pz, T scale) {
    const int H = n / 2 + 1;
    const size_t tot = (size_t)n * H * n;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
        const int w = (int)(e % n);
        const size_t r = e / n;
        const int h = (int)(r % H), v = (int)(r / H);
        // psi_hat * (px py pz scale), the factor built left to right as the reference does
        cx<T> f = cmul(cmul(px[w], py[v]), pz[h]);
        f = {f.x * scale, f.y * scale};
        out[e] = cmul(in[e], f);
    }
}

// periodic trilinear interpolation (pm.jl:220-231, the same sum order)
template <typename T>
__global__ __launch_bounds__(256) void k_rs_trilinear(const T *__restrict__ f, int n, T dx, T dy, T dz, T *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n;
    const int i1 = i + 1 == n ? 0 : i + 1, j1 = j + 1 == n ? 0 : j + 1, k1 = k + 1 == n ? 0 : k + 1;
    auto F = [&](int a, int b, int cc) { return f[(size_t)a + N * ((size_t)b + N * cc)]; };
    const T ex = (T)1 - dx, ey = (T)1 - dy, ez = (T)1 - dz;
    out[(size_t)i + N * ((size_t)j + N * k)] =
        F(i, j, k) * ex * ey * ez + F(i1, j, k) * dx * ey * ez + F(i, j1, k) * ex * dy * ez + F(i, j, k1) * ex * ey * dz +
        F(i1, j1, k) * dx * dy * ez + F(i1, j, k1) * dx * ey * dz + F(i, j1, k1) * ex * dy * dz +
        F(i1, j1, k1) * dx * dy * dz;
}

// Xr_c = mod(q_c + npsi_c + shift + L, L).  Written at point (nr i + o0, nr j + o1, nr k + o2) of the (nr n)^3
// lattice of all point sets of a pass (offset (o0, o1, o2) / nr cells: the sets interleave into a finer
// lattice; nr = 1, o = 0 is the plain layout)
template <typename T>
__global__ __launch_bounds__(256) void k_rs_place(const T *__restrict__ npsi, const T *__restrict__ q1, int n, int c,
                                                  T shift, T L, T *__restrict__ xr, int nr, int o0, int o1, int o2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n, p = (size_t)i + N * ((size_t)j + N * k), NR = (size_t)nr * n;
    const T qc = q1[c == 0 ? i : c == 1 ? j : k];
    const size_t pr = ((size_t)nr * i + o0) + NR * (((size_t)nr * j + o1) + NR * ((size_t)nr * k + o2));
    xr[pr + (size_t)c * NR * NR * NR] = tjmod(((qc + npsi[p]) + shift) + L, L);
}

// The same from NA fields in the transposed layout, of the offsets (o0, o1, o2) and, NA = 2, (o0 + 1, o1, o2):
// transposed through LDS, and two neighbours along x written together, so that lattice rows of nr = 2 are
// written whole.  x0 null: the first set is the particles themselves, at (psi + q) + s (a store per lane at the
// lattice's stride, of a value read along the other axis, took 95 us a component and offset at 256^3, FP32)
template <typename T, int NA>
__global__ __launch_bounds__(256) void k_rs_place_t(const T *__restrict__ x0, const T *__restrict__ x1,
                                                    const T *__restrict__ psi, const T *__restrict__ q1, int n, int c,
                                                    T s, T shift0, T shift1, T L, T *__restrict__ xr, int nr, int o0,
                                                    int o1, int o2) {
    __shared__ T sh[NA][32][33];
    const int i0 = blockIdx.x * 32, j = blockIdx.y, k0 = blockIdx.z * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const size_t N = (size_t)n, NR = (size_t)nr * n;
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + r, k = k0 + tx;
        if (i >= n || k >= n) continue;
        const size_t at = (size_t)k + N * ((size_t)j + N * i);
        if (x0) sh[0][r][tx] = x0[at];
        if constexpr (NA == 2) sh[NA - 1][r][tx] = x1[at];
    }
    __syncthreads();
    T *out = xr + (size_t)c * NR * NR * NR;
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + tx, k = k0 + r;
        if (i >= n || k >= n) continue;
        const T qc = q1[c == 0 ? i : c == 1 ? j : k];
        const size_t pr = ((size_t)nr * i + o0) + NR * (((size_t)nr * j + o1) + NR * ((size_t)nr * k + o2));
        T v0;
        if (x0) v0 = tjmod(((qc + sh[0][tx][r]) + shift0) + L, L);
        else v0 = (psi[(size_t)i + N * ((size_t)j + N * k) + (size_t)c * N * N * N] + qc) + s;
        if constexpr (NA == 2) {
            const T v1 = tjmod(((qc + sh[NA - 1][tx][r]) + shift1) + L, L);
            if (nr == 2) {
                *(cx<T> *)(out + pr) = cx<T>{v0, v1};  // o0 = 0: pr is even
            } else {
                out[pr] = v0;
                out[pr + 1] = v1;
            }
        } else {
            out[pr] = v0;
        }
    }
}

// the particles' own positions of the pass, X_c + s_c = (psi_c + q_c) + s_c (the deposit's arithmetic), at
// points (nr i, nr j, nr k) of the point-set lattice
template <typename T>
__global__ __launch_bounds__(256) void k_rs_shifted(const T *__restrict__ psi, const T *__restrict__ q1, int n, T s0,
                                                    T s1, T s2, int nr, T *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n, p = (size_t)i + N * ((size_t)j + N * k), NR = (size_t)nr * n, NR3 = NR * NR * NR;
    const size_t pr = (size_t)nr * i + NR * ((size_t)nr * j + NR * ((size_t)nr * k));
    out[pr] = (psi[p] + q1[i]) + s0;
    out[pr + NR3] = (psi[p + N * N * N] + q1[j]) + s1;
    out[pr + 2 * NR3] = (psi[p + 2 * N * N * N] + q1[k]) + s2;
}

// unit-mass deposit of the positions X (3, n^3) with device atomics, added to a mesh that the tile
// deposit has already written (float atomics, or int64 fixed point when FIXED)
template <typename T, int W, bool FIXED>
__global__ __launch_bounds__(256) void k_rs_scatter(const T *__restrict__ X, int n, void *mesh, int res, T L,
                                                    double fscale) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n, p = (size_t)i + N * ((size_t)j + N * k), np = N * N * N;
    T w[3][W];
    int cell[3][W];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const T g = tjmod(X[p + a * np], L) / L * (T)res;
        const int b = (W % 2 == 0) ? (int)floor(g) : (int)rint(g);
        const int lo = W == 2 ? 0 : -1;
#pragma unroll
        for (int o = 0; o < W; o++) {
            const int bo = b + lo + o;
            w[a][o] = twk<W>(fabs(g - (T)bo));
            int cc = bo % res;
            cell[a][o] = cc < 0 ? cc + res : cc;
        }
    }
#pragma unroll
    for (int oz = 0; oz < W; oz++)
#pragma unroll
        for (int oy = 0; oy < W; oy++) {
            const size_t row = (size_t)res * ((size_t)cell[1][oy] + (size_t)res * cell[2][oz]);
#pragma unroll
            for (int ox = 0; ox < W; ox++) {
                const T wv = w[0][ox] * w[1][oy] * w[2][oz];
                const size_t cidx = row + cell[0][ox];
                if constexpr (FIXED) {
                    atomicAdd((unsigned long long *)mesh + cidx, (unsigned long long)__double2ll_rn((double)wv * fscale));
                } else {
                    unsafeAtomicAdd((T *)mesh + cidx, wv);
                }
            }
        }
}

// ------------------------------------------------------------------------ reverse mode
// The resampled points enter the density only: the cotangent of their positions (the gather of grad W
// times the density cotangent at each point, on the point lattice) goes back to Psi through the
// transposed interpolation.  d Xr / d npsi and d psi_c / d Psi_c are the identity (the mods are locally
// translations).  Linear: the transpose of the trilinear shift scatters a point's cotangent to its 8
// corners, written here as a gather over the 8 points that use a lattice site.  Fourier: npsi = c2r(P s
// r2c(psi)) has the transpose c2r(conj(P) s r2c(npsibar)) (the half-axis weights of c2r and r2c cancel).

// the cotangent of point set (o0, o1, o2), component c, from the point lattice into the natural or the
// transposed n^3 layout
template <typename T, bool TRANSPOSED>
__global__ __launch_bounds__(256) void k_rs_extract(const T *__restrict__ pl, int n, int nr, int o0, int o1, int o2,
                                                    int c, T *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n, NR = (size_t)nr * n;
    const size_t pr = ((size_t)nr * i + o0) + NR * (((size_t)nr * j + o1) + NR * ((size_t)nr * k + o2));
    out[TRANSPOSED ? (size_t)k + N * ((size_t)j + N * i) : (size_t)i + N * ((size_t)j + N * k)] =
        pl[pr + (size_t)c * NR * NR * NR];
}

// hb (+)= in * conj((px py) pz scale): the forward's phase factor, conjugated
template <typename T, bool ACC>
__global__ __launch_bounds__(256) void k_rs_phase_adj(const cx<T> *__restrict__ in, cx<T> *__restrict__ hb, int n,
                                                      const cx<T> *__restrict__ px, const cx<T> *__restrict__ py,
                                                      const cx<T> *__restrict__ pz, T scale) {
    const int H = n / 2 + 1;
    const size_t tot = (size_t)n * H * n;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
        const int w = (int)(e % n);
        const size_t r = e / n;
        const int h = (int)(r % H), v = (int)(r / H);
        cx<T> f = cmul(cmul(px[w], py[v]), pz[h]);
        f = {f.x * scale, -(f.y * scale)};
        const cx<T> x = cmul(in[e], f);
        hb[e] = ACC ? hb[e] + x : x;
    }
}

// psibar_c (natural layout) += v (transposed layout)
template <typename T>
__global__ __launch_bounds__(256) void k_rs_add_transposed(const T *__restrict__ v, int n, T *__restrict__ psibar_c) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n;
    psibar_c[(size_t)i + N * ((size_t)j + N * k)] += v[(size_t)k + N * ((size_t)j + N * i)];
}

// psibar_c(i, j, k) += sum_{a, b, e in {0, 1}} wx(a) wy(b) wz(e) pbar(i - a, j - b, k - e), the transpose of
// k_rs_trilinear (w(0) = 1 - d, w(1) = d per axis), with pbar the point set's cotangent on the lattice
template <typename T>
__global__ __launch_bounds__(256) void k_rs_trilinear_adj(const T *__restrict__ pl, int n, int nr, int o0, int o1, int o2,
                                                          int c, T dx, T dy, T dz, T *__restrict__ psibar_c) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= n) return;
    const size_t N = (size_t)n, NR = (size_t)nr * n;
    const T *pc = pl + (size_t)c * NR * NR * NR;
    const int im = i == 0 ? n - 1 : i - 1, jm = j == 0 ? n - 1 : j - 1, km = k == 0 ? n - 1 : k - 1;
    auto P = [&](int a, int b, int e) {
        return pc[((size_t)nr * a + o0) + NR * (((size_t)nr * b + o1) + NR * ((size_t)nr * e + o2))];
    };
    const T ex = (T)1 - dx, ey = (T)1 - dy, ez = (T)1 - dz;
    const T v = P(i, j, k) * ex * ey * ez + P(im, j, k) * dx * ey * ez + P(i, jm, k) * ex * dy * ez +
                P(i, j, km) * ex * ey * dz + P(im, jm, k) * dx * dy * ez + P(im, j, km) * dx * ey * dz +
                P(i, jm, km) * ex * dy * dz + P(im, jm, km) * dx * dy * dz;
    psibar_c[(size_t)i + N * ((size_t)j + N * k)] += v;
}

template <typename T>
struct RsLaunch {
    static dim3 pgrid(int n) { return dim3((n + 255) / 256, n, n); }
    static dim3 tgrid(int n) { return dim3((n + 31) / 32, n, (n + 31) / 32); }
    static void wrap(const void *psi, const void *q1, int n, int c, double sc, double L, bool transposed, void *out,
                     hipStream_t st) {
        if (transposed)
            k_rs_wrap_t<T><<<tgrid(n), 256, 0, st>>>((const T *)psi, (const T *)q1, n, c, (T)sc, (T)L, (T *)out);
        else
            k_rs_wrap<T><<<pgrid(n), 256, 0, st>>>((const T *)psi, (const T *)q1, n, c, (T)sc, (T)L, (T *)out);
    }
    static void phase(const void *in, void *out, int n, const void *px, const void *py, const void *pz, double scale,
                      hipStream_t st) {
        k_rs_phase<T><<<2048, 256, 0, st>>>((const cx<T> *)in, (cx<T> *)out, n, (const cx<T> *)px, (const cx<T> *)py,
                                            (const cx<T> *)pz, (T)scale);
    }
    static void trilinear(const void *f, int n, const double *d, void *out, hipStream_t st) {
        k_rs_trilinear<T><<<pgrid(n), 256, 0, st>>>((const T *)f, n, (T)d[0], (T)d[1], (T)d[2], (T *)out);
    }
    static void place(const void *npsi, const void *q1, int n, int c, double shift, double L, void *xr, int nr,
                      const int *o, hipStream_t st) {
        k_rs_place<T><<<pgrid(n), 256, 0, st>>>((const T *)npsi, (const T *)q1, n, c, (T)shift, (T)L, (T *)xr, nr,
                                                o[0], o[1], o[2]);
    }
    static void place_t(const void *x0, const void *x1, int na, const void *psi, const void *q1, int n, int c, double s,
                        const double *shift, double L, void *xr, int nr, const int *o, hipStream_t st) {
        if (na == 2)
            k_rs_place_t<T, 2><<<tgrid(n), 256, 0, st>>>((const T *)x0, (const T *)x1, (const T *)psi, (const T *)q1, n,
                                                         c, (T)s, (T)shift[0], (T)shift[1], (T)L, (T *)xr, nr, o[0],
                                                         o[1], o[2]);
        else
            k_rs_place_t<T, 1><<<tgrid(n), 256, 0, st>>>((const T *)x0, nullptr, (const T *)psi, (const T *)q1, n, c,
                                                         (T)s, (T)shift[0], (T)0, (T)L, (T *)xr, nr, o[0], o[1], o[2]);
    }
    static void extract(const void *pl, int n, int nr, const int *o, int c, bool transposed, void *out,
                        hipStream_t st) {
        if (transposed)
            k_rs_extract<T, true><<<pgrid(n), 256, 0, st>>>((const T *)pl, n, nr, o[0], o[1], o[2], c, (T *)out);
        else
            k_rs_extract<T, false><<<pgrid(n), 256, 0, st>>>((const T *)pl, n, nr, o[0], o[1], o[2], c, (T *)out);
    }
    static void phase_adj(const void *in, void *hb, int n, const void *px, const void *py, const void *pz, double scale,
                          bool acc, hipStream_t st) {
        if (acc)
            k_rs_phase_adj<T, true><<<2048, 256, 0, st>>>((const cx<T> *)in, (cx<T> *)hb, n, (const cx<T> *)px,
                                                          (const cx<T> *)py, (const cx<T> *)pz, (T)scale);
        else
            k_rs_phase_adj<T, false><<<2048, 256, 0, st>>>((const cx<T> *)in, (cx<T> *)hb, n, (const cx<T> *)px,
                                                           (const cx<T> *)py, (const cx<T> *)pz, (T)scale);
    }
    static void add_transposed(const void *v, int n, void *psibar_c, hipStream_t st) {
        k_rs_add_transposed<T><<<pgrid(n), 256, 0, st>>>((const T *)v, n, (T *)psibar_c);
    }
    static void trilinear_adj(const void *pl, int n, int nr, const int *o, int c, const double *d, void *psibar_c,
                              hipStream_t st) {
        k_rs_trilinear_adj<T><<<pgrid(n), 256, 0, st>>>((const T *)pl, n, nr, o[0], o[1], o[2], c, (T)d[0], (T)d[1],
                                                        (T)d[2], (T *)psibar_c);
    }
    static void shifted(const void *psi, const void *q1, int n, const double *sh, int nr, void *out, hipStream_t st) {
        k_rs_shifted<T><<<pgrid(n), 256, 0, st>>>((const T *)psi, (const T *)q1, n, (T)sh[0], (T)sh[1], (T)sh[2], nr,
                                                  (T *)out);
    }
    template <int W>
    static void scatter_w(const void *X, int n, void *mesh, int res, double L, bool fixed, double fscale, hipStream_t st) {
        if (fixed) k_rs_scatter<T, W, true><<<pgrid(n), 256, 0, st>>>((const T *)X, n, mesh, res, (T)L, fscale);
        else k_rs_scatter<T, W, false><<<pgrid(n), 256, 0, st>>>((const T *)X, n, mesh, res, (T)L, fscale);
    }
    static void scatter(const void *X, int n, int W, void *mesh, int res, double L, bool fixed, double fscale,
                        hipStream_t st) {
        if (W == 2) scatter_w<2>(X, n, mesh, res, L, fixed, fscale, st);
        else if (W == 3) scatter_w<3>(X, n, mesh, res, L, fixed, fscale, st);
        else scatter_w<4>(X, n, mesh, res, L, fixed, fscale, st);
    }
};

template <typename T> void resample_ops(ResampleOps &ops) {
    ops.extract = RsLaunch<T>::extract;
    ops.phase_adj = RsLaunch<T>::phase_adj;
    ops.add_transposed = RsLaunch<T>::add_transposed;
    ops.trilinear_adj = RsLaunch<T>::trilinear_adj;
    ops.wrap = RsLaunch<T>::wrap;
    ops.phase = RsLaunch<T>::phase;
    ops.trilinear = RsLaunch<T>::trilinear;
    ops.place = RsLaunch<T>::place;
    ops.place_t = RsLaunch<T>::place_t;
    ops.shifted = RsLaunch<T>::shifted;
    ops.scatter = RsLaunch<T>::scatter;
}

template void resample_ops<float>(ResampleOps &);
template void resample_ops<double>(ResampleOps &);

}  // namespace dj
