// Power spectrum of a deposited density on the device: the accuracy measurement of the PM path.
// Follows the study estimator (studies/eft_shell_crossing/src/measure.jl:403-447) and the
// normalisation of NR/src/analysis/power_spectrum.jl:25-79:
//   delta = mesh * N^3 / n^3 - 1,  P(k) = V <w |delta_k|^2 / |W(k)|^2>_bin / N^6
// with mode weights w = 1 on the two planes the half spectrum keeps unpaired (here kx = 0 and
// kx = N/2) and 2 elsewhere, |W(k)|^2 = prod_a sinc(k_a dx / 2)^(2 W) the mass-assignment window, and
// linear bins b = [kf (b + 1/2), kf (b + 3/2)).  The spectrum is the library's x-halved B layout.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "dj_internal.h"
#include "fft_passes.h"

namespace dj {

template <typename T>
__global__ __launch_bounds__(256) void k_pk_bin(const cx<T> *__restrict__ B, int N, double L, int W, int nbins,
                                                double scale, double *__restrict__ sum_p, double *__restrict__ sum_w,
                                                unsigned long long *__restrict__ cnt) {
    extern __shared__ double sh[];
    double *sp = sh, *sw = sh + nbins;
    unsigned long long *sc = (unsigned long long *)(sh + 2 * nbins);
    for (int b = threadIdx.x; b < nbins; b += blockDim.x) { sp[b] = 0; sw[b] = 0; sc[b] = 0; }
    __syncthreads();
    const int H = N / 2 + 1;
    const size_t tot = (size_t)N * H * N;
    const double kf = 2 * M_PI / L, dx = L / N;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
        int kz = (int)(e % N);
        size_t t = e / N;
        int kx = (int)(t % H), ky = (int)(t / H);
        double k3[3] = {kx * kf, (ky < N / 2 ? ky : ky - N) * kf, (kz < N / 2 ? kz : kz - N) * kf};
        double k = sqrt(k3[0] * k3[0] + k3[1] * k3[1] + k3[2] * k3[2]);
        int b = (int)floor(k / kf - 0.5);
        if (k == 0 || b < 0 || b >= nbins) continue;
        double win = 1;
        if (W > 0)
            for (int a = 0; a < 3; a++) {
                double u = k3[a] * dx / 2, s = u == 0 ? 1.0 : sin(u) / u;
                win *= pow(s, 2 * W);
            }
        cx<T> v = B[e];
        double p = ((double)v.x * v.x + (double)v.y * v.y) * scale;
        double w = (kx == 0 || kx == N / 2) ? 1.0 : 2.0;
        atomicAdd(&sp[b], w * p / win);
        atomicAdd(&sw[b], w);
        atomicAdd(&sc[b], 1ull);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nbins; b += blockDim.x) {
        if (sc[b]) {
            atomicAdd(&sum_p[b], sp[b]);
            atomicAdd(&sum_w[b], sw[b]);
            atomicAdd(&cnt[b], sc[b]);
        }
    }
}

template <typename T>
void pk_bin(const void *B, int N, double L, int W, int nbins, double scale, double *sum_p, double *sum_w,
            unsigned long long *cnt, hipStream_t st) {
    size_t shm = (size_t)nbins * (2 * sizeof(double) + sizeof(unsigned long long));
    k_pk_bin<T><<<2048, 256, shm, st>>>((const cx<T> *)B, N, L, W, nbins, scale, sum_p, sum_w, cnt);
}

template void pk_bin<float>(const void *, int, double, int, int, double, double *, double *, unsigned long long *,
                            hipStream_t);
template void pk_bin<double>(const void *, int, double, int, int, double, double *, double *,
                             unsigned long long *, hipStream_t);


// ------------------------------------------------------------------ binned spectra over given edges
// The binning of evaluate_power_spectrum / evaluate_cross_power_spectrum (NR/src/analysis/power_spectrum.jl:
// 25-123) and of the study estimator (studies/eft_shell_crossing/src/measure.jl:403-447), on the library's
// x-halved spectrum.  The reference halves the z axis: its modes are (i, j, l), i, j < N, l <= N/2, with
// signed wavenumbers (i <= N/2 ? i : i - N) kf.  A stored entry (x, y, z) is the reference's mode (x, y, z)
// when z <= N/2, and the conjugate of its mode (N - x, -y, N - z) when 0 < x < N/2 and z is 0 or >= N/2, with
// the same |F|^2 (and Re conj(F1) F2) and the same |k|: entries on the x = 0 and N/2 planes are one mode or
// none, the others one, or two at z = 0 and N/2.  |k| is formed exactly as the reference does, in FP64, so
// that every mode lands in the reference's bin: sqrt((kx kx + ky ky) + kz kz) >= e exactly when the sum is
// at least pk_threshold(e), so the bins are found by comparing sums.  Per bin |k|, w v, w and the count are
// summed in LDS, then once per block into sums (4 nbins doubles).
//   wmode 0: w = 1/2 on the l = 0 and l = N/2 planes, 1 elsewhere (the auto spectrum and the study
//            estimator, whose 1 / 2 weights have the same ratio); wmode 1: w = 1 (the cross spectrum)
//   W > 0:   v is divided by |W(k)|^2 = prod_a sinc(k_a dx / 2)^(2 W) (mass-assignment window)
// A thread takes one z and PK_XL consecutive x of a y row, so that its entries stay in one bin for a while:
// their sums stay in registers until the bin changes (LDS atomics once per run of entries; neighbouring
// lanes mostly share the bin, so one atomic per entry met 64 others at one address: 482 us a call,
// FP32, over three of 256^3 and one of 512^3 with the window's sin and pow per entry, against 84).  The window's factors are a table in LDS.
// PK_XL is 16, and 4 on meshes up to 64^3, where few threads would walk long runs one after the other: the spectra
// of 32^3 on 32^3 took 251 us with 16 and 215 with 4, of 64^3 on 64^3 259 and 231 (FP32).
constexpr int PK_COPIES = 4;

template <typename T, bool CROSS, bool KSUM, int PK_XL>
__global__ __launch_bounds__(256) void k_pk_edges(const cx<T> *__restrict__ F1, const cx<T> *__restrict__ F2, int N,
                                                  double kf, double dx, int W, int wmode, double scale, PkEdges thr,
                                                  double *__restrict__ sums) {
    extern __shared__ double sh[];
    const int nb = thr.nbins, H = N / 2 + 1;
    double *st = sh, *sb = st + nb + 1, *swin = sb + PK_COPIES * 4 * nb;
    for (int b = threadIdx.x; b <= nb; b += 256) st[b] = thr.e[b];
    for (int b = threadIdx.x; b < PK_COPIES * 4 * nb; b += 256) sb[b] = 0;
    if (W > 0)
        for (int m = threadIdx.x; m < H; m += 256) {
            const double s0 = (double)m * kf * dx / 2, s = s0 == 0 ? 1.0 : sin(s0) / s0;
            swin[m] = pow(s, 2 * W);
        }
    __syncthreads();
    double *mine = sb + (threadIdx.x & (PK_COPIES - 1)) * 4 * nb;
    const double t_lo = st[0], t_hi = st[nb];
    const int runs = (H + PK_XL - 1) / PK_XL;      // runs of x per (y, z)
    const int per_y = runs * N;                    // threads' items of a y row, z fastest
    const int chunks = (per_y + 255) / 256, items = chunks * N;
    for (int it = blockIdx.x; it < items; it += gridDim.x) {
        const int y = it / chunks, q = (it - y * chunks) * 256 + threadIdx.x;
        if (q >= per_y) continue;
        const int run = q / N, z = q - run * N, x0 = run * PK_XL, x1 = min(x0 + PK_XL, H);
        const int my = y <= N / 2 ? y : N - y, mz = z <= N / 2 ? z : N - z;
        const double ky = (double)my * kf, kz = (double)mz * kf, ky2 = ky * ky, kz2 = kz * kz;
        const bool end = z == 0 || z == N / 2;
        const double wend = wmode == 0 && end ? 0.5 : 1.0;
        const cx<T> *f1 = F1 + ((size_t)z + (size_t)N * H * y), *f2 = CROSS ? F2 + ((size_t)z + (size_t)N * H * y) : nullptr;
        int b = -1;                                // the run's bin and its sums
        double lo = 1, hi = 0, ak = 0, ap = 0, aw = 0, ac = 0;
        auto flush = [&]() {
            if (b < 0 || ac == 0) return;
            if (KSUM) atomicAdd(&mine[b], ak);
            atomicAdd(&mine[nb + b], ap);
            atomicAdd(&mine[2 * nb + b], aw);
            atomicAdd(&mine[3 * nb + b], ac);
            ak = ap = aw = ac = 0;
        };
        // the entries of four x are loaded before the first is used
        for (int xb = x0; xb < x1; xb += 4) {
            cx<T> u4[4], w4[4];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const size_t at = (size_t)N * min(xb + d, x1 - 1);
                u4[d] = f1[at];
                if constexpr (CROSS) w4[d] = f2[at];
            }
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const int x = xb + d;
                if (x >= x1) break;
                const bool edge = x == 0 || x == N / 2;
                const double cnt = edge ? (z <= N / 2 ? 1.0 : 0.0) : (end ? 2.0 : 1.0);
                const double kx = (double)x * kf, s = kx * kx + ky2 + kz2;
                if (cnt == 0 || !(s > 0) || s < t_lo || !(s < t_hi)) continue;
                if (!(s >= lo && s < hi)) {
                    flush();
                    int a = 0, c = nb;                 // st[a] <= s < st[c]
                    while (c - a > 1) {
                        const int m = (a + c) >> 1;
                        if (st[m] <= s) a = m; else c = m;
                    }
                    b = a;
                    lo = st[a];
                    hi = st[a + 1];
                }
                const cx<T> u = u4[d];
                double v;
                if constexpr (CROSS) {
                    const cx<T> w2 = w4[d];
                    v = ((double)u.x * w2.x + (double)u.y * w2.y) * scale;
                } else {
                    v = ((double)u.x * u.x + (double)u.y * u.y) * scale;
                }
                if (W > 0) v /= swin[x] * swin[my] * swin[mz];
                const double w = cnt * wend;
                if constexpr (KSUM) ak += cnt * sqrt(s);
                ap += w * v;
                aw += w;
                ac += cnt;
            }
        }
        flush();
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += 256) {
        double t[4] = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < PK_COPIES; c++)
#pragma unroll
            for (int k = 0; k < 4; k++) t[k] += sb[(4 * c + k) * nb + b];
        if (t[3] > 0) {
            if constexpr (KSUM) atomicAdd(&sums[b], t[0]);
            atomicAdd(&sums[nb + b], t[1]);
            atomicAdd(&sums[2 * nb + b], t[2]);
            atomicAdd(&sums[3 * nb + b], t[3]);
        }
    }
}

// the smallest double whose square root (rounded to nearest) is at least e
double pk_threshold(double e) {
    if (!(e > 0)) return 0.0;
    double s = e * e;
    while (std::sqrt(s) < e) s = std::nextafter(s, INFINITY);
    while (s > 0 && std::sqrt(std::nextafter(s, 0.0)) >= e) s = std::nextafter(s, 0.0);
    return s;
}

// Per bin: k_out = mean |k| of its modes (the geometric centre sqrt(e_b e_b+1) of an empty bin, or
// always when centre_only), pk_out = mult sum(w v) / sum(w) (0 when empty), nmodes_out = count / ncomp.
__global__ void k_pk_finalize(const double *__restrict__ sums, PkEdges ed, double mult, int ncomp, int centre_only,
                              double *__restrict__ k_out, double *__restrict__ pk_out, long long *__restrict__ nm_out) {
    const int nb = ed.nbins;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        const double cnt = sums[3 * nb + b], sw = sums[2 * nb + b];
        if (k_out) k_out[b] = (cnt > 0 && !centre_only) ? sums[b] / cnt : sqrt(ed.e[b] * ed.e[b + 1]);
        if (pk_out) pk_out[b] = cnt > 0 ? mult * sums[nb + b] / sw : 0.0;
        if (nm_out) nm_out[b] = (long long)(cnt / ncomp);
    }
}

__global__ void k_fill_zero_d(double *p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0.0;
}

template <typename T>
void pk_edges(const void *F1, const void *F2, int N, double L, int W, int wmode, double scale, const PkEdges &ed,
              bool ksum, double *sums, hipStream_t st) {
    const int nb = ed.nbins, H = N / 2 + 1;
    PkEdges thr{};
    thr.nbins = nb;
    for (int b = 0; b <= nb; b++) thr.e[b] = pk_threshold(ed.e[b]);
    const size_t shm = sizeof(double) * ((size_t)(nb + 1) + PK_COPIES * 4 * (size_t)nb + (W > 0 ? H : 0));
    const int xl = N <= 64 ? 4 : 16;
    // a block's bins reach memory once, so four blocks per CU walk the rows
    const int items = N * (((H + xl - 1) / xl * N + 255) / 256), blocks = std::min(1024, items);
    auto launch = [&](auto kern) {
        kern<<<blocks, 256, shm, st>>>((const cx<T> *)F1, (const cx<T> *)F2, N, 2 * M_PI / L, L / N, W, wmode, scale,
                                       thr, sums);
    };
    auto pick = [&](auto k4, auto k16) { xl == 4 ? launch(k4) : launch(k16); };
    if (F2) ksum ? pick(k_pk_edges<T, true, true, 4>, k_pk_edges<T, true, true, 16>)
                 : pick(k_pk_edges<T, true, false, 4>, k_pk_edges<T, true, false, 16>);
    else ksum ? pick(k_pk_edges<T, false, true, 4>, k_pk_edges<T, false, true, 16>)
              : pick(k_pk_edges<T, false, false, 4>, k_pk_edges<T, false, false, 16>);
}
template void pk_edges<float>(const void *, const void *, int, double, int, int, double, const PkEdges &, bool,
                              double *, hipStream_t);
template void pk_edges<double>(const void *, const void *, int, double, int, int, double, const PkEdges &, bool,
                               double *, hipStream_t);

void pk_finalize(const double *sums, const PkEdges &ed, double mult, int ncomp, bool centre_only, double *k_out,
                 double *pk_out, int64_t *nm_out, hipStream_t st) {
    k_pk_finalize<<<1, 256, 0, st>>>(sums, ed, mult, ncomp, centre_only ? 1 : 0, k_out, pk_out, (long long *)nm_out);
}

void zero_doubles(double *p, int n, hipStream_t st) { k_fill_zero_d<<<(n + 255) / 256, 256, 0, st>>>(p, n); }

// The scratch of dj_field_power_spectrum_noalloc: the bin sums (4 PK_MAX_BINS doubles) in a
// file-scope device array, one per device, held until the process ends.  Host code reaches it only
// through the address hipGetSymbolAddress returns on that device (pk_scratch).
static __device__ __align__(256) double scratch[4 * PK_MAX_BINS];

namespace {
std::mutex g_scratch_mu;
double *g_scratch_ptr[64] = {};
}  // namespace

hipError_t pk_scratch_init(int dev) {
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev]) return hipSuccess;
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess) return e;
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess) g_scratch_ptr[dev] = (double *)p;
    if (cur != dev) (void)hipSetDevice(cur);
    return e;
}

double *pk_scratch(int dev) {
    if (dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_ptr[dev];
}

}  // namespace dj
