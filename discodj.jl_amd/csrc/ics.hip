// Initial conditions of the PM path on the device, in FP64 (the IC pipeline of the reference):
//   white noise w ............ N-GenIC field (seed table on the host, ngenic.cpp; the column
//                              generators on the device) -> real space by the library's c2r
//                              (ngenic_wnoise_real, NR/src/ics/ngenic_gsl.jl:174-177)
//   phi(k) ................... rfft(w) * (-sqrt(P(k) (n/L)^3) / k^2), 0 at k = 0 (grf.jl:118-144)
//   psi_1 .................... irfft(-(i k_c) phi)  (nlpt_core.jl:285-297)
//   psi_2 (n_order = 2) ...... de-aliased on ext = 3n/2: A_ik = irfft_ext(i k_k pad(psi1_i)), the
//                              mu2 source A11 A22 + A11 A33 + A22 A33 - A12 A21 - A13 A31 - A23 A32
//                              times -3/7, crop(rfft_ext(.)), psi_2 = irfft(-1/k^2 (i k_c) .)
//                              (nlpt_fast.jl:27-64, 208-249; nlpt_core.jl:126-177)
//   Psi = D psi1 + D^2 psi2, Pi = psi1 + 2 D psi2 (run_nbody.jl:200-206)
// Spectra are in the library's x-halved B layout  B[kz + N (kx + H ky)].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "dj_internal.h"
#include "fft_passes.h"
#include "ic_modes.h"

namespace dj {

static unsigned g1(size_t n) { return (unsigned)((n + 255) / 256); }

// ---------------------------------------------------------------- N-GenIC white noise on the device
// The column generators of ngenic_field_gsl (NR/src/ics/ngenic_gsl.jl:126-165): GSL ranlxd1 (RANLUX,
// 48-bit subtract-with-borrow in exact double arithmetic, lags 12 and 5, 202 steps per 12 numbers
// delivered; ngenic_gsl.jl:35-98), seeded from the host's seed table, one thread per (i, j) column.
// The twelve state words of each thread live in LDS (stride 256, so a wave's accesses are consecutive)
// because the recurrence indexes them by a running position.  The uniforms are the same bits as the
// host's; sqrt(-log u), cos and sin are the device's FP64 functions (within an ulp or two of the host
// libm's).
namespace {
constexpr double kNgOneBit = 1.0 / 281474976710656.0;  // 2^-48

struct NgGen {
    double *x;  // 12 words at stride 256
    double carry;
    int ir, jr, ir_old;
    __device__ __forceinline__ double &w(int k) { return x[k * 256]; }
    __device__ void seed(uint32_t s) {
        if (s == 0) s = 1;
        uint32_t bits = s & 0x7fffffffu;  // the 31 seed bits xbit[0..30]
        int ib = 0, jb = 18;
        for (int k = 0; k < 12; k++) {
            double v = 0;
            for (int m = 0; m < 48; m++) {
                const uint32_t b = (bits >> ib) & 1u;
                v += v + (double)(1u - b);
                const uint32_t nb = b ^ ((bits >> jb) & 1u);
                bits = (bits & ~(1u << ib)) | (nb << ib);
                ib = ib == 30 ? 0 : ib + 1;
                jb = jb == 30 ? 0 : jb + 1;
            }
            w(k) = kNgOneBit * v;
        }
        carry = 0;
        ir = 11;
        jr = 7;
        ir_old = 0;
    }
    __device__ __forceinline__ void swb() {
        double y = w(jr) - w(ir) - carry;
        if (y < 0) { carry = kNgOneBit; y += 1; } else { carry = 0; }
        w(ir) = y;
        ir = ir == 11 ? 0 : ir + 1;
        jr = jr == 11 ? 0 : jr + 1;
    }
    __device__ double next() {
        ir = ir == 11 ? 0 : ir + 1;
        if (ir == ir_old) {
            for (int k = 0; k < 202; k++) swb();
            ir_old = ir;
        }
        return w(ir);
    }
};
}  // namespace

__global__ __launch_bounds__(256) void k_ngenic_columns(const uint32_t *__restrict__ tab, int res, double *out) {
    __shared__ double xs[12 * 256];
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (size_t)res * res) return;  // no barrier below: each thread's words are its own
    const int i = (int)(t % res), j = (int)(t / res), half = res / 2;
    const int ii = i > 0 ? res - i : 0, jj = j > 0 ? res - j : 0;
    const size_t R = (size_t)res;
    NgGen g;
    g.x = xs + threadIdx.x;
    g.seed(tab[(size_t)i * R + j]);
    const double twopi = 2 * M_PI;
    for (int k = 0; k <= half; k++) {
        const double phase = g.next() * twopi;
        double ampl;
        do { ampl = g.next(); } while (ampl == 0.0 || ampl == 1.0);
        if (i == half || j == half || k == half) continue;
        if (i == 0 && j == 0 && k == 0) continue;
        ampl = sqrt(-log(ampl));
        const double re = ampl * cos(phase), im = ampl * sin(phase);
        auto put = [&](int a, int b, int c, double xr, double xi) {
            const size_t e = (size_t)a + R * ((size_t)b + R * c);
            out[2 * e] = xr;
            out[2 * e + 1] = xi;
        };
        if (k > 0) {
            put(i, j, k, re, im);
        } else if (i == 0) {
            if (j < half) {
                put(0, j, 0, re, im);
                put(0, jj, 0, re, -im);
            }
        } else if (i < half) {
            put(i, j, 0, re, im);
            put(ii, jj, 0, re, -im);
        }
    }
}

__global__ void k_fill_zero_f64(double *p, size_t n) {
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
        p[e] = 0.0;
}

int ngenic_field_device(uint32_t seed, int res, double *d_field, hipStream_t st) {
    const size_t R = (size_t)res, nc = R * R * (res / 2 + 1);
    std::vector<uint32_t> tab(R * R);
    ngenic_seed_table(seed, res, tab.data());
    uint32_t *d_tab = nullptr;
    hipError_t e = hipMalloc(&d_tab, sizeof(uint32_t) * R * R);
    if (e == hipSuccess) e = hipMemcpyAsync(d_tab, tab.data(), sizeof(uint32_t) * R * R, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        k_fill_zero_f64<<<(unsigned)std::min<size_t>(8192, (2 * nc + 255) / 256), 256, 0, st>>>(d_field, 2 * nc);
        k_ngenic_columns<<<g1(R * R), 256, 0, st>>>(d_tab, res, d_field);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (d_tab) (void)hipFree(d_tab);
    return (int)e;
}

// N-GenIC field (z halved, (n, n, n/2+1)) -> B layout (x halved) by Hermitian symmetry, times n^(3/2)
__global__ void k_field_to_blayout(const cx<double> *__restrict__ f, int n, double sc, cx<double> *__restrict__ B) {
    const int H = n / 2 + 1;
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x, tot = (size_t)n * H * n;
    if (e >= tot) return;
    const BIdx k = bidx(e, n);
    cx<double> v;
    if (k.kz <= n / 2) {
        v = f[(size_t)k.kx + n * ((size_t)k.ky + (size_t)n * k.kz)];
    } else {
        const int mx = (n - k.kx) % n, my = (n - k.ky) % n, mz = n - k.kz;
        v = conj(f[(size_t)mx + n * ((size_t)my + (size_t)n * mz)]);
    }
    B[e] = scale(v, sc);
}

void ic_work_free(IcWork &ws) {
    for (void *p : ws.bufs) (void)hipFree(p);
    ws = IcWork{};
}

// the buffers of both directions for (n, order) and room for ntab table entries, kept while they fit
static hipError_t ic_work_ensure(IcWork &ws, int n, int order, int ntab) {
    if (ws.n == n && ws.order >= order && ws.ntab >= ntab) return hipSuccess;
    ic_work_free(ws);
    const size_t ext = 3 * (size_t)n / 2, h = (size_t)n / 2, M = (size_t)n * n * n, HC = (size_t)n * n * (h + 1);
    hipError_t err = hipSuccess;
    auto alloc = [&](size_t bytes) -> void * {
        void *p = nullptr;
        if (err == hipSuccess) err = hipMalloc(&p, bytes);
        if (p) ws.bufs.push_back(p);
        return p;
    };
    auto twiddles = [&](int N) -> void * {
        std::vector<cx<double>> tw(N);
        for (int k = 0; k < N; k++) {
            double a = -2.0 * M_PI * (double)k / (double)N;
            tw[k] = {std::cos(a), std::sin(a)};
        }
        void *d = alloc(sizeof(cx<double>) * N);
        if (d && err == hipSuccess) err = hipMemcpy(d, tw.data(), sizeof(cx<double>) * N, hipMemcpyHostToDevice);
        return d;
    };
    const int cap = std::max(ntab, 4096);
    ws.twn = twiddles(n);
    ws.kt = alloc((size_t)cap * 8);
    ws.pt = alloc((size_t)cap * 8);
    ws.amp = alloc(ic_amplitudes(n) * 8);
    ws.F = alloc(HC * 16);
    ws.Fb = alloc(HC * 16);
    ws.w = alloc(M * 8);
    // line spectra and after-y spectra: of the n grid, and of the ext grid without the pad's zeros
    const bool two = order >= 2;
    const size_t zs = two ? std::max(HC, ext * h * n) : HC, ys = two ? std::max(HC, ext * h * ext) : HC;
    for (int k = 0; k < (two ? 3 : 2); k++) ws.Z[k] = alloc(zs * 16);
    for (int k = 0; k < (two ? 6 : 3); k++) ws.W[k] = ws.A[k] = alloc(ys * 16);
    if (two) {
        ws.twe = twiddles((int)ext);
        ws.G = alloc(HC * 16);
        ws.mu = alloc(ext * ext * ext * 8);
    }
    if (err != hipSuccess) {
        ic_work_free(ws);
        return err;
    }
    ws.n = n;
    ws.order = order;
    ws.ntab = cap;
    return hipSuccess;
}

// Room to keep the forward's second derivatives and the white-noise key, allocated once per workspace; false (and
// no retry) when the device has no room for them
static bool ic_keep_ensure(IcWork &ws, int n) {
    if (ws.fk_room) return ws.fk_room > 0;
    const size_t ext = 3 * (size_t)n / 2, h = (size_t)n / 2, M = (size_t)n * n * n, HC = (size_t)n * n * (h + 1);
    const size_t ys = std::max(HC, ext * h * ext);
    hipError_t err = hipSuccess;
    auto alloc = [&](size_t bytes) -> void * {
        void *p = nullptr;
        if (err == hipSuccess) err = hipMalloc(&p, bytes);
        if (p) ws.bufs.push_back(p);
        return p;
    };
    void *keep[6];
    for (auto &p : keep) p = alloc(ys * 16);
    ws.wkey = alloc(M * 8);
    ws.flag = alloc(sizeof(unsigned));
    if (err != hipSuccess) {
        (void)hipGetLastError();  // an out-of-memory here is not an error of the call
        ws.fk_room = -1;
        return false;
    }
    for (int k = 0; k < 6; k++) ws.A[k] = keep[k];
    ws.fk_room = 1;
    return true;
}

__global__ void k_ic_differs(const unsigned long long *a, const unsigned long long *b, size_t n, unsigned *flag) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && a[i] != b[i]) atomicOr(flag, 1u);
}

// white noise into w: copied from the host or the device, or the N-GenIC field of seed
static hipError_t ic_white(IcWork &ws, FftOps &fn, int n, const double *white, bool on_device, uint32_t seed, double *w,
                           hipStream_t st) {
    const size_t M = (size_t)n * n * n, HC = (size_t)n * (n / 2 + 1) * n;
    if (white)
        return hipMemcpyAsync(w, white, M * 8, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st);
    // the z-halved field (n n (n/2+1) complex values, the size of F, which is free until phi(k)), then to
    // the B layout and back to real space
    hipError_t err = (hipError_t)ngenic_field_device(seed, n, (double *)ws.F, st);
    if (err != hipSuccess) return err;
    const KMult<double> none{};
    k_field_to_blayout<<<g1(HC), 256, 0, st>>>((const cx<double> *)ws.F, n, std::pow((double)n, 1.5),
                                               (cx<double> *)ws.Z[0]);
    fn.zm(ZM_NONE, false, true, ws.Z[0], ws.Z[0], ws.twn, &none, st);
    fn.yi(ws.Z[0], ws.W[0], ws.twn, st);
    fn.xi_scaled(ws.W[0], w, ws.twn, 1.0 / (double)M, st);
    return hipGetLastError();
}

__global__ void k_ic_amplitudes(double *amp, size_t cnt, int n, double L, const double *kt, const double *pt, int ntab) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) amp[i] = ic_amplitude_entry(i, n, L, kt, pt, ntab);
}

// the P(k) table, and the amplitude of every mode length from it (searched once per length instead of once per mode:
// the z pass that applies it took 178 us at n = 256, 64 and 6 for the table so)
static hipError_t ic_tables(IcWork &ws, int n, double L, const double *kt, const double *pt, int ntab, hipStream_t st) {
    hipError_t err = hipMemcpyAsync(ws.kt, kt, ntab * 8, hipMemcpyHostToDevice, st);
    if (err == hipSuccess) err = hipMemcpyAsync(ws.pt, pt, ntab * 8, hipMemcpyHostToDevice, st);
    if (err != hipSuccess) return err;
    const size_t cnt = ic_amplitudes(n);
    k_ic_amplitudes<<<g1(cnt), 256, 0, st>>>((double *)ws.amp, cnt, n, L, (const double *)ws.kt, (const double *)ws.pt,
                                             ntab);
    return hipGetLastError();
}

// phi(k) of the white noise w
static void ic_phi(IcWork &ws, FftOps &fn, const IcPasses &ic, const double *w, double L, hipStream_t st) {
    fn.xf(w, false, ws.W[0], ws.twn, 1.0, st);
    fn.yf(ws.W[0], ws.Z[0], ws.twn, st);
    ic.phi(ws, L, st);
}

// host orchestration; returns a HIP error code (0 = success)
int ics_lpt_device(IcWork &ws, int n, double L, int order, const double *white, bool white_on_device, uint32_t seed,
                   const double *kt_h, const double *pt_h, int ntab, double D, int prec, void *psi_out,
                   void *pi_out, hipStream_t st) {
    FftOps fn{};
    IcPasses ic{};
    if (!fft_dispatch<double>(n, fn) || !ic_passes(n, ic) || (order >= 2 && !ic.has_second)) return (int)hipErrorInvalidValue;
    hipError_t err = ic_work_ensure(ws, n, order, ntab);
    if (err != hipSuccess) return (int)err;
    err = ic_tables(ws, n, L, kt_h, pt_h, ntab, st);
    const bool two = order >= 2, keep = two && ic_keep_ensure(ws, n);
    ws.fk_valid = false;
    double *w = (double *)(keep && white ? ws.wkey : ws.w);  // the key of the kept fields
    if (err == hipSuccess) err = ic_white(ws, fn, n, white, white_on_device, seed, w, st);
    if (err == hipSuccess) {
        ic_phi(ws, fn, ic, w, L, st);
        if (two) {
            ic.second(ws, L, st);
            ic.source(ws, L, st);
        }
        ic.combine(ws, L, D, two, prec, psi_out, pi_out, st);
        err = hipGetLastError();
    }
    const hipError_t es = hipStreamSynchronize(st);
    if (err == hipSuccess) err = es;
    if (err == hipSuccess && keep) {
        ws.fk_valid = true;
        ws.fk_seeded = !white;
        ws.fk_seed = seed;
        ws.fk_n = n;
        ws.fk_order = order;
        ws.fk_L = L;
        ws.fk_kt.assign(kt_h, kt_h + ntab);
        ws.fk_pt.assign(pt_h, pt_h + ntab);
    }
    return (int)err;
}

// Reverse mode of ics_lpt_device: (Psibar, Pibar) of the ICs (device, precision prec) -> the white-noise
// cotangent wbar (n^3 FP64, host or device).  The A_ik's spectra are the last forward's, or computed again from phi(k).
// Each linear step is transposed: on the x-halved spectrum the r2c / c2r pair is adjoint up to the half-axis
// weights w(kx) = 1 at kx = 0 and kx = N/2, 2 otherwise (nlpt_core.jl:682-713): for y = c2r(Y) / M,
// Ybar = w r2c(ybar) / M; for Y = r2c(x), xbar = c2r(Ybar / w).  The source mu is a quadratic form whose
// cotangent per field is mubar times its partner in mu.
int ics_lpt_vjp_device(IcWork &ws, int n, double L, int order, const double *white, bool white_on_device,
                       uint32_t seed, const double *kt_h, const double *pt_h, int ntab, double D, int prec,
                       const void *psibar, const void *pibar, double *wbar, bool wbar_on_device, hipStream_t st) {
    FftOps fn{};
    IcPasses ic{};
    if (!fft_dispatch<double>(n, fn) || !ic_passes(n, ic) || (order >= 2 && !ic.has_second)) return (int)hipErrorInvalidValue;
    const size_t M = (size_t)n * n * n;
    hipError_t err = ic_work_ensure(ws, n, order, ntab);
    if (err != hipSuccess) return (int)err;
    err = ic_tables(ws, n, L, kt_h, pt_h, ntab, st);
    const bool two = order >= 2;
    // The spectra of the last forward serve when they were computed from the same inputs: n, L, order, the
    // same P(k) table values, and the same seed or white-noise values (compared bit for bit on the device)
    bool hit = two && ws.fk_valid && ws.fk_n == n && ws.fk_order == order && ws.fk_L == L &&
               ws.fk_seeded == !white && (white || ws.fk_seed == seed) && ws.fk_kt.size() == (size_t)ntab &&
               std::equal(kt_h, kt_h + ntab, ws.fk_kt.begin()) && std::equal(pt_h, pt_h + ntab, ws.fk_pt.begin());
    double *w = (double *)ws.w;
    if (err == hipSuccess && two && (!hit || white)) err = ic_white(ws, fn, n, white, white_on_device, seed, w, st);
    if (err == hipSuccess && hit && white) {
        unsigned differs = 1;
        err = hipMemsetAsync(ws.flag, 0, sizeof(unsigned), st);
        if (err == hipSuccess) {
            k_ic_differs<<<g1(M), 256, 0, st>>>((const unsigned long long *)w, (const unsigned long long *)ws.wkey, M,
                                                (unsigned *)ws.flag);
            err = hipMemcpyAsync(&differs, ws.flag, sizeof(unsigned), hipMemcpyDeviceToHost, st);
        }
        if (err == hipSuccess) err = hipStreamSynchronize(st);
        hit = err == hipSuccess && !differs;
    }
    if (err == hipSuccess && two && !hit) ic_phi(ws, fn, ic, w, L, st);
    if (err == hipSuccess) {
        ic.combine_adj(ws, L, D, two, prec, psibar, pibar, st);
        if (two) {
            ic.mu_adj(ws, L, st);
            if (!hit) {
                ws.fk_valid = false;
                ic.second(ws, L, st);
            }
            ic.source_adj(ws, L, st);
        }
        // phi = r2c(w) s(k):  wbar = c2r(phibar s / w)
        ic.phi_adj(ws, L, st);
        fn.yi(ws.Z[0], ws.W[0], ws.twn, st);
        fn.xi(ws.W[0], w, ws.twn, st);
        err = hipGetLastError();
        if (err == hipSuccess)
            err = hipMemcpyAsync(wbar, w, M * 8, wbar_on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, st);
    }
    const hipError_t es = hipStreamSynchronize(st);
    return (int)(err == hipSuccess ? es : err);
}

}  // namespace dj
