// Device entry of the FFT passes (fft_passes.h) and their launchers for every supported mesh size.
#include <hip/hip_runtime.h>

#include "dj_internal.h"
#include "fft_shape.h"

namespace dj {

// Shape of the persistent z pass (k_zm_pipe): 4 waves of one line-group each, 1024 points per wave
// (4096 / N lines per workgroup), about 43 KiB of LDS with the twiddle table, three workgroups per CU;
// 384: four lines per wave, which its passes need (wave_ok), two workgroups
template <typename T, int N> struct ZPipeShape {
    static constexpr bool ok = sizeof(T) == 4 && (N == 256 || N == 384 || N == 512 || N == 1024);
    static constexpr int B = !ok ? 1 : N == 384 ? 16 : 4096 / N, NT = 256;
    using P = Passes<T, N, B, NT>;
    static constexpr int GROUPS_PER_CU = N == 384 ? 2 : 3;
};

// Each kernel runs its line FFTs wave by wave (run_wave) when the engine's pass shapes allow it,
// with workgroup barriers only around the twiddle table and the transposed (strided) side of a pass;
// otherwise every FFT pass ends with a workgroup barrier (run).
template <typename T, int N, typename IN>
__global__ __launch_bounds__(256) void k_xf(const IN *__restrict__ mesh, cx<T> *__restrict__ A,
                                            const cx<T> *__restrict__ tw, double fixed_scale) {
    using S = FftShape<T, N>;
    using P = typename S::P;
    __shared__ cx<T> lds[P::EX::LDS_ELEMS];
    // the twiddle table in LDS (read by the transforms and the post-processing; through the caches the pass took
    // 1.92 against 1.62 ms at 1024^3 in FP32, at three workgroups per CU instead of four, and 25 against 21 us at
    // 192^3, 432 against 400 us at 512^3 in FP64)
    __shared__ cx<T> twl[N];
    const cx<T> *t = stage_twiddles<T, N, true>(tw, twl, threadIdx.x, 256);
    const int lb = xcd_block(blockIdx.x, gridDim.x), yb = lb % (N / S::B), z = lb / (N / S::B);
    if constexpr (P::EX::wave_ok()) {
        P::xf_load_w(mesh, lds, yb, z, threadIdx.x, fixed_scale);
        __syncthreads();
        P::EX::template run_wave<-1, 2>(lds, t, threadIdx.x);
        __syncthreads();
    } else {
        P::xf_load(mesh, lds, yb, z, threadIdx.x, fixed_scale);
        __syncthreads();
        P::EX::template run<-1, 2>(lds, t, threadIdx.x);
    }
    P::xf_store(lds, t, A, yb, z, threadIdx.x);
}

// SC: the output multiplied by s as it is stored; MUL: the spectrum multiplied by tab[kx] as it is loaded
template <typename T, int N, bool SC = false, bool MUL = false>
__global__ __launch_bounds__((FftShape<T, N>::NTXI)) void k_xi(const cx<T> *__restrict__ A, T *__restrict__ mesh,
                                            const cx<T> *__restrict__ tw, T s = (T)1,
                                            const cx<T> *__restrict__ tab = nullptr) {
    using S = FftShape<T, N>;
    using P = typename S::PXI;
    __shared__ cx<T> lds[P::EX::LDS_ELEMS];
    // the twiddle table in LDS, staged while the block's loads are in flight (1.99 against 1.56 ms at 1024^3 in
    // FP32, 426 against 374 us at 512^3 in FP64)
    __shared__ cx<T> twl[N];
    const int lb = xcd_block(blockIdx.x, gridDim.x), yb = lb % (N / S::BXI), z = lb / (N / S::BXI);
    cx<T> va[P::XI_CNT], vb[P::XI_CNT];
    P::xi_fetch(A, yb, z, threadIdx.x, va, vb);
    const cx<T> *t = stage_twiddles<T, N, true>(tw, twl, threadIdx.x, S::NTXI);
    __syncthreads();
    P::template xi_pre<MUL>(lds, t, threadIdx.x, va, vb, tab);
    __syncthreads();
    if constexpr (P::EX::wave_ok()) {
        P::EX::template run_wave<+1, 2>(lds, t, threadIdx.x);
        P::template xi_store_w<SC>(lds, mesh, yb, z, threadIdx.x, s);
    } else {
        P::EX::template run<+1, 2>(lds, t, threadIdx.x);
        P::template xi_store<SC>(lds, mesh, yb, z, threadIdx.x, s);
    }
}

template <typename T, int N>
__global__ __launch_bounds__((FftShape<T, N>::NTY)) void k_yf(const cx<T> *__restrict__ A, cx<T> *__restrict__ Bm,
                                                             const cx<T> *__restrict__ tw) {
    using S = FftShape<T, N>;
    using P = typename S::PY;
    __shared__ cx<T> lds[P::EF::LDS_ELEMS];
    __shared__ cx<T> twl[S::TWL ? N : 1];
    const int lb = xcd_block(blockIdx.x, gridDim.x), zb = lb % (N / S::B), kx = lb / (N / S::B);
    const cx<T> *t = stage_twiddles<T, N, S::TWL>(tw, twl, threadIdx.x, S::NTY);
    if constexpr (P::EF::wave_ok()) {
        P::y_load_a_w(A, lds, zb, kx, threadIdx.x);
        __syncthreads();
        P::EF::template run_wave<-1, 1>(lds, t, threadIdx.x);
        __syncthreads();
    } else {
        P::y_load_a(A, lds, zb, kx, threadIdx.x);
        __syncthreads();
        P::EF::template run<-1, 1>(lds, t, threadIdx.x);
    }
    P::y_store_b(lds, Bm, zb, kx, threadIdx.x);
}

// MUL: the spectrum multiplied by tab[ky] as it is loaded
template <typename T, int N, bool MUL = false>
__global__ __launch_bounds__((FftShape<T, N>::NTY)) void k_yi(const cx<T> *__restrict__ Bm, cx<T> *__restrict__ A,
                                                             const cx<T> *__restrict__ tw,
                                                             const cx<T> *__restrict__ tab = nullptr) {
    using S = FftShape<T, N>;
    using P = typename S::PY;
    __shared__ cx<T> lds[P::EF::LDS_ELEMS];
    __shared__ cx<T> twl[S::TWL ? N : 1];
    const int lb = xcd_block(blockIdx.x, gridDim.x), zb = lb % (N / S::B), kx = lb / (N / S::B);
    const cx<T> *t = stage_twiddles<T, N, S::TWL>(tw, twl, threadIdx.x, S::NTY);
    P::template y_load_b<MUL>(Bm, lds, zb, kx, threadIdx.x, tab);
    __syncthreads();
    if constexpr (P::EF::wave_ok()) {
        P::EF::template run_wave<+1, 1>(lds, t, threadIdx.x);
        P::y_store_a_w(lds, A, zb, kx, threadIdx.x);
    } else {
        P::EF::template run<+1, 1>(lds, t, threadIdx.x);
        P::y_store_a(lds, A, zb, kx, threadIdx.x);
    }
}

// z lines of B: optional forward transform, multiplier, optional inverse; in may equal out
template <typename T, int N, int MODE, bool FWD, bool INV>
__global__ __launch_bounds__((FftShape<T, N>::NTY)) void k_zm(const cx<T> *in, cx<T> *out, const cx<T> *__restrict__ tw,
                                                             KMult<T> K) {
    using S = FftShape<T, N>;
    using P = typename S::PY;
    __shared__ cx<T> lds[P::EF::LDS_ELEMS];
    __shared__ cx<T> twl[S::TWL ? N : 1];
    const int b = blockIdx.x;
    const cx<T> *t = stage_twiddles<T, N, S::TWL>(tw, twl, threadIdx.x, S::NTY);
    if constexpr (P::EF::wave_ok()) {
        P::z_load_w(in, lds, b, threadIdx.x);
        __syncthreads();  // the twiddle table; from here on every wave works on its own lines
        if constexpr (FWD) P::EF::template run_wave<-1, 1>(lds, t, threadIdx.x);
        if constexpr (MODE != ZM_NONE) {
            P::template z_mult_w<MODE>(lds, K, b, threadIdx.x);
            P::EF::wave_sync();
        }
        if constexpr (INV) P::EF::template run_wave<+1, 1>(lds, t, threadIdx.x);
        P::z_store_w(lds, out, b, threadIdx.x);
    } else {
        P::z_load(in, lds, b, threadIdx.x);
        __syncthreads();
        if constexpr (FWD) P::EF::template run<-1, 1>(lds, t, threadIdx.x);
        if constexpr (MODE != ZM_NONE) {
            P::template z_mult<MODE>(lds, K, b, threadIdx.x);
            __syncthreads();
        }
        if constexpr (INV) P::EF::template run<+1, 1>(lds, t, threadIdx.x);
        P::z_store(lds, out, b, threadIdx.x);
    }
}

// The z pass of the spectral gradient: forward, times -K_phi, then two inverse transforms, of that product into
// out (the x and y components are its transforms with i k_x and i k_y, which the inverse x and y passes apply)
// and of i k_z times it into outz.  One read and two writes of the spectrum; a forward pass and three inverse
// ones made four and four (512^3, FP32: 1.06 ms against 0.46).  in may equal out.
template <typename T, int N>
__global__ __launch_bounds__((FftShape<T, N>::NTY)) void k_zm_ik(const cx<T> *in, cx<T> *out, cx<T> *__restrict__ outz,
                                                                const cx<T> *__restrict__ tw, KMult<T> K) {
    using S = FftShape<T, N>;
    using P = typename S::PY;
    constexpr int H = N / 2 + 1, NT = S::NTY;
    constexpr bool WV = P::EF::wave_ok();
    // a thread's elements: its wave's lines in steps of 64, or the tile's in steps of the workgroup
    constexpr int E = WV ? P::EF::LW * N : S::B * N, STEP = WV ? 64 : NT, CNT = (E + STEP - 1) / STEP;
    __shared__ cx<T> lds[P::EF::LDS_ELEMS];
    __shared__ cx<T> twl[S::TWL ? N : 1];
    const int b = blockIdx.x, wave = threadIdx.x >> 6;
    const int e0 = WV ? wave * E : 0, t0 = WV ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
    const cx<T> *t = stage_twiddles<T, N, S::TWL>(tw, twl, threadIdx.x, NT);
    auto sync = [&]() {
        if constexpr (WV) P::EF::wave_sync();
        else __syncthreads();
    };
    if constexpr (WV) P::z_load_w(in, lds, b, threadIdx.x);
    else P::z_load(in, lds, b, threadIdx.x);
    __syncthreads();
    if constexpr (WV) P::EF::template run_wave<-1, 1>(lds, t, threadIdx.x);
    else P::EF::template run<-1, 1>(lds, t, threadIdx.x);
    cx<T> gz[CNT];
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = e0 + t0 + STEP * c, l = i / N, kz = i - l * N;
        if (E % STEP != 0 && t0 + STEP * c >= E) continue;
        const int L = b * S::B + l, ky = L / H, kx = L - ky * H;
        const cx<T> v = scale(lds[P::EF::idx(l, kz)], -K.kphi(kx, ky, kz));
        lds[P::EF::idx(l, kz)] = v;
        const T k = K.gf[kz].y;  // i k_z, its Nyquist zeroed
        gz[c] = {-(k * v.y), k * v.x};
    }
    sync();
    auto inverse_to = [&](cx<T> *dst) {
        if constexpr (WV) {
            P::EF::template run_wave<+1, 1>(lds, t, threadIdx.x);
            P::z_store_w(lds, dst, b, threadIdx.x);
        } else {
            P::EF::template run<+1, 1>(lds, t, threadIdx.x);
            P::z_store(lds, dst, b, threadIdx.x);
        }
    };
    inverse_to(out);
    sync();
#pragma unroll
    for (int c = 0; c < CNT; c++) {
        const int i = e0 + t0 + STEP * c, l = i / N;
        if (E % STEP != 0 && t0 + STEP * c >= E) continue;
        lds[P::EF::idx(l, i - l * N)] = gz[c];
    }
    sync();
    inverse_to(outz);
}

// The inverse z pass of lines multiplied by tab[kz] as they are loaded
template <typename T, int N>
__global__ __launch_bounds__((FftShape<T, N>::NTY)) void k_zi_mul(const cx<T> *__restrict__ in, cx<T> *__restrict__ out,
                                                                 const cx<T> *__restrict__ tw,
                                                                 const cx<T> *__restrict__ tab) {
    using S = FftShape<T, N>;
    using P = typename S::PY;
    __shared__ cx<T> lds[P::EF::LDS_ELEMS];
    __shared__ cx<T> twl[S::TWL ? N : 1];
    const int b = blockIdx.x;
    const cx<T> *t = stage_twiddles<T, N, S::TWL>(tw, twl, threadIdx.x, S::NTY);
    const auto src = [&](size_t e) { return cmul(in[e], tab[(unsigned)(e % N)]); };
    if constexpr (P::EF::wave_ok()) {
        P::z_load_src_w(src, lds, b, threadIdx.x);
        __syncthreads();  // the twiddle table; from here on every wave works on its own lines
        P::EF::template run_wave<+1, 1>(lds, t, threadIdx.x);
        P::z_store_w(lds, out, b, threadIdx.x);
    } else {
        P::z_load_src(src, lds, b, threadIdx.x);
        __syncthreads();
        P::EF::template run<+1, 1>(lds, t, threadIdx.x);
        P::z_store(lds, out, b, threadIdx.x);
    }
}

// The z pass as a persistent kernel (three workgroups per CU, block b, b + G, b + 2G, ... for G
// workgroups): each wave holds the next block's lines in registers while it transforms and stores
// the current block's, so a block's loads overlap the previous block's transforms and stores
// instead of waiting for another workgroup on the CU.  The multiplier's kz-dependent table values
// are the same for every block and are read once; the per-line ones (kx, ky) are read before the
// next block's loads are issued, so that waiting for them does not wait for those loads.  The
// arithmetic of the multiplier is KMult::kphi's, in its order.  FP32 on 256^3 to 1024^3 meshes (a
// lane's elements keep one kz per step; 384^3: 179 -> 100 us; in FP64 the held lines take the registers of a
// wave's transforms: 192^3 37 -> 46 us, 512^3 613 -> 657), the potential multiplier without window deconvolution or
// transfer function.
template <typename T, int N, int MODE, bool FWD, bool INV>
__global__ __launch_bounds__((ZPipeShape<T, N>::NT), (ZPipeShape<T, N>::GROUPS_PER_CU)) void k_zm_pipe(
    const cx<T> *in, cx<T> *out, const cx<T> *__restrict__ tw, KMult<T> K, int nblocks) {
    using S = ZPipeShape<T, N>;
    using P = typename S::P;
    using EF = typename P::EF;
    constexpr int B = S::B, H = N / 2 + 1, LW = EF::LW, E = LW * N, CNT = E / 64;
    static_assert(N % 64 == 0 && E % 64 == 0 && EF::wave_ok(), "lanes keep one kz per step");
    __shared__ cx<T> lds[EF::LDS_ELEMS];
    __shared__ cx<T> twl[N];
    const cx<T> *t = stage_twiddles<T, N, true>(tw, twl, threadIdx.x, S::NT);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool lap0 = K.lap_order == 0;
    // element c of a lane: wave line wave LW + (64 c) / N, kz = (64 c) % N + lane
    T zt[CNT];
    if constexpr (MODE == ZM_POT) {
#pragma unroll
        for (int c = 0; c < CNT; c++) {
            const int kz = (64 * c) % N + lane;
            zt[c] = lap0 ? K.k2f[kz] : K.tf[kz];
        }
    }
    cx<T> pf[CNT];
    auto fetch = [&](int blk) {
        const cx<T> *src = in + (size_t)N * B * blk + (size_t)wave * E;
#pragma unroll
        for (int c = 0; c < CNT; c++) pf[c] = src[lane + 64 * c];
    };
    int b = blockIdx.x;
    if (b < nblocks) fetch(b);
    __syncthreads();  // the twiddle table
    while (b < nblocks) {
#pragma unroll
        for (int c = 0; c < CNT; c++) lds[EF::idx(wave * LW + (64 * c) / N, (64 * c) % N + lane)] = pf[c];
        // per-line multiplier parts: th[kx] + tf[ky] (or k2h[kx] + k2f[ky])
        T lt[LW];
        int lkx[LW], lky[LW];
        if constexpr (MODE == ZM_POT) {
#pragma unroll
            for (int w = 0; w < LW; w++) {
                const int L = b * B + wave * LW + w, ky = L / H, kx = L - ky * H;
                lkx[w] = kx;
                lky[w] = ky;
                lt[w] = lap0 ? K.k2h[kx] + K.k2f[ky] : K.th[kx] + K.tf[ky];
            }
        }
        const int bn = b + (int)gridDim.x;
        if (bn < nblocks) fetch(bn);
        EF::wave_sync();
        if constexpr (FWD) EF::template run_wave<-1, 1>(lds, t, threadIdx.x);
        if constexpr (MODE == ZM_POT) {
#pragma unroll
            for (int c = 0; c < CNT; c++) {
                const int w = (64 * c) / N, kz = (64 * c) % N + lane;
                const int i = EF::idx(wave * LW + w, kz);
                T kp;
                if (lkx[w] == 0 && lky[w] == 0 && kz == 0) {
                    kp = (T)0;
                } else {
                    const T il = lap0 ? (T)-1 / (lt[w] + zt[c]) : (T)1 / (lt[w] + zt[c]);
                    kp = il * K.scale;
                }
                lds[i] = scale(lds[i], kp);
            }
            EF::wave_sync();
        }
        if constexpr (INV) EF::template run_wave<+1, 1>(lds, t, threadIdx.x);
        cx<T> *dst = out + (size_t)N * B * b + (size_t)wave * E;
#pragma unroll
        for (int c = 0; c < CNT; c++) dst[lane + 64 * c] = lds[EF::idx(wave * LW + (64 * c) / N, (64 * c) % N + lane)];
        EF::wave_sync();  // the reads above before the next block's writes
        b = bn;
    }
}

// workgroups of the persistent z pass: per_cu on every CU of the current device, a multiple of 8
static int persistent_groups(int per_cu, int nb) {
    static int cus = 0;
    if (!cus) {
        int dev = 0, n = 0;
        cus = (hipGetDevice(&dev) == hipSuccess &&
               hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
                  ? n
                  : 256;
    }
    int g = ((per_cu * cus) / 8) * 8;
    if (g < 8) g = 8;
    return g < nb ? g : nb;
}

template <typename T, int N>
struct FftN {
    using S = FftShape<T, N>;
    using P = typename S::P;
    static void xf(const void *mesh, bool fixed, void *A, const void *tw, double fscale, hipStream_t st) {
        if (fixed)
            k_xf<T, N, long long><<<P::XBLOCKS(), 256, 0, st>>>((const long long *)mesh, (cx<T> *)A,
                                                               (const cx<T> *)tw, fscale);
        else
            k_xf<T, N, T><<<P::XBLOCKS(), 256, 0, st>>>((const T *)mesh, (cx<T> *)A, (const cx<T> *)tw, fscale);
    }
    static void zm_ik(const void *in, void *out, void *outz, const void *tw, const void *Kp, hipStream_t st) {
        k_zm_ik<T, N><<<P::ZBLOCKS(), S::NTY, 0, st>>>((const cx<T> *)in, (cx<T> *)out, (cx<T> *)outz, (const cx<T> *)tw,
                                                       *(const KMult<T> *)Kp);
    }
    static void zi_mul(const void *in, void *out, const void *tw, const void *tab, hipStream_t st) {
        k_zi_mul<T, N><<<P::ZBLOCKS(), S::NTY, 0, st>>>((const cx<T> *)in, (cx<T> *)out, (const cx<T> *)tw,
                                                        (const cx<T> *)tab);
    }
    static void yi_mul(const void *Bm, void *A, const void *tw, const void *tab, hipStream_t st) {
        k_yi<T, N, true><<<P::YBLOCKS(), S::NTY, 0, st>>>((const cx<T> *)Bm, (cx<T> *)A, (const cx<T> *)tw,
                                                          (const cx<T> *)tab);
    }
    static void xi_mul(const void *A, void *mesh, const void *tw, const void *tab, double s, hipStream_t st) {
        using PX = typename S::PXI;
        k_xi<T, N, true, true><<<PX::XBLOCKS(), S::NTXI, 0, st>>>((const cx<T> *)A, (T *)mesh, (const cx<T> *)tw, (T)s,
                                                                  (const cx<T> *)tab);
    }
    static void xi(const void *A, void *mesh, const void *tw, hipStream_t st) {
        using PX = typename S::PXI;
        k_xi<T, N><<<PX::XBLOCKS(), S::NTXI, 0, st>>>((const cx<T> *)A, (T *)mesh, (const cx<T> *)tw);
    }
    static void xi_scaled(const void *A, void *mesh, const void *tw, double s, hipStream_t st) {
        using PX = typename S::PXI;
        k_xi<T, N, true><<<PX::XBLOCKS(), S::NTXI, 0, st>>>((const cx<T> *)A, (T *)mesh, (const cx<T> *)tw, (T)s);
    }
    static void yf(const void *A, void *Bm, const void *tw, hipStream_t st) {
        k_yf<T, N><<<P::YBLOCKS(), S::NTY, 0, st>>>((const cx<T> *)A, (cx<T> *)Bm, (const cx<T> *)tw);
    }
    static void yi(const void *Bm, void *A, const void *tw, hipStream_t st) {
        k_yi<T, N><<<P::YBLOCKS(), S::NTY, 0, st>>>((const cx<T> *)Bm, (cx<T> *)A, (const cx<T> *)tw);
    }
    static void zm(int mode, bool fwd, bool inv, const void *in, void *out, const void *tw, const void *Kp,
                   hipStream_t st) {
        const KMult<T> &K = *(const KMult<T> *)Kp;
        const cx<T> *i = (const cx<T> *)in;
        cx<T> *o = (cx<T> *)out;
        const cx<T> *t = (const cx<T> *)tw;
        dim3 g(P::ZBLOCKS()), b(S::NTY);
        if constexpr (ZPipeShape<T, N>::ok) {
            if (mode == ZM_POT && fwd && inv && !K.kg && !K.mf) {
                using ZP = ZPipeShape<T, N>;
                const int nb = ZP::P::ZBLOCKS();
                k_zm_pipe<T, N, ZM_POT, true, true><<<persistent_groups(ZP::GROUPS_PER_CU, nb), ZP::NT, 0, st>>>(i, o, t, K, nb);
                return;
            }
        }
#define ZM(M, F, I) k_zm<T, N, M, F, I><<<g, b, 0, st>>>(i, o, t, K)
        if (mode == ZM_POT && fwd && inv) ZM(ZM_POT, true, true);
        else if (mode == ZM_NONE && fwd && !inv) ZM(ZM_NONE, true, false);
        else if (mode == ZM_NONE && !fwd && inv) ZM(ZM_NONE, false, true);
        else if (mode == ZM_NONE && fwd && inv) ZM(ZM_NONE, true, true);
        else if (mode == ZM_GRADX && !fwd && inv) ZM(ZM_GRADX, false, true);
        else if (mode == ZM_GRADY && !fwd && inv) ZM(ZM_GRADY, false, true);
        else if (mode == ZM_GRADZ && !fwd && inv) ZM(ZM_GRADZ, false, true);
#undef ZM
    }
};

template <typename T>
bool fft_dispatch(int N, FftOps &ops) {
#define CASE(n)                         \
    case n:                             \
        ops.xf = FftN<T, n>::xf;        \
        ops.xi = FftN<T, n>::xi;        \
        ops.xi_scaled = FftN<T, n>::xi_scaled; \
        ops.xi_mul = FftN<T, n>::xi_mul; \
        ops.yi_mul = FftN<T, n>::yi_mul; \
        ops.zi_mul = FftN<T, n>::zi_mul; \
        ops.zm_ik = FftN<T, n>::zm_ik; \
        ops.yf = FftN<T, n>::yf;        \
        ops.yi = FftN<T, n>::yi;        \
        ops.zm = FftN<T, n>::zm;        \
        ops.lines_per_block = FftN<T, n>::S::B; \
        return true;
    switch (N) {
        CASE(16) CASE(24) CASE(32) CASE(48) CASE(64) CASE(96) CASE(128) CASE(192) CASE(256) CASE(384)
        CASE(512) CASE(768) CASE(1024)
    }
#undef CASE
    return false;
}

template bool fft_dispatch<float>(int, FftOps &);
template bool fft_dispatch<double>(int, FftOps &);

}  // namespace dj
