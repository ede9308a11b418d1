// Particle-side kernels of the PM step: kick, drift and the interpolation in particle order.
//
// Particles are the reference's column-major (n,n,n,3) arrays: component c of particle i + n (j + n k) is at
// that index + c n^3.
#include <hip/hip_runtime.h>

#include "dj_internal.h"
#include "stencil.h"

namespace dj {

template <typename T>
__global__ __launch_bounds__(256) void k_drift(T *__restrict__ psi, const T *__restrict__ mom, int64_t n3, T dd) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n3) psi[i] = psi[i] + dd * mom[i];
}

// out = psi + dd mom (out may be psi), the same arithmetic as k_drift; with CK, psi and mom are also
// copied to ckp and ckm as they are read (the checkpoint of a step, without copy passes of its own)
template <typename T, bool CK>
__global__ __launch_bounds__(256) void k_drift_to(T *out, const T *psi, const T *__restrict__ mom, T *__restrict__ ckp,
                                                  T *__restrict__ ckm, int64_t n3, T dd) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    const T p = psi[i], m = mom[i];
    if constexpr (CK) {
        ckp[i] = p;
        ckm[i] = m;
    }
    out[i] = p + dd * m;
}

template <typename T>
__global__ __launch_bounds__(256) void k_kick_drift(T *__restrict__ psi, T *__restrict__ mom,
                                                    const T *__restrict__ acc, int64_t n3, T alpha, T beta,
                                                    T dd2, T dd1n, int has_next, int ns, SortGate gate) {
    if (gate.closed()) return;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    T a = acc[i];
    if (ns > 1) a = a / (T)ns;
    T m = alpha * mom[i] + beta * a;
    T s = psi[i] + dd2 * m;
    if (has_next) s = s + dd1n * m;
    mom[i] = m;
    psi[i] = s;
}

// One component of the force at every particle, read from the mesh at the W^3 cells: bound by the latency of its
// scattered reads.  A tile of LDS serves them better once the particles are many, but needs the tile lists: see
// ik_in_particle_order for the line and its figures.
template <typename T, int W, int MODE>
__global__ __launch_bounds__(256) void k_gather_comp(const T *__restrict__ psi, const T *__restrict__ q1, int n, T sx,
                                                     T sy, T sz, const T *__restrict__ f, int res, T L, int comp,
                                                     T *__restrict__ acc) {
    const unsigned np = (unsigned)n * n * n, p = blockIdx.x * 256u + threadIdx.x;
    if (p >= np) return;
    const unsigned i = p % n, r = p / n, j = r % n, k = r / n;
    const T X[3] = {(psi[p] + q1[i]) + sx, (psi[p + (size_t)np] + q1[j]) + sy, (psi[p + 2 * (size_t)np] + q1[k]) + sz};
    T w[3][W];
    int c[3][W];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const T g = tjmod(X[a], L) / L * (T)res;
        const int b = twbase<W>(g) + twlo<W>();
#pragma unroll
        for (int o = 0; o < W; o++) {
            w[a][o] = twk<W>(fabs(g - (T)(b + o)));
            c[a][o] = timod(b + o, res);
        }
    }
    T s = 0;
#pragma unroll
    for (int oz = 0; oz < W; oz++)
#pragma unroll
        for (int oy = 0; oy < W; oy++) {
            const size_t row = (size_t)res * (c[1][oy] + (size_t)res * c[2][oz]);
#pragma unroll
            for (int ox = 0; ox < W; ox++) s += f[row + c[0][ox]] * (w[0][ox] * w[1][oy] * w[2][oz]);
        }
    T &out = acc[p + comp * (size_t)np];
    if constexpr (MODE == GATHER_ACC) s = out + s;
    out = s;
}

template <typename T>
__global__ __launch_bounds__(256) void k_scale(T *__restrict__ x, int64_t n, T s) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] * s;
}

__global__ __launch_bounds__(256) void k_zero(uint4 *__restrict__ x, size_t n16, uint8_t *tail, size_t ntail) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n16; i += stride) x[i] = make_uint4(0, 0, 0, 0);
    if (blockIdx.x == 0 && threadIdx.x < ntail) tail[threadIdx.x] = 0;
}

// ------------------------------------------------------------------------------------ launchers
static unsigned lgrid(int64_t n) { return (unsigned)((n + 255) / 256); }

template <typename T>
static void drift(void *psi, const void *mom, int64_t n3, double dd, hipStream_t st) {
    k_drift<T><<<lgrid(n3), 256, 0, st>>>((T *)psi, (const T *)mom, n3, (T)dd);
}

template <typename T>
static void drift_to(void *out, const void *psi, const void *mom, void *ck_psi, void *ck_mom, int64_t n3, double dd,
                     hipStream_t st) {
    if (ck_psi && ck_mom)
        k_drift_to<T, true><<<lgrid(n3), 256, 0, st>>>((T *)out, (const T *)psi, (const T *)mom, (T *)ck_psi,
                                                      (T *)ck_mom, n3, (T)dd);
    else
        k_drift_to<T, false><<<lgrid(n3), 256, 0, st>>>((T *)out, (const T *)psi, (const T *)mom, nullptr, nullptr,
                                                       n3, (T)dd);
}

template <typename T>
static void kick_drift(void *psi, void *mom, const void *acc, int64_t n3, const KickArgs &k, hipStream_t st) {
    k_kick_drift<T><<<lgrid(n3), 256, 0, st>>>((T *)psi, (T *)mom, (const T *)acc, n3, (T)k.alpha, (T)k.beta,
                                               (T)k.dd2, (T)k.dd1_next, k.has_next, k.nshifts, k.gate);
}

template <typename T>
static void gather_comp(const void *psi, const void *q1, int n, const double *sh, const void *field, int res, double L,
                        int W, int mode, int comp, void *acc, hipStream_t st) {
    auto launch = [&](auto kern) {
        kern<<<lgrid((int64_t)n * n * n), 256, 0, st>>>((const T *)psi, (const T *)q1, n, (T)sh[0], (T)sh[1], (T)sh[2],
                                                        (const T *)field, res, (T)L, comp, (T *)acc);
    };
    const bool add = mode == GATHER_ACC;
    if (W == 2) add ? launch(k_gather_comp<T, 2, GATHER_ACC>) : launch(k_gather_comp<T, 2, GATHER_ASSIGN>);
    else if (W == 3) add ? launch(k_gather_comp<T, 3, GATHER_ACC>) : launch(k_gather_comp<T, 3, GATHER_ASSIGN>);
    else add ? launch(k_gather_comp<T, 4, GATHER_ACC>) : launch(k_gather_comp<T, 4, GATHER_ASSIGN>);
}

template <typename T>
static void scale(void *x, int64_t n, double s, hipStream_t st) {
    k_scale<T><<<lgrid(n), 256, 0, st>>>((T *)x, n, (T)s);
}

static void zero(void *x, size_t bytes, hipStream_t st) {
    size_t n16 = bytes / 16, tail = bytes - n16 * 16;
    unsigned blocks = (unsigned)((n16 + 255) / 256);
    if (blocks > 65536u * 4) blocks = 65536u * 4;
    if (blocks == 0) blocks = 1;
    k_zero<<<blocks, 256, 0, st>>>((uint4 *)x, n16, (uint8_t *)x + n16 * 16, tail);
}

template <typename T> void part_ops(PartOps &ops) {
    ops.drift = drift<T>;
    ops.drift_to = drift_to<T>;
    ops.kick_drift = kick_drift<T>;
    ops.gather_comp = gather_comp<T>;
    ops.scale = scale<T>;
    ops.zero = zero;
}

template void part_ops<float>(PartOps &);
template void part_ops<double>(PartOps &);

}  // namespace dj
