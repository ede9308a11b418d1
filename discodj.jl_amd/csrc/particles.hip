// Particle-side kernels of the PM step: kick and drift.
//
// Particles are the reference's column-major (n,n,n,3) arrays: component c of particle i + n (j + n k) is at
// that index + c n^3.
#include <hip/hip_runtime.h>

#include "dj_internal.h"

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
    ops.scale = scale<T>;
    ops.zero = zero;
}

template void part_ops<float>(PartOps &);
template void part_ops<double>(PartOps &);

}  // namespace dj
