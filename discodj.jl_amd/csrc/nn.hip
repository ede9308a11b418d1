// Learned force correction: a residual 3-D convolution net on the PM mesh, BF16 weights and
// activations, FP32 accumulation on MFMA (v_mfma_f32_16x16x16bf16_1k).  There is no counterpart in the
// reference; the net adds a potential correction to the PM potential before the gradient and the gather.
//
//   x0 = (log(1 + max(delta, -0.999)), a)            delta = mesh / rho_bar - 1, a = scale factor
//   z1 = W1 * x0 + b1,  h1 = relu(z1)
//   z2 = W2 * h1 + b2,  h2 = h1 + relu(z2)
//   z3 = W3 * h2 + b3,  h3 = h2 + relu(z3)
//   dphi = s_out (W4 * h3 + b4)                       (*: periodic 3x3x3 convolution, 16 channels)
//
// Tensors are channel-last: t[v * 16 + c], v = x + N (y + N z), BF16 (round to nearest even).  Every
// layer is stored as W[27][16][16] (tap, out, in) padded with zeros (layer 1 has 2 inputs, layer 4 one
// output).  One wave computes 16 output channels of 16 voxels of an x row: per tap one MFMA with
// A = the tap's weights (16 out x 16 in) and B = the 16 voxels' input channels; the transposed
// convolution of the backward pass is the same kernel with the flipped, transposed taps.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dj_internal.h"

namespace dj {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

// FP32 -> BF16 round to nearest even (the conversion instruction); BF16 -> FP32 exact
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned short f2bf(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }
__device__ __forceinline__ s4v f2bf4(f4v x) { return __builtin_bit_cast(s4v, __builtin_convertvector(x, bf4)); }
__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

__device__ __forceinline__ float nn_input(float dens, float inv_rho) {
    const float d = dens * inv_rho - 1.0f;
    return log1pf(fmaxf(d, -0.999f));
}

__device__ __forceinline__ int nn_wrap(int v, int N) { return v < 0 ? v + N : (v >= N ? v - N : v); }

enum { NN_IN_H = 0, NN_IN_FIELD = 1, NN_IN_GRAD = 2 };  // B: 16-channel tensor / density field / 1-channel float
enum { NN_EPI_HIDDEN = 0, NN_EPI_OUT = 1, NN_EPI_BWD = 2 };
enum { NN_RES_NONE = 0, NN_RES_INPUT = 1, NN_RES_TENSOR = 2 };  // the residual: none, the layer's input, another tensor

// One block marches along z over a 64 (x) x 8 (y) footprint: the input planes z-1, z, z+1 (with a one-voxel x-y
// halo, 66 x 10 voxels) sit in a three-slot LDS ring, so each input voxel is read from memory about 1.3 times
// instead of once per tap.  Two blocks share a CU (64.5 KiB of LDS each).  Wave w computes y rows 2w, 2w+1 of the
// plane (8 segments of 16 voxels), per tap one MFMA per segment.  The taps' weights (A) stay in registers for
// the whole march; an input row (B) is read from LDS once for the two output rows that use it (48 reads of 8
// bytes a lane and input plane instead of 72); and the plane after the next is loaded into registers while the
// current one is computed, so a plane costs its MFMAs (16 cycles each, 216 a wave) and not the loads' latency.
// Every output adds its taps in the order dz, dy, dx.  Hidden layer at 256^3: 0.34 ms (matrix cores 62 % busy),
// against 0.56 with A in LDS, every tap its own read and the loads before the barrier; first layer 0.17 (0.35),
// last 0.27 (0.41).
constexpr int NN_TX = 64, NN_TY = 8, NN_PX = NN_TX + 2, NN_PY = NN_TY + 2, NN_PV = NN_PX * NN_PY;
// A 16-channel plane in LDS is four planes of 8-byte units (4 channels), NN_PVP units apart: a wave's read of 16
// neighbouring voxels' units in each is 4 x 128 contiguous bytes that meet no bank twice (NN_PVP = 16 mod 32
// puts neighbouring channel groups on the two halves of the 64 banks).  Channel-last voxels, 32 bytes apart,
// made 30 LDS cycles of every 8.
constexpr int NN_PVP = 688;
static_assert(NN_PVP >= NN_PV && NN_PVP % 32 == 16, "channel planes on alternating bank halves");

// This thread's part of an input plane of the footprint: PER units in registers between load() and store().
// 16-channel tensors move in 16-byte halves of a voxel; a field becomes one 4-byte pair (bf16(input),
// bf16(cval)) per voxel (gradient field: scaled by inv_rho).
template <int IN> struct PlaneStage {
    static constexpr bool H = IN == NN_IN_H;
    static constexpr int UNITS = H ? 2 * NN_PV : NN_PV, PER = (UNITS + 255) / 256;
    using Unit = typename std::conditional<H, uint4, float>::type;
    unsigned off[PER];  // of the unit in the plane (units of 8 channels, or voxels)
    Unit v[PER];
    __device__ __forceinline__ void init(int N, int x0, int y0) {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int u = min((int)threadIdx.x + 256 * k, UNITS - 1), vox = H ? u >> 1 : u;
            const int xi = vox % NN_PX, yi = vox / NN_PX;
            const unsigned p = (unsigned)nn_wrap(x0 - 1 + xi, N) + (unsigned)N * (unsigned)nn_wrap(y0 - 1 + yi, N);
            off[k] = H ? 2 * p + (u & 1) : p;
        }
    }
    __device__ __forceinline__ void load(const unsigned short *hin, const float *fin, int N, int z) {
        const size_t zb = (size_t)N * N * nn_wrap(z, N);
#pragma unroll
        for (int k = 0; k < PER; k++) {
            if constexpr (H) v[k] = ((const uint4 *)hin)[2 * zb + off[k]];
            else v[k] = fin[zb + off[k]];
        }
    }
    __device__ __forceinline__ void store(unsigned short *slot, float inv_rho, unsigned c1) const {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int u = threadIdx.x + 256 * k;
            if (u >= UNITS) continue;
            if constexpr (H) {
                uint2 *d = (uint2 *)slot + (u & 1) * (2 * NN_PVP) + (u >> 1);
                d[0] = make_uint2(v[k].x, v[k].y);
                d[NN_PVP] = make_uint2(v[k].z, v[k].w);
            } else {
                const float x = IN == NN_IN_FIELD ? nn_input(v[k], inv_rho) : v[k] * inv_rho;
                ((unsigned *)slot)[u] = (unsigned)f2bf(x) | c1;
            }
        }
    }
};
template <int IN> constexpr size_t nn_conv_lds() { return 3 * (IN == NN_IN_H ? (size_t)NN_PVP * 32 : (size_t)NN_PV * 4); }

template <int IN, int EPI, int RES>
__global__ __launch_bounds__(256, 2) void k_nn_conv(int N, int tz, const unsigned short *__restrict__ hin,
                                                    const float *__restrict__ fin, float inv_rho, float cval,
                                                    const s4v *__restrict__ wsw, const float *__restrict__ bias,
                                                    const unsigned short *__restrict__ res,
                                                    const unsigned short *__restrict__ zmask,
                                                    unsigned short *__restrict__ out_z, unsigned short *__restrict__ out_h,
                                                    float *__restrict__ out_f, float oscale) {
    extern __shared__ unsigned char nn_smem[];
    constexpr int SLOT = IN == NN_IN_H ? NN_PVP * 16 : NN_PV * 2, NA = IN == NN_IN_H ? 27 : 4;
    unsigned short *ring = (unsigned short *)nn_smem;  // 3 planes
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, cg = 4 * (lane >> 4), lx = lane & 15;
    const int nbx = N / NN_TX, nby = N / NN_TY;
    const int x0 = (blockIdx.x % nbx) * NN_TX, y0 = ((blockIdx.x / nbx) % nby) * NN_TY,
              z0 = (blockIdx.x / (nbx * nby)) * tz;
    s4v a[NA];
#pragma unroll
    for (int t = 0; t < NA; t++) a[t] = wsw[t * 64 + lane];
    float bs[4] = {0, 0, 0, 0};
    if constexpr (EPI == NN_EPI_HIDDEN) {
#pragma unroll
        for (int j = 0; j < 4; j++) bs[j] = bias[cg + j];
    } else if constexpr (EPI == NN_EPI_OUT) {
        bs[0] = bias[0];
    }
    const unsigned c1 = (unsigned)f2bf(cval) << 16;
    PlaneStage<IN> st;
    st.init(N, x0, y0);
    // slots of planes z-1, z, z+1
    unsigned short *s0 = ring, *s1 = ring + SLOT, *s2 = ring + 2 * SLOT;
    st.load(hin, fin, N, z0 - 1);
    st.store(s0, inv_rho, c1);
    st.load(hin, fin, N, z0);
    st.store(s1, inv_rho, c1);
    st.load(hin, fin, N, z0 + 1);
    for (int z = z0; z < z0 + tz; z++) {
        st.store(s2, inv_rho, c1);
        if (z + 1 < z0 + tz) st.load(hin, fin, N, z + 2);
        __syncthreads();  // planes z-1, z, z+1 in LDS
        f4v acc[8];
#pragma unroll
        for (int sg = 0; sg < 8; sg++) acc[sg] = {0, 0, 0, 0};
        if constexpr (IN == NN_IN_H) {
#pragma unroll
            for (int dz = 0; dz < 3; dz++) {
                const s4v *sh = (const s4v *)(dz == 0 ? s0 : dz == 1 ? s1 : s2) + (lane >> 4) * NN_PVP +
                                2 * wave * NN_PX + lx;
#pragma unroll
                for (int yr = 0; yr < 4; yr++)  // input rows 2w - 1 + yr: dy = yr of row 2w, yr - 1 of row 2w + 1
#pragma unroll
                    for (int dx = 0; dx < 3; dx++) {
                        s4v b[4];
#pragma unroll
                        for (int sg = 0; sg < 4; sg++) b[sg] = sh[yr * NN_PX + sg * 16 + dx];
                        if (yr < 3)
#pragma unroll
                            for (int sg = 0; sg < 4; sg++)
                                acc[sg] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[dz * 9 + yr * 3 + dx], b[sg],
                                                                                   acc[sg], 0, 0, 0);
                        if (yr > 0)
#pragma unroll
                            for (int sg = 0; sg < 4; sg++)
                                acc[4 + sg] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[dz * 9 + (yr - 1) * 3 + dx],
                                                                                       b[sg], acc[4 + sg], 0, 0, 0);
                    }
            }
        } else {
            // two input channels: one MFMA takes 8 taps x 2 channels (K = 16), 4 MFMAs for the 27 taps
            // (the 5 extra taps have zero weights); lane k-group 4 (lane / 16) + j reads taps
            // 8 q + 2 (lane / 16) + j / 2, channel j % 2
            auto slot = [&](int dz) { return (const unsigned *)(dz == 0 ? s0 : dz == 1 ? s1 : s2); };
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int t1 = min(8 * q + 2 * (lane >> 4), 26), t2 = min(t1 + 1, 26);
                const unsigned *p1 = slot(t1 / 9) + ((t1 / 3) % 3) * NN_PX + t1 % 3 + 2 * wave * NN_PX + lx,
                               *p2 = slot(t2 / 9) + ((t2 / 3) % 3) * NN_PX + t2 % 3 + 2 * wave * NN_PX + lx;
#pragma unroll
                for (int sg = 0; sg < 8; sg++) {
                    const int v0 = (sg >> 2) * NN_PX + (sg & 3) * 16;
                    const unsigned u1 = p1[v0], u2 = p2[v0];
                    const s4v b = {(short)(u1 & 0xffffu), (short)(u1 >> 16), (short)(u2 & 0xffffu), (short)(u2 >> 16)};
                    acc[sg] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[q], b, acc[sg], 0, 0, 0);
                }
            }
        }
        // epilogue: lane holds D[cg + j][lx] of each segment: channels cg..cg+3 of one voxel.  What it reads from
        // memory is read for all segments before the first store (a wait for a load waits for earlier stores).
        auto voxel = [&](int sg) {
            return (size_t)(x0 + (sg & 3) * 16 + lx) +
                   (size_t)N * ((size_t)(y0 + 2 * wave + (sg >> 2)) + (size_t)N * z);
        };
        if constexpr (EPI == NN_EPI_OUT) {
            if (cg == 0)
#pragma unroll
                for (int sg = 0; sg < 8; sg++) out_f[voxel(sg)] = oscale * (acc[sg][0] + bs[0]);
        } else {
            s4v rr[8], m[8];
#pragma unroll
            for (int sg = 0; sg < 8; sg++) {
                if constexpr (RES == NN_RES_INPUT)  // its centre cell is in the LDS ring
                    rr[sg] = ((const s4v *)s1)[(lane >> 4) * NN_PVP + (2 * wave + (sg >> 2) + 1) * NN_PX +
                                               (sg & 3) * 16 + lx + 1];
                else if constexpr (RES == NN_RES_TENSOR) rr[sg] = *(const s4v *)(res + voxel(sg) * 16 + cg);
                else rr[sg] = {0, 0, 0, 0};
                if constexpr (EPI == NN_EPI_BWD) m[sg] = *(const s4v *)(zmask + voxel(sg) * 16 + cg);
            }
#pragma unroll
            for (int sg = 0; sg < 8; sg++) {
                f4v zo, ho;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float rv = bf2f((unsigned short)rr[sg][j]);
                    if constexpr (EPI == NN_EPI_HIDDEN) {
                        const float zz = acc[sg][j] + bs[j];
                        zo[j] = zz;
                        ho[j] = rv + fmaxf(zz, 0.0f);
                    } else {
                        const float g = rv + acc[sg][j];
                        ho[j] = g;
                        zo[j] = bf2f((unsigned short)m[sg][j]) > 0.0f ? g : 0.0f;
                    }
                }
                if (out_z) *(s4v *)(out_z + voxel(sg) * 16 + cg) = f2bf4(zo);  // pre-activations: kept for training only
                *(s4v *)(out_h + voxel(sg) * 16 + cg) = f2bf4(ho);
            }
        }
        __syncthreads();  // plane z - 1's slot takes plane z + 2 next
        unsigned short *t = s0;
        s0 = s1;
        s1 = s2;
        s2 = t;
    }
}

// One block's partial weight and bias gradients (27 x 16 x 16 + 16 floats), and the slices of blocks the
// first reduction pass sums
constexpr int NN_WP = 27 * 16 * 16 + 16, NN_WSLICES = 16, NN_WBLOCKS = 2048;

// Weight gradient dW[t][co][ci] += sum_v gz(v, co) x(v + off(t), ci) and db[co] += sum_v gz(v, co).
// A block takes rows of 64 voxels (x chunks), stages gz (64 x 16) and the 9 neighbouring input rows
// (66 x 16 each, periodic) in LDS, and each of its 4 waves accumulates the MFMAs of taps w, w+4, ...
// over the voxels (K = 16 voxels per MFMA) in registers.  Each block writes its sums to its row of part,
// and k_nn_wreduce1/2 add the rows in a fixed order: no atomics, so a training run repeats bit for bit.
template <int IN, int GA>
__global__ __launch_bounds__(256) void k_nn_wgrad(int N, const unsigned short *__restrict__ hin, const float *__restrict__ fin,
                                                  float inv_rho, float cval, const unsigned short *__restrict__ gz,
                                                  const float *__restrict__ gf, float gscale, float *__restrict__ part) {
    __shared__ unsigned short sA[64 * 16];
    __shared__ unsigned short sB[9 * 66 * 16];
    __shared__ float sdbp[4][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int chunks = N / 64, nrows = chunks * N * N;
    float dbacc = 0;  // threads < 16: channel threadIdx.x's bias gradient over the block's rows, in row order
    f4v acc[7];
#pragma unroll
    for (int i = 0; i < 7; i++) acc[i] = {0, 0, 0, 0};
    for (int r = blockIdx.x; r < nrows; r += gridDim.x) {
        const int x0 = (r % chunks) * 64, y = (r / chunks) % N, z = r / (chunks * N);
        __syncthreads();  // previous row's LDS reads are done
        // the previous row's four partial bias sums, in order (written before that row's MFMAs)
        if (r != (int)blockIdx.x && threadIdx.x < 16)
            dbacc += ((sdbp[0][threadIdx.x] + sdbp[1][threadIdx.x]) + sdbp[2][threadIdx.x]) + sdbp[3][threadIdx.x];
        // gz of the row: 64 voxels x 16 channels (GA: a 1-channel float field in channel 0, scaled)
        for (int e = threadIdx.x; e < 64 * 16; e += 256) {
            const int vx = e >> 4, c = e & 15;
            const size_t v = (size_t)(x0 + vx) + (size_t)N * ((size_t)y + (size_t)N * z);
            unsigned short g;
            if constexpr (GA) g = c == 0 ? f2bf(gscale * gf[v]) : (unsigned short)0;
            else g = gz[v * 16 + c];
            sA[e] = g;
        }
        // the input rows (y + dy, z + dz), x from x0 - 1 to x0 + 64
        for (int e = threadIdx.x; e < 9 * 66 * 16; e += 256) {
            const int c = e & 15, xi = (e >> 4) % 66, rr = (e >> 4) / 66;
            const int yy = nn_wrap(y + rr % 3 - 1, N), zz = nn_wrap(z + rr / 3 - 1, N), xx = nn_wrap(x0 + xi - 1, N);
            const size_t v = (size_t)xx + (size_t)N * ((size_t)yy + (size_t)N * zz);
            unsigned short h;
            if constexpr (IN == NN_IN_H) h = hin[v * 16 + c];
            else h = c == 0 ? f2bf(nn_input(fin[v], inv_rho)) : (c == 1 ? f2bf(cval) : (unsigned short)0);
            sB[e] = h;
        }
        __syncthreads();
        if (threadIdx.x < 64) {  // bias: one channel per 4 threads, 16 voxels each
            const int c = threadIdx.x & 15, q = threadIdx.x >> 4;
            float s = 0;
            for (int vx = q * 16; vx < q * 16 + 16; vx++) s += bf2f(sA[vx * 16 + c]);
            sdbp[q][c] = s;
        }
        const int cg = 4 * (lane >> 4), cl = lane & 15;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
            s4v a;
#pragma unroll
            for (int j = 0; j < 4; j++) a[j] = (short)sA[(kc * 16 + cg + j) * 16 + cl];
#pragma unroll
            for (int i = 0; i < 7; i++) {
                const int t = wave + 4 * i;
                if (t < 27) {
                    const int dx = t % 3 - 1, rr = t / 3;  // rr = (dz + 1) 3 + (dy + 1)
                    s4v b;
#pragma unroll
                    for (int j = 0; j < 4; j++) b[j] = (short)sB[(rr * 66 + kc * 16 + cg + j + dx + 1) * 16 + cl];
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[i], 0, 0, 0);
                }
            }
        }
    }
    // D[co = cg + j][ci = lane & 15] of tap t: each element is one lane's
    float *mine = part + (size_t)blockIdx.x * NN_WP;
    const int cg = 4 * (lane >> 4), cl = lane & 15;
#pragma unroll
    for (int i = 0; i < 7; i++) {
        const int t = wave + 4 * i;
        if (t < 27) {
#pragma unroll
            for (int j = 0; j < 4; j++) mine[(t * 16 + cg + j) * 16 + cl] = acc[i][j];
        }
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        if ((int)blockIdx.x < nrows)  // the last row's partial sums
            dbacc += ((sdbp[0][threadIdx.x] + sdbp[1][threadIdx.x]) + sdbp[2][threadIdx.x]) + sdbp[3][threadIdx.x];
        mine[27 * 16 * 16 + threadIdx.x] = dbacc;
    }
}

// Fixed-order sums of the blocks' rows of part: slice y of the nb rows into part2[y] (each thread sums
// rows g, g + 4, ... of the slice, then the four threads' sums in order), then the slices in order into
// dW (the first 27 x 16 x 16 values) and db
__global__ __launch_bounds__(256) void k_nn_wreduce1(const float *__restrict__ part, int nb, float *__restrict__ part2) {
    __shared__ float s4[4][64];
    const int o = threadIdx.x & 63, g = threadIdx.x >> 6, i = blockIdx.x * 64 + o;
    const int per = (nb + NN_WSLICES - 1) / NN_WSLICES, b0 = blockIdx.y * per, b1 = min(nb, b0 + per);
    float a = 0;
    if (i < NN_WP)
        for (int b = b0 + g; b < b1; b += 4) a += part[(size_t)b * NN_WP + i];
    s4[g][o] = a;
    __syncthreads();
    if (g == 0 && i < NN_WP) part2[(size_t)blockIdx.y * NN_WP + i] = ((s4[0][o] + s4[1][o]) + s4[2][o]) + s4[3][o];
}
__global__ __launch_bounds__(256) void k_nn_wreduce2(const float *__restrict__ part2, float *__restrict__ dW,
                                                     float *__restrict__ db) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NN_WP) return;
    float a = 0;
    for (int sl = 0; sl < NN_WSLICES; sl++) a += part2[(size_t)sl * NN_WP + i];
    if (i < 27 * 16 * 16) dW[i] += a;
    else db[i - 27 * 16 * 16] += a;
}

// lane-ordered BF16 A operands of the forward (W[t][co][ci] at lane (co, ci / 4)) and of the
// transposed convolution (W[26 - t][co][ci] at lane (ci, co / 4)) of one layer
// packed A operands of a two-channel input (8 taps x 2 channels per K = 16): forward A[co][k] =
// W[t][co][ch], transposed A[ci][k] = W[26 - t][ch][ci], t = 8 q + 2 (k / 4) + (k % 4) / 2, ch = k % 2,
// zero for t >= 27
__global__ void k_nn_swizzle_packed(const float *__restrict__ W, s4v *__restrict__ fwd, s4v *__restrict__ bwd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4 * 64) return;
    const int q = i / 64, l = i % 64, row = l & 15;
    s4v f, b;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int t = 8 * q + 2 * (l >> 4) + j / 2, ch = j % 2;
        f[j] = (short)(t < 27 ? f2bf(W[(t * 16 + row) * 16 + ch]) : 0);
        b[j] = (short)(t < 27 ? f2bf(W[((26 - t) * 16 + ch) * 16 + row]) : 0);
    }
    fwd[i] = f;
    bwd[i] = b;
}

__global__ void k_nn_swizzle(const float *__restrict__ W, s4v *__restrict__ fwd, s4v *__restrict__ bwd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 27 * 64) return;
    const int t = i / 64, l = i % 64;
    s4v f, b;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        f[j] = (short)f2bf(W[(t * 16 + (l & 15)) * 16 + 4 * (l >> 4) + j]);
        b[j] = (short)f2bf(W[((26 - t) * 16 + 4 * (l >> 4) + j) * 16 + (l & 15)]);
    }
    fwd[i] = f;
    bwd[i] = b;
}

// Adam (Kingma & Ba 2015) on the FP32 master parameters; mask zeroes the padding
__global__ void k_nn_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                          const float *__restrict__ mask, int n, float lr, float b1, float b2, float eps, float c1,
                          float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] * mask[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi, vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// out += s in  (the correction into the potential); r = acc - target and its squared sum
__global__ void k_nn_axpy(float *__restrict__ out, const float *__restrict__ in, size_t n, float s) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += s * in[i];
}
// Each of the NN_LOSS_BLOCKS blocks sums its grid-stride share of r^2 in a fixed order into sum[block], and
// k_nn_loss_total adds the block sums in a fixed order into sum[NN_LOSS_BLOCKS]: the loss repeats bit for bit
constexpr int NN_LOSS_BLOCKS = 1024;
__global__ __launch_bounds__(256) void k_nn_residual(const float *__restrict__ acc, const float *__restrict__ tgt,
                                                     float *__restrict__ abar, size_t n, float gs,
                                                     double *__restrict__ sum) {
    __shared__ double red[256];
    double s = 0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)NN_LOSS_BLOCKS * 256) {
        const float r = acc[i] - tgt[i];
        abar[i] = gs * r;
        s += (double)r * r;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) sum[blockIdx.x] = red[0];
}
__global__ __launch_bounds__(256) void k_nn_loss_total(double *sum) {
    __shared__ double red[256];
    double s = 0;
    for (int i = threadIdx.x; i < NN_LOSS_BLOCKS; i += 256) s += sum[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) sum[NN_LOSS_BLOCKS] = red[0];
}

// convolution blocks below which a block takes fewer planes (one to a CU; a training step at 64^3: 1.27 ms with 128,
// 1.15 with 256 and 512)
constexpr int NN_MIN_BLOCKS = 256;
static unsigned ngrid(size_t n, int b) { return (unsigned)((n + b - 1) / b); }

struct NnLaunch {
    static void conv(int in, int epi, int N, const void *hin, const void *fin, double inv_rho, double cval,
                     const void *wsw, const void *bias, const void *res, const void *zmask, void *out_z, void *out_h,
                     void *out_f, double oscale, hipStream_t st) {
        // planes per block: 16, fewer where that leaves the chip's 512 block slots half empty (a 64^3 mesh in
        // segments of 16 runs on 32 blocks)
        const int cols = (N / NN_TX) * (N / NN_TY);
        int tz = 16;
        while (tz > 1 && cols * (N / tz) < NN_MIN_BLOCKS) tz /= 2;
        const dim3 g(cols * (N / tz));
#define NN_C(I, E, R)                                                                                                \
    do {                                                                                                             \
        (void)hipFuncSetAttribute((const void *)k_nn_conv<I, E, R>, hipFuncAttributeMaxDynamicSharedMemorySize,       \
                                  (int)nn_conv_lds<I>());                                                             \
        k_nn_conv<I, E, R><<<g, 256, nn_conv_lds<I>(), st>>>(                                                          \
            N, tz, (const unsigned short *)hin, (const float *)fin, (float)inv_rho, (float)cval, (const s4v *)wsw,     \
            (const float *)bias, (const unsigned short *)res, (const unsigned short *)zmask, (unsigned short *)out_z,  \
            (unsigned short *)out_h, (float *)out_f, (float)oscale);                                                   \
    } while (0)
        if (in == NN_IN_FIELD) NN_C(NN_IN_FIELD, NN_EPI_HIDDEN, NN_RES_NONE);
        else if (in == NN_IN_GRAD) NN_C(NN_IN_GRAD, NN_EPI_BWD, NN_RES_NONE);
        else if (epi == NN_EPI_HIDDEN) NN_C(NN_IN_H, NN_EPI_HIDDEN, NN_RES_INPUT);
        else if (epi == NN_EPI_OUT) NN_C(NN_IN_H, NN_EPI_OUT, NN_RES_NONE);
        else NN_C(NN_IN_H, NN_EPI_BWD, NN_RES_TENSOR);
#undef NN_C
    }
    static void wgrad(int in, int ga, int N, const void *hin, const void *fin, double inv_rho, double cval, const void *gz,
                      const void *gf, double gscale, void *dW, void *db, void *part, hipStream_t st) {
        const int nrows = (N / 64) * N * N, blocks = nrows < NN_WBLOCKS ? nrows : NN_WBLOCKS;
        float *p1 = (float *)part, *p2 = p1 + (size_t)NN_WBLOCKS * NN_WP;
#define NN_W(I, G)                                                                                                     \
    k_nn_wgrad<I, G><<<blocks, 256, 0, st>>>(N, (const unsigned short *)hin, (const float *)fin, (float)inv_rho,        \
                                             (float)cval, (const unsigned short *)gz, (const float *)gf, (float)gscale, p1)
        if (in == NN_IN_FIELD) NN_W(NN_IN_FIELD, 0);
        else if (ga) NN_W(NN_IN_H, 1);
        else NN_W(NN_IN_H, 0);
#undef NN_W
        k_nn_wreduce1<<<dim3(ngrid(NN_WP, 64), NN_WSLICES), 256, 0, st>>>(p1, blocks, p2);
        k_nn_wreduce2<<<ngrid(NN_WP, 256), 256, 0, st>>>(p2, (float *)dW, (float *)db);
    }
    static size_t wgrad_scratch_bytes() { return sizeof(float) * (size_t)NN_WP * (NN_WBLOCKS + NN_WSLICES); }
    static void swizzle(const void *W, void *fwd, void *bwd, void *pfwd, void *pbwd, hipStream_t st) {
        k_nn_swizzle<<<ngrid(27 * 64, 256), 256, 0, st>>>((const float *)W, (s4v *)fwd, (s4v *)bwd);
        k_nn_swizzle_packed<<<1, 256, 0, st>>>((const float *)W, (s4v *)pfwd, (s4v *)pbwd);
    }
    static void adam(void *p, const void *g, void *m, void *v, const void *mask, int n, double lr, double b1, double b2,
                     double eps, double c1, double c2, hipStream_t st) {
        k_nn_adam<<<ngrid(n, 256), 256, 0, st>>>((float *)p, (const float *)g, (float *)m, (float *)v,
                                                 (const float *)mask, n, (float)lr, (float)b1, (float)b2, (float)eps,
                                                 (float)c1, (float)c2);
    }
    static void axpy(void *out, const void *in, size_t n, double s, hipStream_t st) {
        k_nn_axpy<<<ngrid(n, 256), 256, 0, st>>>((float *)out, (const float *)in, n, (float)s);
    }
    static void residual(const void *acc, const void *tgt, void *abar, size_t n, double gs, void *sum, hipStream_t st) {
        k_nn_residual<<<NN_LOSS_BLOCKS, 256, 0, st>>>((const float *)acc, (const float *)tgt, (float *)abar, n, (float)gs,
                                                     (double *)sum);
        k_nn_loss_total<<<1, 256, 0, st>>>((double *)sum);
    }
    static size_t residual_sum_doubles() { return NN_LOSS_BLOCKS + 1; }
};

void nn_ops(NnOps &ops) {
    ops.conv = NnLaunch::conv;
    ops.wgrad = NnLaunch::wgrad;
    ops.wgrad_scratch_bytes = NnLaunch::wgrad_scratch_bytes;
    ops.swizzle = NnLaunch::swizzle;
    ops.adam = NnLaunch::adam;
    ops.axpy = NnLaunch::axpy;
    ops.residual = NnLaunch::residual;
    ops.residual_sum_doubles = NnLaunch::residual_sum_doubles;
}

}  // namespace dj
