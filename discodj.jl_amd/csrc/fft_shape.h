// Workgroup shapes of the transforms' passes and what their kernels share.
#pragma once

#include <hip/hip_runtime.h>

#include "fft_passes.h"

namespace dj {

template <typename T, int N> struct FftShape {
    // lines per workgroup: about 64 KiB of LDS for the y/z tiles, at most 16, dividing N
    static constexpr int target = 65536 / (N * (int)sizeof(cx<T>));
    static constexpr int B = (N % 16 == 0 && target >= 16) ? 16
                           : (N % 8 == 0 && target >= 8) ? 8
                           : (N % 4 == 0 && target >= 4) ? 4
                           : (N % 2 == 0 && target >= 2) ? 2 : 1;
    // x passes (half-length packed lines, about 32 KiB of LDS) run 256 threads; the y/z passes run
    // 512 once a radix-16 pass has at least that many butterflies, so that the two workgroups their
    // LDS tile allows per CU still hold 16 waves
    static constexpr int NT = 256;
    static constexpr int NTY = (B * N / 16 >= 512) ? 512 : 256;
    using P = Passes<T, N, B, NT>;
    using PY = Passes<T, N, B, NTY>;
    // the N-entry twiddle table moves into LDS when two workgroups of the y/z tile plus table
    // still fit a CU (160 KiB); otherwise the passes read it through the caches
    static constexpr bool TWL = (PY::EF::LDS_ELEMS + N) * sizeof(cx<T>) <= 80 * 1024;
    // the c2r x pass at 1024^3 (FP32): 16 lines per workgroup and 512 threads, so that its transposed
    // loads read whole 128-byte lines of a block's own (1.99 against 2.12 ms with 8 lines and 256)
    static constexpr int BXI = (sizeof(T) == 4 && N == 1024) ? 16 : B;
    static constexpr int NTXI = BXI == B ? NT : 512;
    using PXI = Passes<T, N, BXI, NTXI>;
};

// The hardware hands workgroup b to XCD b % 8.  Logical block (b % 8) (nb / 8) + b / 8 puts runs of
// consecutive logical blocks on one XCD, where they run close in time: neighbouring line groups
// whose transposed loads and stores share 128-byte lines then meet in that XCD's L2 instead of
// fetching each line twice from HBM.
__device__ __forceinline__ int xcd_block(int b, int nb) { return (nb & 7) ? b : (b & 7) * (nb >> 3) + (b >> 3); }

// the twiddle table for a workgroup: a copy in LDS, or the global table
template <typename T, int N, bool TWL>
__device__ __forceinline__ const cx<T> *stage_twiddles(const cx<T> *__restrict__ tw, cx<T> *twl, int tid, int nt) {
    if constexpr (TWL) {
        for (int i = tid; i < N; i += nt) twl[i] = tw[i];
        return twl;  // the caller's barrier after the tile load covers this copy
    } else {
        return tw;
    }
}

}  // namespace dj
