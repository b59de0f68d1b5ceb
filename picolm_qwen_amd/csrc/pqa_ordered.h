// The operand image of the reference-order projection (pqa_exact.hip), shared with
// the kernel that splits the inputs (pqa_batch.hip).
#pragma once

#include "pqa_device.h"

namespace pqa {

constexpr int kOrdTile = 32;                      // tokens and rows per workgroup
constexpr int kOrdK = 64;                         // k elements per stage: 8 of each of the 8 sequences
constexpr int kOrdStageF = kOrdTile * kOrdK;      // floats of one operand's stage

__host__ __device__ inline int ord_stages(bool q8, int n) { return q8 ? (n + 255) / 256 * 4 : (n + kOrdK - 1) / kOrdK; }

// element k of a row: its stage, and its float within the stage's image at lane row `r`
__device__ __forceinline__ void ord_place(bool q8, int k, int r, int& st, int& f) {
    int c, j;  // sequence and element of the stage
    if (q8) {
        st = (k >> 8) * 4 + ((k >> 3) & 3);
        c = (k >> 5) & 7;
        j = k & 7;
    } else {
        st = k >> 6;
        c = k & 7;
        j = (k >> 3) & 7;
    }
    const int q = q8 ? c >> 1 : c & 3, b = q8 ? c & 1 : c >> 2;
    f = (2 * q + (j >> 2)) * 256 + (32 * b + r) * 4 + (j & 3);
}

// Image of src [rows][ld] (n columns used; any 4-byte alignment): a workgroup of 256
// threads makes four stages (Q8_0: a round) of one tile. Rows past the last repeat
// it, columns past n are zero. img: 4 kOrdStageF floats of LDS, 16-byte aligned.
template <bool Q8>
__device__ __forceinline__ void ordered_image_tile(const float* __restrict__ src, int ld, int rows, int n,
                                                   float* __restrict__ dst, int group, int tile, float* img) {
    const int tid = threadIdx.x;
    const int nst = ord_stages(Q8, n), st0 = 4 * group, ns = min(4, nst - st0);
    // thread = column: the tile's rows one after the other, 1 KB of a row at a time
    const int k = kOrdK * st0 + tid;
    float v[kOrdTile];
#pragma unroll
    for (int r = 0; r < kOrdTile; r++) {
        const int row = min(tile * kOrdTile + r, rows - 1);
        v[r] = k < n ? src[(size_t)row * ld + k] : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < kOrdTile; r++) {
        int st, f;
        ord_place(Q8, k, r, st, f);
        img[(st - st0) * kOrdStageF + f] = v[r];
    }
    __syncthreads();
    floatx4* o = (floatx4*)(dst + ((size_t)tile * nst + st0) * kOrdStageF);
    for (int i = tid; i < ns * kOrdStageF / 4; i += 256) o[i] = ((const floatx4*)img)[i];
}

}  // namespace pqa
