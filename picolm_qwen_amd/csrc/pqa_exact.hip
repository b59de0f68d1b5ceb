// The K and V projections of a whole prompt in the reference's own summation
// order, so that the cache rows a prompt writes are the reference's bits.
//
// Model::forward_batch projects each prompt token with TensorOps::matmul_bias
// (cpp/model.hpp:503-546 -> cpp/tensor.hpp:134-143), and vec_dot
// (cpp/quant.hpp:342-356) fixes the order of every sum:
//   F32 rows, and F16 / Q4_0 / Q4_K / Q6_K rows after dequantize_row
//   (cpp/quant.hpp:176-281): vec_dot_f32_f32's SSE2 loop (:297-319), two
//   4-lane accumulators over groups of 8, i.e. 8 chains (element i goes to
//   chain i mod 8, in increasing i), every product and sum rounded on its
//   own; then t_l = chain l + chain l+4 and (t0 + t2) + (t1 + t3) (:288-294);
//   Q8_0 rows (:321-340): per 32-element block sum += q * x in order, then
//   sumf += d * sum in block order;
//   then out + bias (vec_add).
// Nothing here reorders a sum. The vector ALU bounds both halves of it, the
// products and the ordered additions: it starts a wave's next instruction every
// 5 cycles but takes one of another wave in between (32 additions: 162 cycles
// with one wave per SIMD, 80 per wave with two), so waves per SIMD count for
// twice. The products come from v_mfma_f32_32x32x1_2b with C = 0, 2 x 32 x 32
// of them round(w * x) in 65-72 cycles; it shares the vector ALU (no overlap was
// measured), but takes its operands as one row and one token per lane where a
// register tile reads 16 values for 64 products. Its bits are v_mul_f32's for
// subnormals, infinities and NaN alike, up to the sign of a zero (2^27 products
// of random and special bit patterns compared; the tests send such inputs and weights
// through the whole projection), which no sum that starts at +0 shows. (A shape with K > 1 would fuse its own additions and round otherwise.)
//
// ordered_kernel: a workgroup of 4 waves owns 32 tokens x 32 rows. The sums of a
// (token, row) pair run as 8 independent sequences over 64-element stages:
//   chain types  sequence c = chain c, the stage's elements 8 j + c (j < 8);
//   Q8_0         sequence c = block c of a round of 8 blocks (4 stages), the
//                stage's 8 elements j of it.
// A wave takes two sequences as the MFMA's two blocks (chains q and q + 4, or
// blocks 2 q and 2 q + 1): 32 sums and 32 products per lane, so that four waves
// fit a SIMD and a tile alone keeps four busy. No operand is shared between the
// waves, so LDS would only add instructions, which are what the kernel is short
// of: both operands come as images in the order the lanes read them (below), two
// 16-byte loads each per stage, requested two stages ahead (one for Q8_0). At the
// end (Q8_0: of each round) the waves' sums meet in LDS and each wave finishes a
// quarter of the tile in the reference's order.
// Short prompts run 16 x 16 tiles with four sequences per wave (below).
// K and V together, 2 x 1024 rows x 2560: 2048 tokens 353 us (a 64 x 64 register
// tile with VALU multiplies, a launch each: 506 us), 75 tokens 26 us (226 us). 2048
// tokens run at 163 cycles per MFMA and its 32 additions, against 143 measured for
// the two alone at four waves per SIMD.
//
// Image of a matrix [rows][n] (n rounded up to whole stages, Q8_0 whole rounds,
// with zeros): per tile of 32 rows and stage, [wave q][half h][lane][4]: lane l is
// row l % 32 and the wave's sequence l / 32, the four floats are elements
// 4 h .. 4 h + 3 of that sequence's 8.
#include <algorithm>

#include "pqa_device.h"
#include "pqa_internal.h"
#include "pqa_ordered.h"

namespace pqa {

typedef float floatx32 __attribute__((ext_vector_type(32)));

constexpr int kOrdThreads = 256;                  // 4 waves

struct OrderedArgs {
    const float* w[2];  // images of the weight rows (Q8_0: the int8 values as floats)
    const float* d[2];  // Q8_0: [rows][n / 32] block scales; else unused
    const uint8_t* b[2];  // bias [rows] (F32 or F16) or null
    int bt[2];
    float* out[2];  // out[t * ldo + r]
    const float* x;  // image of the inputs
    int n_tok, rows, n, ldo;
    int rtiles;  // row tiles per matrix
};

__device__ __forceinline__ float ord_bias(const uint8_t* b, int bt, int r) {
    return bt == GG_F32 ? ((const float*)b)[r] : f16_bits_to_f32(((const uint16_t*)b)[r]);
}

// S: tokens and rows per MFMA tile. 32: the workgroup is one tile, a wave takes
// two sequences (v_mfma_f32_32x32x1_2b). 16: two tiles of 16 tokens x 16 rows, two
// waves each, a wave takes four (v_mfma_f32_16x16x1_4b), for prompts whose 32 x 32
// tiles would leave SIMDs idle or with a lone wave.
template <int S> struct OrdMfma;
template <> struct OrdMfma<32> {
    typedef floatx32 Acc;
    __device__ static Acc mul(float a, float b, Acc z) { return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, z, 0, 0, 0); }
};
template <> struct OrdMfma<16> {
    typedef floatx16 Acc;
    __device__ static Acc mul(float a, float b, Acc z) { return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, z, 0, 0, 0); }
};

template <bool Q8, int S>
__global__ __launch_bounds__(kOrdThreads, 4) void ordered_kernel(const OrderedArgs a) {
#pragma clang fp contract(off)
    constexpr int PD = Q8 ? 2 : 3;  // stages in registers (Q8_0: a third does not fit four waves per SIMD)
    constexpr int NB = 64 / S;                 // sequences per wave = MFMA blocks
    constexpr int NR = S * S / 64;             // results per lane of a whole tile
    constexpr int WT = 8 / NB;                 // waves per tile
    constexpr int NF = NR / WT;                // results a wave finishes
    constexpr int NX = Q8 ? 8 : S == 32 ? 4 : 2;  // exchanged values per result: blocks, or waves
    __shared__ float ex[4 / WT][NX * NR * 64];    // [tile][block or wave][result][lane]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = w % WT, half = w / WT;          // wave of its tile; the tile's rows 16 half .. +15
    const int li = lane % S, blk_l = lane / S;    // token / row and MFMA block of the lane's operands
    const int mat = (int)blockIdx.x >= a.rtiles ? 1 : 0;
    const int rt = (int)blockIdx.x - mat * a.rtiles;
    const int r0 = rt * kOrdTile + half * S, t0 = (int)blockIdx.y * S;
    const int nst = ord_stages(Q8, a.n);
    // the lane's sequence; chain types so that the chains l and l + 4 (and, with
    // four blocks, l + 2 and l + 6) of the final sum meet in one lane
    const int seq = Q8 ? NB * q + blk_l : S == 32 ? q + 4 * blk_l : q + (blk_l & 1) * 4 + (blk_l >> 1) * 2;
    int st_unused, f_x, f_w;  // the lane's 16 bytes of a stage (half 0)
    ord_place(Q8, Q8 ? 32 * seq : seq, t0 % kOrdTile + li, st_unused, f_x);
    ord_place(Q8, Q8 ? 32 * seq : seq, half * S + li, st_unused, f_w);
    const float* xt = a.x + (size_t)(t0 / kOrdTile) * nst * kOrdStageF + f_x;
    const float* wt = a.w[mat] + (size_t)rt * nst * kOrdStageF + f_w;

    floatx4 xv[PD][2], wv[PD][2];
    auto load = [&](int st, int p) __attribute__((always_inline)) {
        const size_t o = (size_t)min(st, nst - 1) * kOrdStageF;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            xv[p][h] = *(const floatx4*)(xt + o + 256 * h);
            wv[p][h] = *(const floatx4*)(wt + o + 256 * h);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    typename OrdMfma<S>::Acc acc;  // sums of this wave's sequences: MFMA result layout, block b at NR b
    typename OrdMfma<S>::Acc zero;
#pragma unroll
    for (int e = 0; e < NB * NR; e++) acc[e] = zero[e] = 0.0f;
    float sumf[Q8 ? NF : 1];  // Q8_0: results NF q ..
#pragma unroll
    for (int e = 0; e < (Q8 ? NF : 1); e++) sumf[e] = 0.0f;

    auto compute = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
            float x = xv[p][u >> 2][u & 3];
            asm volatile("" : "+v"(x));  // keeps this MFMA behind the sums before it: one product buffer
            const typename OrdMfma<S>::Acc pr = OrdMfma<S>::mul(x, wv[p][u >> 2][u & 3], zero);
#pragma unroll
            for (int e = 0; e < NB * NR; e++) acc[e] = acc[e] + pr[e];
            asm volatile("" : "+v"(acc));
        }
        __builtin_amdgcn_sched_barrier(0);
    };

#pragma unroll
    for (int p = 0; p < PD; p++) load(p, p);
    auto step = [&](int st, int p) __attribute__((always_inline)) {
        compute(p);
        load(st + PD, p);
        if constexpr (Q8) {
            if ((st & 3) == 3) {
                // the round's 8 blocks: d * sum of each, then added in block order
                const int blk0 = 2 * (st & ~3), nblk = a.n / 32;
                const float* dr = a.d[mat] + (size_t)min(r0 + li, a.rows - 1) * nblk;
                float d[NB];
#pragma unroll
                for (int b = 0; b < NB; b++) d[b] = dr[min(blk0 + NB * q + b, nblk - 1)];
                __syncthreads();  // the last round has been read
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int e = 0; e < NR; e++) ex[half][((NB * q + b) * NR + e) * 64 + lane] = d[b] * acc[NR * b + e];
                __syncthreads();
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    if (blk0 + b < nblk) {
#pragma unroll
                        for (int e = 0; e < NF; e++) sumf[e] = sumf[e] + ex[half][(b * NR + NF * q + e) * 64 + lane];
                    }
                }
#pragma unroll
                for (int e = 0; e < NB * NR; e++) acc[e] = 0.0f;
            }
        }
    };
    // whole groups of PD stages, then the rest: without an exit inside the loop
    // every wait leaves the later stages' loads in flight
    int st = 0;
    for (; st + PD <= nst; st += PD) {
#pragma unroll
        for (int p = 0; p < PD; p++) step(st + p, p);
    }
#pragma unroll
    for (int p = 0; p < PD - 1; p++)
        if (st + p < nst) step(st + p, p);

    // chain types: t = chain l + chain l+4, then (t0 + t2) + (t1 + t3); with four
    // blocks wave q holds t_q and t_{q+2}, so their sum is its own
    if constexpr (!Q8) {
#pragma unroll
        for (int e = 0; e < NR; e++) {
            float t = acc[e] + acc[NR + e];
            if constexpr (S == 16) t = t + (acc[2 * NR + e] + acc[3 * NR + e]);
            ex[half][(q * NR + e) * 64 + lane] = t;
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < NF; u++) {
        const int e = NF * q + u;  // result register of the MFMA layout
        float res;
        if constexpr (Q8) {
            res = sumf[u];
        } else {
            const float* p = ex[half] + e * 64 + lane;
            if constexpr (S == 32) res = (p[0] + p[2 * NR * 64]) + (p[NR * 64] + p[3 * NR * 64]);
            else res = p[0] + p[NR * 64];
        }
        const int tok = t0 + (S == 32 ? 8 * (e >> 2) + 4 * blk_l + (e & 3) : 4 * blk_l + e);
        const int r = r0 + li;
        if (tok < a.n_tok && r < a.rows) {
            const uint8_t* bias = a.b[mat];
            a.out[mat][(size_t)tok * a.ldo + r] = bias ? res + ord_bias(bias, a.bt[mat], r) : res;
        }
    }
}

template <bool Q8>
__global__ __launch_bounds__(kOrdThreads) void ordered_image_kernel(const float* __restrict__ src, int ld, int rows,
                                                                    int n, float* __restrict__ dst) {
    __shared__ __attribute__((aligned(16))) float img[4 * kOrdStageF];
    ordered_image_tile<Q8>(src, ld, rows, n, dst, (int)blockIdx.x, (int)blockIdx.y, img);
}

// Q8_0 rows -> the int8 values as floats [rows][n] and the block scales
// [rows][n / 32] (fp16 d widened exactly). One thread per 32-element block.
__global__ __launch_bounds__(256) void q8_unpack_kernel(const uint8_t* __restrict__ w, int stride, int rows, int n,
                                                        float* __restrict__ q, float* __restrict__ d) {
    const int nblk = n / 32;
    const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= (long long)rows * nblk) return;
    const int row = (int)(gid / nblk), blk = (int)(gid % nblk);
    const uint8_t* b = w + (size_t)row * stride + 34 * blk;
    d[gid] = f16_bits_to_f32((uint16_t)(b[0] | (b[1] << 8)));
    float* o = q + (size_t)row * n + 32 * blk;
    for (int j = 0; j < 32; j++) o[j] = (float)(int8_t)b[2 + j];
}

// Floats of the image of [rows][n], and of a matrix's prepared copy (Q8_0: the
// image, then the block scales).
size_t ordered_image_floats(bool q8, int rows, int n) {
    return (size_t)((rows + kOrdTile - 1) / kOrdTile) * ord_stages(q8, n) * kOrdStageF;
}
size_t exact_matrix_floats(int type, int rows, int n) {
    const bool q8 = type == GG_Q8_0;
    return ordered_image_floats(q8, rows, n) + (q8 ? (size_t)rows * (n / 32) : 0);
}

hipError_t launch_ordered_image(bool q8, const float* src, int ld, int rows, int n, float* dst, hipStream_t s) {
    if (rows <= 0 || n <= 0 || ld < n) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((ord_stages(q8, n) + 3) / 4), (unsigned)((rows + kOrdTile - 1) / kOrdTile));
    if (q8) hipLaunchKernelGGL(ordered_image_kernel<true>, grid, dim3(kOrdThreads), 0, s, src, ld, rows, n, dst);
    else hipLaunchKernelGGL(ordered_image_kernel<false>, grid, dim3(kOrdThreads), 0, s, src, ld, rows, n, dst);
    return hipGetLastError();
}

hipError_t prepare_exact_matrix(int type, const void* w, int stride, int rows, int n, float* rows_f32, float* dst,
                                hipStream_t s) {
    const bool q8 = type == GG_Q8_0;
    hipError_t e;
    if (q8) {
        const long long items = (long long)rows * (n / 32);
        hipLaunchKernelGGL(q8_unpack_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s,
                           (const uint8_t*)w, stride, rows, n, rows_f32, dst + ordered_image_floats(q8, rows, n));
        e = hipGetLastError();
    } else {
        e = launch_dequant_rows(type, w, stride, rows, n, rows_f32, s);
    }
    return e != hipSuccess ? e : launch_ordered_image(q8, rows_f32, n, rows, n, dst, s);
}

hipError_t launch_ordered_project(const OrderedProj* p, int nmat, int rows, int n, const float* x_image, int n_tok,
                                  int ldo, int cu_count, hipStream_t s) {
    if (rows <= 0 || n_tok <= 0 || n <= 0 || n % 8 || nmat < 1 || nmat > 2) return hipErrorInvalidValue;
    const bool q8 = p[0].type == GG_Q8_0;
    if (q8 && n % 32) return hipErrorInvalidValue;
    OrderedArgs a;
    for (int i = 0; i < 2; i++) {
        const OrderedProj& m = p[i < nmat ? i : 0];
        if ((m.type == GG_Q8_0) != q8) return hipErrorInvalidValue;
        a.w[i] = m.prepared;
        a.d[i] = q8 ? m.prepared + ordered_image_floats(q8, rows, n) : nullptr;
        a.b[i] = (const uint8_t*)m.bias;
        a.bt[i] = m.btype;
        a.out[i] = m.out;
    }
    a.x = x_image;
    a.n_tok = n_tok;
    a.rows = rows;
    a.n = n;
    a.ldo = ldo;
    a.rtiles = (rows + kOrdTile - 1) / kOrdTile;
    // 16 x 16 tiles where 32 x 32 ones leave SIMDs idle or with a lone wave (which
    // adds at half the rate): 75 tokens x 2 x 1024 rows x 2560 34 -> 26 us, 10 tokens
    // 34 -> 19; from the second wave per SIMD on both take the same time
    const long long wgs = (long long)a.rtiles * nmat * ((n_tok + kOrdTile - 1) / kOrdTile);
    const int S = wgs <= cu_count ? 16 : 32;
    const dim3 grid((unsigned)(a.rtiles * nmat), (unsigned)((n_tok + S - 1) / S));
#define PQA_ORD(Q, SS) hipLaunchKernelGGL((ordered_kernel<Q, SS>), grid, dim3(kOrdThreads), 0, s, a)
    if (q8) {
        if (S == 16) PQA_ORD(true, 16);
        else PQA_ORD(true, 32);
    } else {
        if (S == 16) PQA_ORD(false, 16);
        else PQA_ORD(false, 32);
    }
#undef PQA_ORD
    return hipGetLastError();
}

}  // namespace pqa
