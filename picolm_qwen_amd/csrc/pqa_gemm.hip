// C[m][n] = A_hi B_hi^T + A_hi B_lo^T + A_lo B_hi^T: the three products of
// fp16 operands split into hi and lo parts (pqa_batch.hip), fp32 accumulation
// and output, on v_mfma_f32_32x32x16_f16, each operand loaded once. A row of
// A holds hi at halfs [0, kh) and lo at [kh, 2 kh), likewise B; kh is a
// multiple of 32 (the callers pad with zeros). The batched Q/K/V and output
// projections use it with A = the split inputs (tokens) and B = the split
// weights (rows).
//
// Workgroup tile 64 MI (m) x 64 NJ (n), 4 waves in a 2 x 2 grid, each wave MI x
// NJ accumulators of 32 x 32 (4 x 3: 256 x 192, 192 AGPRs). K runs in 32-wide
// tiles through NS LDS stages: A_hi and A_lo (64-byte rows), B_hi and B_lo,
// filled by direct global->LDS loads (global_load_lds_dwordx4), NS - 1 stages
// ahead. Within a row, 16-byte chunk c sits at position c ^ ((r >> 2) & 3), so
// the 16 rows one pass of an MFMA operand read touches fall on distinct banks.
//
// Per tile, 2 k-steps of 16, each 3 MI NJ MFMAs (3 products; an accumulator is
// reused every MI NJ MFMAs) on 2 (MI + NJ) operand reads: two thirds of the
// load and LDS-read bytes per MFMA of one GEMM over the concatenated
// [hi | hi | lo] . [hi | lo | hi] rows (measured 3-4 % faster than that form
// at 2048 x 6144 x 3 x 2560, where it replaced it). Between the MFMAs of a
// k-step go the operand reads of the next k-step. The workgroup barrier sits
// after k-step 0 (every read of the tile has been issued and has completed by
// then); after it, k-step 1's MFMAs carry the reads of the next tile's k-step
// 0 and, spread evenly, the loads of the tile NS after this one into the stage
// just freed.
//
// Where the tiles of a product do not fill the chip, K is split over several
// workgroups per tile, each with a result of its own ("slice"), summed by the
// reader in slice order.
//
// Tiles are ordered n-major (t = tn * mb + tm, slices outermost) and dealt to
// the 8 XCDs in contiguous runs: workgroup i runs on XCD i mod 8, so the tiles
// that run together on one XCD share their A and B row blocks in that XCD's L2
// (at 2048 x 6144: 8 m-blocks x 4 n-blocks per XCD).
//
// Rows past m (n) load the last row (clamped, never stored).
#include "pqa_device.h"
#include "pqa_internal.h"

namespace pqa {

constexpr int kGemmWaves = 4;
constexpr int kGemmThreads = 64 * kGemmWaves;
constexpr int kG3BK = kGemmBK;
constexpr int kG3RowB = kG3BK * 2;  // 64 bytes per tile row

template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ int g3_swz(int r) { return (r >> 2) & 3; }

struct Gemm3Args {
    const _Float16* a;
    const _Float16* b;
    float* c;
    int m, n, kh, lda, ldb, ldc;
    int mb, nb;
    int slices;           // K ranges; slice i at c + i * slice_stride
    size_t slice_stride;  // floats
};

// waves per SIMD the accumulators leave room for
constexpr int g3_occupancy(int mi, int nj) { return mi * nj > 4 ? 1 : 2; }

template <int MI, int NJ, int NS>
__global__ __launch_bounds__(kGemmThreads, g3_occupancy(MI, NJ)) void gemm_f16x3_nt_kernel(const Gemm3Args g) {
    constexpr int BM = 64 * MI, BN = 64 * NJ;
    constexpr int ASUB = BM * kG3RowB;           // A_hi or A_lo
    constexpr int BSUB = BN * kG3RowB;           // B_hi or B_lo
    constexpr int STAGE = 2 * ASUB + 2 * BSUB;
    constexpr int LOADS = STAGE / 1024 / kGemmWaves;  // 1 KB DMA pieces per wave and tile
    constexpr int FRAGS = 2 * (MI + NJ);         // operand reads per k-step
    constexpr int MFMAS = 3 * MI * NJ;           // MFMAs per k-step
    static_assert(STAGE % (1024 * kGemmWaves) == 0, "whole 1 KB DMA pieces per wave");
    __shared__ __attribute__((aligned(1024))) char lds[NS][STAGE];

    const int T = g.mb * g.nb * g.slices;
    const int xcd = blockIdx.x & 7, jx = blockIdx.x >> 3;
    const int q8 = T >> 3, r8 = T & 7;
    if (jx >= q8 + (xcd < r8 ? 1 : 0)) return;  // whole workgroup, before any barrier
    const int ts = xcd * q8 + min(xcd, r8) + jx;
    const int slice = ts / (g.mb * g.nb), t = ts - slice * (g.mb * g.nb);
    const int tn = t / g.mb, tm = t - tn * g.mb;
    const int m0 = tm * BM, n0 = tn * BN;

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // k tiles [kt0, kt0 + KT) of the slice (every slice has one: slices <= tiles)
    const int KA = g.kh / kG3BK;
    const int kt0 = (int)((long long)KA * slice / g.slices);
    const int KT = (int)((long long)KA * (slice + 1) / g.slices) - kt0;

    // ---- loads: the stage is A_hi, A_lo, B_hi, B_lo in pieces of 16 rows of
    // 64 B (4 MI, 4 MI, 4 NJ, 4 NJ of them); wave w fills pieces w, w + 4, ...;
    // lane l lands at row l / 4, position l % 4 ----
    unsigned goff[LOADS];
    const _Float16* gbase[LOADS];
    unsigned ldst[LOADS];
#pragma unroll
    for (int ii = 0; ii < LOADS; ii++) {
        const int piece = w + kGemmWaves * ii;
        const int part = ii < MI ? 0 : ii < 2 * MI ? 1 : ii < 2 * MI + NJ ? 2 : 3;
        const int first = 4 * (part == 0 ? 0 : part == 1 ? MI : part == 2 ? 2 * MI : 2 * MI + NJ);
        const int row = 16 * (piece - first) + (lane >> 2);
        const int chunk = (lane & 3) ^ g3_swz(row);
        if (part < 2) {
            const int gr = min(m0 + row, g.m - 1) - m0;
            gbase[ii] = g.a + (size_t)m0 * g.lda + (part == 1 ? g.kh : 0) + (size_t)kt0 * kG3BK;
            goff[ii] = (unsigned)(((size_t)gr * g.lda + 8 * chunk) * 2);
        } else {
            const int gr = min(n0 + row, g.n - 1) - n0;
            gbase[ii] = g.b + (size_t)n0 * g.ldb + (part == 3 ? g.kh : 0) + (size_t)kt0 * kG3BK;
            goff[ii] = (unsigned)(((size_t)gr * g.ldb + 8 * chunk) * 2);
        }
        ldst[ii] = (unsigned)(piece * 1024);
    }
    const unsigned lds0 = lds_addr(&lds[0][0]);
    auto load = [&](int kt, int stage, int ii) {
        lds_dma_b128(gbase[ii] + (size_t)kt * kG3BK, goff[ii], lds0 + (unsigned)(stage * STAGE) + ldst[ii]);
    };

    // ---- operand reads: wave (wm, wn) = (w & 1, w >> 1); k-step s reads
    // chunk 2 s + l / 32 of its rows ----
    const int wm = w & 1, wn = w >> 1;
    const int l32 = lane & 31, hk = lane >> 5;
    int offa[MI][2], offb[NJ][2];
#pragma unroll
    for (int s2 = 0; s2 < 2; s2++) {
        const int c = 2 * s2 + hk;
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const int r = wm * 32 * MI + 32 * i + l32;
            offa[i][s2] = r * kG3RowB + 16 * (c ^ g3_swz(r));
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int r = wn * 32 * NJ + 32 * j + l32;
            offb[j][s2] = 2 * ASUB + r * kG3RowB + 16 * (c ^ g3_swz(r));
        }
    }
    // fragments: [slot][0 hi / 1 lo][block]
    half8 fa[2][2][MI], fb[2][2][NJ];
    auto read = [&](const char* st, int s2, int slot, int idx) {
        if (idx < 2 * MI) {
            const int lo = idx >= MI, i = idx - (lo ? MI : 0);
            fa[slot][lo][i] = *(const half8*)(st + offa[i][s2] + lo * ASUB);
        } else {
            const int lo = idx >= 2 * MI + NJ, j = idx - 2 * MI - (lo ? NJ : 0);
            fb[slot][lo][j] = *(const half8*)(st + offb[j][s2] + lo * BSUB);
        }
    };
    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;
    // MFMA q of a k-step: product q / (MI NJ) (hi.hi, hi.lo, lo.hi), block
    // q % (MI NJ)
    auto mfma = [&](int slot, int q) {
        const int p = q / (MI * NJ), idx = q % (MI * NJ);
        const int i = idx / NJ, j = idx % NJ;
        const half8 av = fa[slot][p == 2 ? 1 : 0][i];
        const half8 bv = fb[slot][p == 1 ? 1 : 0][j];
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc[i][j], 0, 0, 0);
    };

    // ---- prologue: tiles 0 .. NS - 1 in flight, tile 0 landed everywhere ----
#pragma unroll
    for (int s = 0; s < NS; s++) {
        if (s < KT) {
#pragma unroll
            for (int ii = 0; ii < LOADS; ii++) load(s, s, ii);
        }
    }
    if (KT >= NS) wait_vm<LOADS*(NS - 1)>();
    else wait_vm<0>();
    __syncthreads();
#pragma unroll
    for (int idx = 0; idx < FRAGS; idx++) read(lds[0], 0, 0, idx);

    // the reads of a k-step among the MFMAs of the one before: one after each of
    // the first FRAGS, or spread when there are more reads than MFMAs
    constexpr int RM = FRAGS < MFMAS ? FRAGS : MFMAS;
    int stage = 0;
    for (int kt = 0; kt < KT; kt++) {
        const char* st = lds[stage];
        const int nstage = stage + 1 == NS ? 0 : stage + 1;
        const bool next = kt + 1 < KT;
        // k-step 0, with the reads of k-step 1 between its MFMAs
#pragma unroll
        for (int q = 0; q < MFMAS; q++) {
            mfma(0, q);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int idx = 0; idx < FRAGS; idx++)
                if (q == idx * RM / FRAGS) read(st, 1, 1, idx);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (next) {
            // this wave's loads of tile kt + 1 (those of up to NS - 2 later tiles
            // stay in flight)
            if (kt + NS - 1 < KT) wait_vm<LOADS*(NS - 2)>();
            else wait_vm<0>();
            __syncthreads();  // everyone's; every read of tile kt has completed
        }
        // k-step 1: the reads of tile kt + 1's k-step 0 (the last tile re-reads
        // its own stage, unused) and the loads of tile kt + NS into this stage
        const char* sn = next ? lds[nstage] : st;
        const bool more = kt + NS < KT;
#pragma unroll
        for (int q = 0; q < MFMAS; q++) {
            mfma(1, q);
            __builtin_amdgcn_sched_barrier(0);
            if (more) {
#pragma unroll
                for (int ii = 0; ii < LOADS; ii++)
                    if (q == (ii * MFMAS) / LOADS) load(kt + NS, stage, ii);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int idx = 0; idx < FRAGS; idx++)
                if (q == idx * RM / FRAGS) read(sn, 0, 0, idx);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage = nstage;
    }

    float* c = g.c + slice * g.slice_stride;
#pragma unroll
    for (int i = 0; i < MI; i++) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int col = n0 + wn * 32 * NJ + 32 * j + l32;
            if (col >= g.n) continue;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int row = m0 + wm * 32 * MI + 32 * i + 8 * (e >> 2) + 4 * hk + (e & 3);
                if (row < g.m) c[(size_t)row * g.ldc + col] = acc[i][j][e];
            }
        }
    }
}

template <int MI, int NJ, int NS>
static hipError_t launch_g3(Gemm3Args g, hipStream_t stream) {
    g.mb = (g.m + 64 * MI - 1) / (64 * MI);
    g.nb = (g.n + 64 * NJ - 1) / (64 * NJ);
    const long long tiles = (long long)g.mb * g.nb * g.slices;
    const long long groups = (tiles + 7) / 8 * 8;
    if (groups > 0x7FFFFFFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_f16x3_nt_kernel<MI, NJ, NS>), dim3((unsigned)groups), dim3(kGemmThreads), 0, stream, g);
    return hipGetLastError();
}

hipError_t launch_gemm_f16x3_nt(const GemmPlan& plan, const _Float16* a, int lda, const _Float16* b, int ldb, float* c,
                                int ldc, size_t slice_stride, int m, int n, int kh, hipStream_t stream) {
    if (m <= 0 || n <= 0 || kh <= 0 || kh % kG3BK != 0 || lda < 2 * kh || ldb < 2 * kh || ldc < n || lda % 8 ||
        ldb % 8 || plan.slices < 1 || plan.slices > kh / kG3BK)
        return hipErrorInvalidValue;
    if ((size_t)256 * lda * 2 >= (1ull << 31) || (size_t)192 * ldb * 2 >= (1ull << 31)) return hipErrorInvalidValue;
    Gemm3Args g;
    g.a = a;
    g.b = b;
    g.c = c;
    g.m = m;
    g.n = n;
    g.kh = kh;
    g.lda = lda;
    g.ldb = ldb;
    g.ldc = ldc;
    g.slices = plan.slices;
    g.slice_stride = slice_stride;
    switch (10 * plan.mi + plan.nj) {
        case 43: return launch_g3<4, 3, 2>(g, stream);
        case 42: return launch_g3<4, 2, 2>(g, stream);
        case 22: return launch_g3<2, 2, 2>(g, stream);
        case 21: return launch_g3<2, 1, 3>(g, stream);
        case 11: return launch_g3<1, 1, 4>(g, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pqa
