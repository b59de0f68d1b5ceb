// Attention at the head sizes 80, 96, 112, 160, 192 and 256 on the matrix cores,
// for decode and prefill alike; the contracts are those of pqa_general.hip, whose
// VALU kernels keep the other sizes (one wave per token and KV head there, bound
// by load latency and by 2 fp32 operations per key, head and dim).
//
// The general path computes in fp32, so every operand that is not an fp16 cache
// value is split into two fp16 parts with 22 significant bits together: q hi + lo
// (each row first scaled by a power of two so that its largest element lies in
// [2^14, 2^15)) against K, and P = 2^11 exp2(score - max) as hi + 2^-11 lo against
// V, the two parts into sums of their own; all sums in fp32. Rows (query heads of
// one KV head, token by token) are packed 16 to a wave: S^T = K Q^T and O^T += V^T P^T
// on v_mfma_f32_16x16x32_f16, in whose layouts a lane's scores are already its
// operand of the second product. A last
// half k-step of 16 dims (80, 112) takes v_mfma_f32_16x16x16_f16.
//
// K and V tiles of 64 keys (32 in a decode and at 256) arrive by direct global->LDS
// loads, 16-byte chunk c of row r at slot c ^ x(r) (x within the largest power of two
// that divides the chunks per row), free of bank conflicts for the K operand reads and
// the transposing V reads alike.
//   prefill  4 waves of 16 rows share each tile (two buffers, one barrier per
//            tile);
//   decode   the waves take a KV head's tiles in turn, each with two tiles of its
//            own in flight behind the small operands; the wave with the last tile
//            norms, rotates and rounds the new row, writes it to the cache and into
//            its LDS tile. The waves' results meet in LDS.
// Either may cut the keys into ranges (workgroups) whose partials gen_merge_kernel
// combines.
//
// Measured per layer against the VALU kernels, inputs changing from call to call:
// decode of 32 / 8 heads of 96 at 9000 44 -> 22 us (13 us for the 27.6 MB of cache,
// merge 4; the rest is the gap between two launches), 8 / 2 heads of 256 at 4 37 -> 16;
// prefill of 700 tokens at head size 96 226 -> 41 us (kernel 207 -> 25; its bound is
// the chain of one tile: operand reads, products, softmax, products). The same inputs
// again, 32 / 8 heads at 9000: 112 34.2 -> 17.7 us, 160 40.5 -> 21.8, 192 44.5 -> 23.6,
// 256 53.4 -> 26.8 (at 32000 91.6 -> 57.2); one query head per KV head, 32 of 96 52.5 ->
// 30.1, of 80 46.7 -> 29.1. The error against 64-bit sums over 75 decode and prefill
// shapes is 0.45 to 1.01 times theirs. Other multiples of 16 up to 256 would fit the
// template: each size is two kernels more, and no model that this library names has one.
//
// Infinities: a split product can turn inf into NaN (inf * 0, inf - inf), and a
// masked key's V row still enters the product with weight 0. A row whose result is
// not finite is therefore computed again by gen_rows, with fp32 q and P, only its
// own keys and no split.
#include <algorithm>

#include "pqa_general.h"

namespace pqa {

constexpr int kGmRows = 16;    // rows per wave
// P = 2^11 exp2(score - max), rescaled when a score passes the maximum by more than
// kGmSlack log2 units: at most 2^15, within fp16. (The factor is exact; 11 added to the
// exponent would round it at 2^-21.) Its low part is scaled by kGmLo to the exponents of
// the high part, and so needs sums of its own: unscaled, both parts end at fp16's 2^-24,
// and of a key at 2^-30 of the largest weight nothing is left (2e-4 of an output that
// many such keys beside an attention sink make up; now 3e-8, as with fp32 weights). 22
// bits hold down to 2^-25 of the largest weight and 16 at 2^-31, where a score's own
// fp32 step is 2^-19. The second sums cost 3-4 % of a prefill at head size 112 or more
// (up to 7 % at 256) and 0.1-0.8 us of a decode.
constexpr float kGmSlack = 4.0f;
constexpr float kGmScale = 2048.0f;
constexpr float kGmLo = 2048.0f;

struct GenMmaArgs {
    GenSrc q, k, v;
    const float* qn;  // [hd] or null
    const float* kn;
    const float* cos_tab;  // [S][hd / 2]
    const float* sin_tab;
    uint16_t* kc;  // the layer's cache
    uint16_t* vc;
    float* out;       // [n_tok][nh * hd] with one range
    float* part_acc;  // [nrange][n_tok * nh][hd]
    float* part_ml;   // [nrange][n_tok * nh][2]
    int start, n_tok, nh, g, n_kv, kv_dim, rope, rows, nblk, nrange;
    int qvec, ovec;  // q / out rows may move as 16-byte vectors
    float qscale;
};

__host__ __device__ constexpr int gm_pow2(int ch) { return ch % 16 == 0 ? 16 : ch % 8 == 0 ? 8 : ch % 4 == 0 ? 4 : ch % 2 == 0 ? 2 : 1; }

template <int HD, int KEYS>
struct GmTile {
    static_assert(HD % 16 == 0 && HD <= 256, "head sizes of the MFMA kernels");
    static constexpr int CH = HD / 8;                 // 16-byte chunks per row
    static constexpr int ROWB = HD * 2;
    static constexpr int BYTES = KEYS * ROWB;
    static constexpr int NI = BYTES / 1024;           // 1 KB loads per operand
    static constexpr int P2 = gm_pow2(CH);
    static constexpr int PER = 16 / P2;               // rows after which the bank of a chunk repeats
    __device__ static int xk(int r) { return (r / PER) & (P2 - 1); }
    __device__ static int xv(int r) { return (2 * (r / PER)) & (P2 - 1); }
};

// waves of a decode workgroup: two tiles each within the LDS
template <int HD>
constexpr int gm_decode_waves() { return HD <= 128 ? 4 : 2; }

// keys per tile: 64 in a prefill (a tile of 32 is one dependent chain of short
// products, 1.1 us at head size 96) unless two of them and the q rows exceed the
// LDS; 32 in a decode, whose waves have two tiles each
template <int HD, bool DECODE>
constexpr int gm_keys() { return DECODE || HD > 192 ? 32 : 64; }

__device__ __forceinline__ float4 gm_load4(const GenSrc& s, int t, int c, int vec) {
    if (s.w_inv || !vec) return float4{gen_load(s, t, c), gen_load(s, t, c + 1), gen_load(s, t, c + 2), gen_load(s, t, c + 3)};
    return *(const float4*)(s.p + (size_t)t * s.ld + c);
}

// Four of a wave's rows again, rows row0 .. row0 + 3 of which those in `bad`: the rows
// at q (fp32, prepared), each over its own keys of tiles first, first + step, ... below
// end, in fp32. Row, m and l of each go to res, m_out and l_out in the scale of the MFMA
// path (res may alias q). Lane = key for the scores (64 keys at a time), lane = pair of
// dims for the sums over V, whose rows come 16 or 32 at a time, ahead of the sums over
// those before; four rows share each K and V load. With an infinite V row in the cache
// (every row of a wave again), per layer, the VALU kernels' time in brackets: 700 tokens
// of 32 / 8 heads of 96 270 us (210), 32 / 32 of 80 267 (340), 8 / 2 of 256 439 (272: 88
// workgroups); decode at 9000 keys 21 (33), 55 (46) and 27 us (46). One row after the
// other, each with K and V loads of its own, took 2460, 2390, 1900, 67, 157 and 38.
template <int HD, int KEYS>
__device__ __forceinline__ void gen_rows(const GenMmaArgs& a, const uint16_t* kbase, const uint16_t* vbase, const float* q,
                                         int row0, unsigned bad, int first, int step, int end, int lane, float* res,
                                         float* m_out, float* l_out) {
    constexpr int QS = HD + 4, NP = (HD / 2 + 63) / 64;  // LDS row stride; dim pairs per lane
    constexpr int TPI = 64 / KEYS;                       // tiles at a time
    constexpr int VB = 32 / NP;                          // V rows at a time
    const size_t stride = (size_t)a.kv_dim;
    int qp[4];
#pragma unroll
    for (int r = 0; r < 4; r++) qp[r] = a.start + min(row0 + r, a.rows - 1) / a.g;
    const int qlast = qp[3];
    float m[4], l[4], acc[4][2 * NP];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        m[r] = -1e30f;
        l[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < 2 * NP; i++) acc[r][i] = 0.0f;
    }
    // the first key of batch b of V rows, of tiles kt, kt + step; past qlast: nothing
    auto batch_key = [&](int kt, int b) __attribute__((always_inline)) {
        const int tile = kt + VB * b / KEYS * step;
        return tile < end ? tile * KEYS + VB * b % KEYS : qlast + 1;
    };
    auto load_v = [&](int kt, int b, uint32_t (&v)[VB][NP]) __attribute__((always_inline)) {
        const int key0 = batch_key(kt, b);
        if (key0 > qlast) return;
#pragma unroll
        for (int u = 0; u < VB; u++) {
            const uint16_t* vr = vbase + (size_t)min(key0 + u, qlast) * stride;
#pragma unroll
            for (int i = 0; i < NP; i++) v[u][i] = 2 * (lane + 64 * i) < HD ? *(const uint32_t*)(vr + 2 * (lane + 64 * i)) : 0u;
        }
    };
    auto add_v = [&](int kt, int b, const uint32_t (&v)[VB][NP], const float (&p)[4]) __attribute__((always_inline)) {
        const int key0 = batch_key(kt, b);
        if (key0 > qlast) return;
        auto add = [&](int u, int r) __attribute__((always_inline)) {
            const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p[r]), VB * b + u));
#pragma unroll
            for (int i = 0; i < NP; i++) {
                acc[r][2 * i] = fmaf(pj, f16_bits_to_f32((uint16_t)(v[u][i] & 0xFFFFu)), acc[r][2 * i]);
                acc[r][2 * i + 1] = fmaf(pj, f16_bits_to_f32((uint16_t)(v[u][i] >> 16)), acc[r][2 * i + 1]);
            }
        };
        if (key0 + VB - 1 <= qp[0]) {  // every key is every row's
#pragma unroll
            for (int u = 0; u < VB; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) add(u, r);
        } else {
#pragma unroll
            for (int u = 0; u < VB; u++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (key0 + u <= qp[r]) add(u, r);
        }
    };
    for (int kt = first; kt < end && kt * KEYS <= qlast; kt += TPI * step) {
        uint32_t v[2][VB][NP];
        load_v(kt, 0, v[0]);
        const int tile = kt + lane / KEYS * step, key = tile * KEYS + lane % KEYS;
        const bool in = tile < end && key <= qlast;
        const u32x4* kr = (const u32x4*)(kbase + (size_t)(in ? key : kt * KEYS) * stride);
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll (NP == 1 ? 8 : 4)
        for (int c = 0; c < HD / 8; c++) {
            const u32x4 u = kr[c];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float* x = q + r * QS + 8 * c;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    s[r] = fmaf(x[2 * e], f16_bits_to_f32((uint16_t)(u[e] & 0xFFFFu)), s[r]);
                    s[r] = fmaf(x[2 * e + 1], f16_bits_to_f32((uint16_t)(u[e] >> 16)), s[r]);
                }
            }
        }
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool valid = in && key <= qp[r];
            const float sv = valid ? s[r] : -__builtin_huge_valf();
            const float mn = fmaxf(m[r], group_max<64>(sv));
            const float corr = fast_exp2(m[r] - mn);
            p[r] = valid ? fast_exp2(sv - mn) * kGmScale : 0.0f;
            l[r] = l[r] * corr + group_sum<64>(p[r]);
            m[r] = mn;
#pragma unroll
            for (int i = 0; i < 2 * NP; i++) acc[r][i] *= corr;
        }
#pragma unroll
        for (int b = 0; b < 64 / VB; b++) {
            if (b + 1 < 64 / VB) load_v(kt, b + 1, v[(b + 1) & 1]);
            add_v(kt, b, v[b & 1], p);
        }
    }
    wave_sync();  // q has been read
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (!((bad >> r) & 1u)) continue;
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (2 * (lane + 64 * i) < HD) *(float2*)(res + r * QS + 2 * (lane + 64 * i)) = float2{acc[r][2 * i], acc[r][2 * i + 1]};
        if (lane == 0) {
            m_out[r] = m[r];
            l_out[r] = l[r];
        }
    }
}

// DECODE: one row group (16 query heads of one KV head at one token), waves on
// different key tiles; else 4 row groups on the same tiles.
template <int HD, bool DECODE>
__global__ __launch_bounds__(DECODE ? 64 * gm_decode_waves<HD>() : 256, !DECODE && HD <= 96 ? 2 : 1) void gen_mma_kernel(const GenMmaArgs a) {
    constexpr int KEYS = gm_keys<HD, DECODE>(), KB = KEYS / 16;
    using T = GmTile<HD, KEYS>;
    constexpr int NW = DECODE ? gm_decode_waves<HD>() : 4;
    constexpr int RW = DECODE ? 1 : 4, KW = NW / RW;  // row groups, key groups
    constexpr int KS = HD / 32, DB = HD / 16;
    constexpr bool HALF = HD % 32 != 0;
    constexpr int QS = HD + 4;                        // LDS row stride of a q row
    constexpr int NBUF = 2;
    constexpr int LPW = (2 * T::NI + RW - 1) / RW;    // loads per wave and tile
    constexpr int LPR = 4 * KW;                       // lanes per q row in its preparation
    constexpr int D4 = HD / 4;
    static_assert(!DECODE || kGmRows * QS * 4 <= 4 * T::BYTES, "a decode wave's result fits its tile buffers");
    __shared__ __attribute__((aligned(1024))) char lds[KW][NBUF][2][T::BYTES];  // [key group][buffer][K, V]
    __shared__ __attribute__((aligned(16))) float sq[RW][kGmRows * QS];  // prepared q; a prefill wave's result later
    __shared__ float s_scale[RW][kGmRows];
    __shared__ float s_ml[NW][2][kGmRows];
    __shared__ __attribute__((aligned(16))) uint16_t s_new[2][DECODE ? HD : 8];
    // decode: cos and sin [HD / 2] each, the norm weights of q and k, k and v
    constexpr int ACOS = 0, ASIN = HD / 2, AQN = HD, AKN = 2 * HD, AK = 3 * HD, AV = 4 * HD;
    __shared__ __attribute__((aligned(16))) float s_aux[DECODE ? 5 * HD : 4];

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = w % RW, wk = w / RW;
    const int c16 = lane & 15, g16 = lane >> 4;
    const int kvh = (int)blockIdx.x % a.n_kv, rest = (int)blockIdx.x / a.n_kv;
    const int blk = a.nblk - 1 - rest / a.nrange, range = rest % a.nrange;  // the longest blocks first
    const int R0 = (blk * RW + wr) * kGmRows;
    const int rlast = a.rows - 1;
    const int last_blk = min(a.rows, (blk + 1) * RW * kGmRows) - 1;
    const int kend = a.start + last_blk / a.g + 1;                    // keys of the block
    const int klim = DECODE ? max(a.start, 1) : kend;                 // rows that are in the cache (row 0 exists)
    const int ktiles = (kend + KEYS - 1) / KEYS;
    const int tile0 = (int)((long long)ktiles * range / a.nrange) + wk;  // this wave's tiles: tile0, tile0 + KW, ...
    const int tile1 = (int)((long long)ktiles * (range + 1) / a.nrange);
    const size_t rowb = (size_t)a.kv_dim * 2;
    const char* kbase = (const char*)(a.kc + (size_t)kvh * HD);
    const char* vbase = (const char*)(a.vc + (size_t)kvh * HD);

    // ---- K/V loads: piece pp of a tile is 1 KB load pp % NI of operand pp / NI;
    // the row waves share the pieces (the last one may be loaded twice) ----
    unsigned goff[LPW];
#pragma unroll
    for (int i = 0; i < LPW; i++) {
        const int pp = min(wr + RW * i, 2 * T::NI - 1);
        const int L = 64 * (pp % T::NI) + lane, r = L / T::CH;
        goff[i] = (unsigned)(r * rowb) + 16u * (unsigned)((L % T::CH) ^ (pp < T::NI ? T::xk(r) : T::xv(r)));
    }
    auto issue = [&](int kt, int buf) __attribute__((always_inline)) {
        if (kt >= tile1) return;
        const int key0 = kt * KEYS;
        const bool full = key0 + KEYS <= klim;
        const int k0 = min(key0, klim - 1);  // a tile of the new row alone reads the row before it
#pragma unroll
        for (int i = 0; i < LPW; i++) {
            const int pp = min(wr + RW * i, 2 * T::NI - 1);
            unsigned off = goff[i];
            if (!full) {  // rows past the last one repeat it (masked, or overwritten by the new row)
                const int L = 64 * (pp % T::NI) + lane, r = L / T::CH;
                off = (unsigned)(min(r, klim - 1 - k0) * rowb) +
                      16u * (unsigned)((L % T::CH) ^ (pp < T::NI ? T::xk(r) : T::xv(r)));
            }
            const char* src = (pp < T::NI ? kbase : vbase) + (size_t)k0 * rowb;
            lds_dma_b128(src, off, lds_addr(&lds[wk][buf][pp < T::NI ? 0 : 1][(pp % T::NI) * 1024]));
        }
    };
    // ---- decode: q, k, v, the RoPE row and the norm weights go to LDS by direct
    // loads too, ahead of the K/V tiles, so that the wave can wait for them alone
    // (a wait the compiler places would cover the tiles in flight) ----
    float* qreg = sq[wr];
    const bool owner = DECODE && range == a.nrange - 1 && tile0 < tile1 && (tile1 - 1 - tile0) % KW == 0;
    if constexpr (DECODE) {
        auto fetch = [&](const float* src, int n, float* dst) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < (HD + 63) / 64; i++)
                if (64 * i + lane < n) lds_dma_b32(src, 256u * i + 4u * lane, lds_addr(dst) + 256u * i);
        };
        const int nrow = min(kGmRows, rlast + 1 - R0);
        const float* q0 = a.q.p + (size_t)(kvh * a.g + R0) * HD;
        for (int r = wk; r < nrow; r += KW) fetch(q0 + (size_t)r * HD, HD, qreg + r * QS);
        for (int r = nrow + wk; r < kGmRows; r += KW)
            for (int e = lane; e < HD; e += 64) qreg[r * QS + e] = 0.0f;
        const size_t rp = (size_t)a.start * (HD / 2);
        if (wk == 0) {
            fetch(a.cos_tab + rp, HD / 2, s_aux + ACOS);
            fetch(a.sin_tab + rp, HD / 2, s_aux + ASIN);
        }
        if (wk == KW - 1 && a.qn) fetch(a.qn, HD, s_aux + AQN);
        if (owner) {
            if (a.kn) fetch(a.kn, HD, s_aux + AKN);
            fetch(a.k.p + (size_t)kvh * HD, HD, s_aux + AK);
            fetch(a.v.p + (size_t)kvh * HD, HD, s_aux + AV);
        }
    }
    issue(tile0, 0);
    if constexpr (DECODE) issue(tile0 + KW, 1);

    // ---- q: normed, rotated, scaled, fp32 in LDS; its largest element's exponent ----
    // Rows wk, wk + KW, ... of a decode's 16, the wave's own 16 in a prefill; LPR
    // lanes each.
    if constexpr (DECODE) {
        const int mine = tile0 >= tile1 ? 0 : tile0 + KW >= tile1 ? 1 : 2;
        if (mine == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LPW < 63 ? 2 * LPW : 63) : "memory");
        else if (mine == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    {
        const int pr = (lane / LPR) * KW + wk, sub = lane % LPR;
        const int Rc = min(R0 + pr, rlast), tok = Rc / a.g;
        const int col0 = (kvh * a.g + Rc - tok * a.g) * HD;
        const bool live = R0 + pr <= rlast;
        float* row = qreg + pr * QS;
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < (D4 + LPR - 1) / LPR; i++) {
            const int f = sub + LPR * i;
            if (f < D4) {
                float4 x;
                if constexpr (DECODE) {
                    x = *(const float4*)(row + 4 * f);
                } else {
                    x = gm_load4(a.q, tok, col0 + 4 * f, a.qvec);
                    if (!live) x = float4{0.0f, 0.0f, 0.0f, 0.0f};
                    *(float4*)(row + 4 * f) = x;
                }
                ss = fmaf(x.x, x.x, fmaf(x.y, x.y, fmaf(x.z, x.z, fmaf(x.w, x.w, ss))));
            }
        }
        wave_sync();
        float sc = a.qscale;
        if (a.qn) sc = sc / sqrtf(group_sum<LPR>(ss) / (float)HD + 1e-6f);
        const size_t half = HD / 2;
        const float* cr = DECODE ? s_aux + ACOS : a.cos_tab + (size_t)(a.start + tok) * half;
        const float* sr = DECODE ? s_aux + ASIN : a.sin_tab + (size_t)(a.start + tok) * half;
        const float* qn = DECODE ? s_aux + AQN : a.qn;
        float mx = 0.0f;
#pragma unroll
        for (int i = 0; i < (HD / 2 + LPR - 1) / LPR; i++) {
            const int p = sub + LPR * i;
            if (p < HD / 2) {
                int e0, e1;
                rope_pair(a.rope, p, HD, e0, e1);
                float x0 = row[e0] * sc, x1 = row[e1] * sc;
                if (a.qn) {
                    x0 *= qn[e0];
                    x1 *= qn[e1];
                }
                rope_rotate_fma(x0, x1, cr[p], sr[p]);
                row[e0] = x0;
                row[e1] = x1;
                mx = fmaxf(mx, fmaxf(fabsf(x0), fabsf(x1)));
            }
        }
        mx = group_max<LPR>(mx);
        // 2^s with the largest element in [2^14, 2^15); 1 for zero and non-finite rows
        const int be = (int)((__float_as_uint(mx) >> 23) & 0xFFu);
        const int s = be == 0 || be == 255 ? 0 : min(141 - be, 126);
        if (sub == 0) s_scale[wr][pr] = __uint_as_float((unsigned)(127 + s) << 23);
    }
    // ---- decode: the new row (the wave whose tiles end the range that ends the
    // keys; each block of more than 16 heads writes the same bytes) ----
    if constexpr (DECODE) {
        if (owner) {
            float* s_k = s_aux + AK;
            if (a.kn) {
                const float sc = rms_scale_ref_quad<HD>(s_k, lane & 3);
                wave_sync();
                for (int e = lane; e < HD; e += 64) s_k[e] = rms_apply(s_k[e], sc, s_aux[AKN + e]);
                wave_sync();
            }
            const float* cr = s_aux + ACOS;
            const float* sr = s_aux + ASIN;
            const size_t off = (size_t)a.start * a.kv_dim + (size_t)kvh * HD;
            for (int p = lane; p < HD / 2; p += 64) {
                int e0, e1;
                rope_pair(a.rope, p, HD, e0, e1);
                float x0 = s_k[e0], x1 = s_k[e1];
                rope_rotate(x0, x1, cr[p], sr[p]);
                const uint16_t h0 = f32_to_f16_ref(x0), h1 = f32_to_f16_ref(x1);
                s_new[0][e0] = h0;
                s_new[0][e1] = h1;
                a.kc[off + e0] = h0;
                a.kc[off + e1] = h1;
            }
            for (int e = lane; e < HD; e += 64) {
                const uint16_t h = f32_to_f16_ref(s_aux[AV + e]);
                s_new[1][e] = h;
                a.vc[off + e] = h;
            }
        }
    }
    if constexpr (KW > 1) __syncthreads();  // every wave's q rows
    else wave_sync();

    // q as the B operand: row c16, dims 32 ks + 8 g16 .. +7 (half step: 4 g16 .. +3)
    half8 qh[KS], ql[KS];
    half4 qh4 = {}, ql4 = {};
    const float scl = s_scale[wr][c16];
    const float sinv = __uint_as_float((254u << 23) - __float_as_uint(scl));  // 1 / scl
    {
        const float* row = qreg + c16 * QS;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x = row[32 * ks + 8 * g16 + e] * scl;
                qh[ks][e] = (_Float16)x;
                ql[ks][e] = (_Float16)(x - (float)qh[ks][e]);
            }
        if constexpr (HALF) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = row[32 * KS + 4 * g16 + e] * scl;
                qh4[e] = (_Float16)x;
                ql4[e] = (_Float16)(x - (float)qh4[e]);
            }
        }
    }

    // operand addresses in a tile: K row c16 (+ 16), V rows 4 g16 + c16 / 4 (+ 16);
    // the swizzle of row r + 16 is that of row r
    int koff[KS], voff[DB];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) koff[ks] = c16 * T::ROWB + 16 * ((4 * ks + g16) ^ T::xk(c16));
    const int koffh = c16 * T::ROWB + 16 * ((4 * KS + (g16 >> 1)) ^ T::xk(c16)) + 8 * (g16 & 1);
    const int vr0 = 4 * g16 + (c16 >> 2);
#pragma unroll
    for (int db = 0; db < DB; db++)
        voff[db] = vr0 * T::ROWB + 16 * ((2 * db + ((c16 & 3) >> 1)) ^ T::xv(vr0)) + 8 * (c16 & 1);

    const int qpos = a.start + min(R0 + c16, rlast) / a.g;             // of the lane's row
    const int qmin = a.start + min(R0, rlast) / a.g;                   // of the wave's first row
    const int qmax = R0 <= rlast ? a.start + min(R0 + kGmRows - 1, rlast) / a.g : -1;
    float m_run = -1e30f, l_run = 0.0f;
    floatx4 o[DB], ol[DB];  // O^T: dims 16 db + 4 g16 .. +3 of row c16; from the high and the low parts of P
#pragma unroll
    for (int db = 0; db < DB; db++) o[db] = ol[db] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    auto compute = [&](int kt, int buf) __attribute__((always_inline)) {
        const int key0 = kt * KEYS;
        char* kl = lds[wk][buf][0];
        char* vl = lds[wk][buf][1];
        if constexpr (DECODE) {
            if (owner && key0 + KEYS > a.start) {  // the last tile: the new row into its place
                const int r = a.start - key0;
                if (lane < T::CH) {
                    *(u32x4*)(kl + r * T::ROWB + 16 * (lane ^ T::xk(r))) = ((const u32x4*)s_new[0])[lane];
                    *(u32x4*)(vl + r * T::ROWB + 16 * (lane ^ T::xv(r))) = ((const u32x4*)s_new[1])[lane];
                }
                wave_sync();
            }
        }
        floatx4 s[KB];
#pragma unroll
        for (int kb = 0; kb < KB; kb++) s[kb] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            half8 kf[KB];
#pragma unroll
            for (int kb = 0; kb < KB; kb++) kf[kb] = *(const half8*)(kl + koff[ks] + kb * 16 * T::ROWB);
#pragma unroll
            for (int kb = 0; kb < KB; kb++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[kb], qh[ks], s[kb], 0, 0, 0);
#pragma unroll
            for (int kb = 0; kb < KB; kb++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[kb], ql[ks], s[kb], 0, 0, 0);
        }
        if constexpr (HALF) {
            half4 kf[KB];
#pragma unroll
            for (int kb = 0; kb < KB; kb++) kf[kb] = *(const half4*)(kl + koffh + kb * 16 * T::ROWB);
#pragma unroll
            for (int kb = 0; kb < KB; kb++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x16f16(kf[kb], qh4, s[kb], 0, 0, 0);
#pragma unroll
            for (int kb = 0; kb < KB; kb++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x16f16(kf[kb], ql4, s[kb], 0, 0, 0);
        }
        // keys key0 + 16 kb + 4 g16 + e of row c16
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int e = 0; e < 4; e++) s[kb][e] *= sinv;
        if (key0 + KEYS - 1 > qmin) {
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (key0 + 16 * kb + 4 * g16 + e > qpos) s[kb][e] = -__builtin_huge_valf();
        }
        float mx = s[0][0];
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int e = 0; e < 4; e++) mx = fmaxf(mx, s[kb][e]);
        mx = max_x32(max_x16(mx));
        if (__any(mx > m_run + kGmSlack)) {
            const float m_new = fmaxf(m_run, mx);
            const float corr = fast_exp2(m_run - m_new);
            m_run = m_new;
            l_run *= corr;
            if (kt > tile0) {  // the first tile has nothing to rescale
#pragma unroll
                for (int db = 0; db < DB; db++) {
                    o[db] *= corr;
                    ol[db] *= corr;
                }
            }
        }
        // k-step h: keys 4 g16 .. +3 of key block 2 h, then of block 2 h + 1
        half8 ph[KB / 2], pl[KB / 2];
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float p = fast_exp2(s[kb][e] - m_run) * kGmScale;
                l_run += p;
                const _Float16 hi = (_Float16)p;
                ph[kb >> 1][4 * (kb & 1) + e] = hi;
                pl[kb >> 1][4 * (kb & 1) + e] = (_Float16)((p - (float)hi) * kGmLo);
            }
#pragma unroll
        for (int h = 0; h < KB / 2; h++)
#pragma unroll
            for (int db = 0; db < DB; db++) {
                half4 part[2];
#pragma unroll
                for (int t = 0; t < 2; t++)
                    part[t] = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) short4v*)(vl + voff[db] + (32 * h + 16 * t) * T::ROWB)));
                const half8 vf = {part[0][0], part[0][1], part[0][2], part[0][3],
                                  part[1][0], part[1][1], part[1][2], part[1][3]};
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph[h], o[db], 0, 0, 0);
                ol[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl[h], ol[db], 0, 0, 0);
            }
    };

    int buf = 0;
    for (int kt = tile0; kt < tile1; kt += KW) {
        if constexpr (RW > 1) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads of the tile
            __syncthreads();                                   // everyone's; the other buffer is free
            issue(kt + 1, buf ^ 1);
            if (kt * KEYS <= qmax) compute(kt, buf);
        } else {
            if (kt + KW < tile1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory");  // the next tile's stay in flight
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            compute(kt, buf);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the buffer has been read
            issue(kt + 2 * KW, buf);
        }
        buf ^= 1;
    }

    // ---- the wave's result to LDS: rows of HD floats, the maximum and the sum ----
    // (a prefill wave's over its own q rows, a decode wave's over its tiles)
    float* res = DECODE ? (float*)&lds[wk][0][0][0] : qreg;
    const float l = sum_x32(sum_x16(l_run));
    float chk = l * 0.0f;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[db][e] = fmaf(ol[db][e], 1.0f / kGmLo, o[db][e]);
            chk = fmaf(o[db][e], 0.0f, chk);
        }
    const unsigned long long badl = __ballot(!(chk == 0.0f) && R0 + c16 <= rlast);
    const unsigned bad = (unsigned)((badl | badl >> 16 | badl >> 32 | badl >> 48) & 0xFFFFu);
    if (!((bad >> c16) & 1u)) {
#pragma unroll
        for (int db = 0; db < DB; db++) *(floatx4*)(res + c16 * QS + 16 * db + 4 * g16) = o[db];
        if (g16 == 0) {
            s_ml[w][0][c16] = m_run;
            s_ml[w][1][c16] = l;
        }
    }
    wave_sync();
    if (bad) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the new row's stores
#pragma unroll 1
        for (int r = 0; r < kGmRows; r += 4) {
            if (!((bad >> r) & 15u)) continue;
            gen_rows<HD, KEYS>(a, (const uint16_t*)kbase, (const uint16_t*)vbase, qreg + r * QS, R0 + r, bad >> r, tile0, KW,
                               tile1, lane, res + r * QS, &s_ml[w][0][r], &s_ml[w][1][r]);
        }
        wave_sync();
    }
    if constexpr (KW > 1) __syncthreads();
    const bool partial = a.nrange > 1;
    const int nrow = min(kGmRows, rlast + 1 - R0);
    for (int it = KW > 1 ? tid : lane; it < nrow * D4; it += KW > 1 ? 64 * NW : 64) {
        const int r = it / D4, d4 = it - r * D4;
        float M = -1e30f, L = 0.0f;
        floatx4 A = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (KW == 1) {
            M = s_ml[w][0][r];
            L = s_ml[w][1][r];
            A = *(const floatx4*)(res + r * QS + 4 * d4);
        } else {
#pragma unroll
            for (int k = 0; k < KW; k++) M = fmaxf(M, s_ml[k][0][r]);
#pragma unroll
            for (int k = 0; k < KW; k++) {
                const float e = fast_exp2(s_ml[k][0][r] - M);
                L = fmaf(e, s_ml[k][1][r], L);
                A += e * *(const floatx4*)((const float*)&lds[k][0][0][0] + r * QS + 4 * d4);
            }
        }
        const int R = R0 + r;
        const size_t orow = (size_t)(R / a.g) * a.nh + kvh * a.g + R % a.g;
        if (partial) {
            const size_t slot = (size_t)range * a.n_tok * a.nh + orow;
            *(floatx4*)(a.part_acc + slot * HD + 4 * d4) = A;
            if (d4 == 0) *(float2*)(a.part_ml + 2 * slot) = float2{M, L};
        } else {
            A *= 1.0f / L;
            float* d = a.out + orow * HD + 4 * d4;
            if (a.ovec) {
                *(floatx4*)d = A;
            } else {
                *(float2*)d = float2{A[0], A[1]};
                *(float2*)(d + 2) = float2{A[2], A[3]};
            }
        }
    }
}

// out = sum_s 2^(m_s - M) acc_s / sum_s 2^(m_s - M) l_s over the ranges of one
// output row: sg groups of hd / 4 threads per row, group j on ranges j, j + sg,
// ..., summed through LDS. (An empty range has m = -1e30, weight 0.)
constexpr int kGmMaxRanges = 256;
__global__ __launch_bounds__(256) void gen_merge_kernel(const float* __restrict__ part_acc,
                                                        const float* __restrict__ part_ml, float* __restrict__ out,
                                                        int rows, int nrange, int hd, int sg, int ovec) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int d4n = hd >> 2, tpr = sg * d4n, rpw = 256 / tpr;
    const int tid = threadIdx.x, rl = tid / tpr, j = (tid - rl * tpr) / d4n, d4 = tid - rl * tpr - j * d4n;
    const int row = (int)blockIdx.x * rpw + rl;
    const bool live = rl < rpw && row < rows;
    float* s_m = sm;                                  // [rpw][nrange] maxima, then [rpw][nrange] sums
    float* s_l = sm + rpw * nrange;
    floatx4* s_a = (floatx4*)(sm + ((2 * rpw * nrange + 3) & ~3));  // [rpw][sg][d4n]
    if (live)
        for (int i = tid - rl * tpr; i < nrange; i += tpr) {
            const float2 ml = *(const float2*)(part_ml + 2 * ((size_t)i * rows + row));
            s_m[rl * nrange + i] = ml.x;
            s_l[rl * nrange + i] = ml.y;
        }
    __syncthreads();
    float M = -1e30f, L = 0.0f;
    floatx4 A = {0.0f, 0.0f, 0.0f, 0.0f};
    if (live) {
        for (int i = 0; i < nrange; i++) M = fmaxf(M, s_m[rl * nrange + i]);
        for (int i = 0; i < nrange; i++) L = fmaf(fast_exp2(s_m[rl * nrange + i] - M), s_l[rl * nrange + i], L);
#pragma unroll 8
        for (int i = j; i < nrange; i += sg) {
            const floatx4 v = *(const floatx4*)(part_acc + ((size_t)i * rows + row) * hd + 4 * d4);
            A += fast_exp2(s_m[rl * nrange + i] - M) * v;
        }
        s_a[tid] = A;
    }
    __syncthreads();
    if (live && j == 0) {
        for (int k = 1; k < sg; k++) A += s_a[tid + k * d4n];
        A *= 1.0f / L;
        float* o = out + (size_t)row * hd + 4 * d4;
        if (ovec) {
            *(floatx4*)o = A;
        } else {
            *(float2*)o = float2{A[0], A[1]};
            *(float2*)(o + 2) = float2{A[2], A[3]};
        }
    }
}

template <int HD>
static void launch_gm(const GenMmaArgs& a, bool decode, unsigned grid, hipStream_t s) {
    if (decode) hipLaunchKernelGGL((gen_mma_kernel<HD, true>), dim3(grid), dim3(64 * gm_decode_waves<HD>()), 0, s, a);
    else hipLaunchKernelGGL((gen_mma_kernel<HD, false>), dim3(grid), dim3(256), 0, s, a);
}

hipError_t launch_gen_mma(pqa_ctx* ctx, int layer, int start, int n_tok, const DecodeWorkspace* ws, const GenSrc& q,
                          const GenSrc& k, const GenSrc& v, float* out) {
    const int hd = ctx->head_dim;
    const bool decode = ws != nullptr;
    const size_t part_rows = decode ? (size_t)ws->max_splits * ctx->n_heads : ctx->pf_rows;
    const bool norm = ctx->has_qk_norm[layer] != 0;
    GenMmaArgs a;
    a.q = q;
    a.k = k;
    a.v = v;
    a.qn = norm ? ctx->qk_norm + (size_t)layer * 2 * hd : nullptr;
    a.kn = norm ? ctx->qk_norm + (size_t)layer * 2 * hd + hd : nullptr;
    a.cos_tab = ctx->rope_cos;
    a.sin_tab = ctx->rope_sin;
    a.kc = ctx->key_cache + (size_t)layer * ctx->layer_elems;
    a.vc = ctx->val_cache + (size_t)layer * ctx->layer_elems;
    a.out = out;
    a.start = start;
    a.n_tok = n_tok;
    a.nh = ctx->n_heads;
    a.g = ctx->kv_mul;
    a.n_kv = ctx->n_kv_heads;
    a.kv_dim = (int)ctx->kv_dim;
    a.rope = ctx->rope_style;
    a.rows = n_tok * ctx->kv_mul;
    const int rpb = decode ? kGmRows : 4 * kGmRows;
    a.nblk = (a.rows + rpb - 1) / rpb;
    a.qvec = ((uintptr_t)q.p & 15) == 0 && q.ld % 4 == 0;
    a.ovec = ((uintptr_t)out & 15) == 0;
    a.qscale = 1.4426950408889634f / sqrtf((float)hd);
    // Ranges. Decode: about one workgroup per CU, each wave at least one 32-key tile; up
    // to four tiles per wave the second launch costs more than it gives (32 / 8 heads of
    // 96: 384 keys 8.9 us in one launch and 10.0 in two, 512 9.9 and 10.1, 640 10.9 and
    // 10.2; with the two waves of the sizes from 160 on the two meet at two tiles, 8 / 2
    // heads of 256: 192 keys 15.7 and 14.8, 256 keys 17.6 and 14.9). Prefill: as long as
    // the blocks leave CUs idle and a range keeps 512 keys, for each prepares its q rows
    // again and is merged (32 / 8 heads of 96, ranges of 256, 512 and 1024 keys: 512 tokens
    // at 0 29.9, 21.4 and 21.4 us, 64 tokens at 3000 28.2, 26.2 and 32.2; with two KV heads
    // 256 is the better, 64 tokens at 2000 of 8 / 2 heads of 256 34.8, 45.3 and 67.0).
    const int tiles = (start + n_tok + 31) / 32;
    const long long wgs = (long long)a.nblk * a.n_kv;
    const int kw = decode ? (hd <= 128 ? 4 : 2) : 1;
    long long ranges = std::max<long long>(1, (decode ? ctx->cu_count : 2LL * ctx->cu_count) / wgs);
    ranges = std::min<long long>(ranges, decode ? (tiles <= 4 * kw ? 1 : (tiles + kw - 1) / kw) : std::max(1, tiles / 16));
    ranges = std::min<long long>(ranges, kGmMaxRanges);
    const size_t orows = (size_t)n_tok * a.nh;
    ranges = std::max<long long>(1, std::min<long long>(ranges, (long long)(part_rows / orows)));
    float *part_acc = nullptr, *part_ml = nullptr;
    if (ranges > 1) {
        part_acc = decode ? ws->part_acc : range_partials(ctx, layer);
        if (part_acc) part_ml = decode ? ws->part_ml : part_acc + part_rows * hd;
        else ranges = 1;
    }
    a.part_acc = part_acc;
    a.part_ml = part_ml;
    a.nrange = (int)ranges;
    const long long grid = wgs * ranges;
    if (grid > 0x7FFFFFFF || orows > 0x7FFFFFFF) return hipErrorInvalidValue;
    switch (hd) {
#define PQA_GM(H) case H: launch_gm<H>(a, decode, (unsigned)grid, ctx->stream); break;
        PQA_GM(80) PQA_GM(96) PQA_GM(112) PQA_GM(160) PQA_GM(192) PQA_GM(256)
#undef PQA_GM
        default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ranges == 1) return e;
    const int sg = std::min<int>((int)ranges, 256 / (hd / 4)), rpw = 256 / (sg * (hd / 4));
    const size_t lds = ((2 * (size_t)rpw * ranges + 3) & ~(size_t)3) * 4 + 256 * 16;
    hipLaunchKernelGGL(gen_merge_kernel, dim3((unsigned)((orows + rpw - 1) / rpw)), dim3(256), lds, ctx->stream,
                       (const float*)part_acc, (const float*)part_ml, out, (int)orows, (int)ranges, hd, sg, a.ovec);
    return hipGetLastError();
}

}  // namespace pqa
