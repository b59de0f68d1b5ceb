// What the kernels of the general head sizes share (pqa_general.hip,
// pqa_general_mma.hip).
#pragma once

#include "pqa_device.h"
#include "pqa_internal.h"

namespace pqa {

// One q/k/v operand: column c of token t at p[t * ld + c]; with w_inv the
// value is the batched GEMM's scaled result, p * (w_inv[c] * x_inv[t]) + b[c].
struct GenSrc {
    const float* p;
    int ld;
    const float* w_inv;
    const float* x_inv;
    const uint8_t* b;
    int bt;
};

__device__ __forceinline__ float gen_load(const GenSrc& s, int t, int c) {
    float v = s.p[(size_t)t * s.ld + c];
    if (s.w_inv) {
        v = v * (s.w_inv[c] * s.x_inv[t]);
        if (s.b) v = v + (s.bt == GG_F32 ? ((const float*)s.b)[c] : f16_bits_to_f32(((const uint16_t*)s.b)[c]));
    }
    return v;
}

// Attention of one layer on the MFMA kernels: a decode with ws (n_tok 1; appends the
// new row itself) or, with ws null, a prompt (its rows already appended).
hipError_t launch_gen_mma(pqa_ctx* ctx, int layer, int start, int n_tok, const DecodeWorkspace* ws, const GenSrc& q,
                          const GenSrc& k, const GenSrc& v, float* out);

}  // namespace pqa
