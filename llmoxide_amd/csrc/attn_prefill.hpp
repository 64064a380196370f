// What the prefill kernels share: their arguments, the visible range of a
// query, and small register and wait helpers.
#pragma once

#include "common.hpp"

namespace lmx {

struct PrefillArgs {
    const void* q;
    const f16* k;
    const f16* v;
    const f16* k_cur;
    const f16* v_cur;
    float* out;
    const float* gate;  // NULL, or the output gate: out *= sigmoid(gate[row * gate_stride + d])
    int q_stride, gate_stride;
    int H, Hkv, G, kv_dim;
    int base_pos, window, n_tokens, bidi;
    int n_qtiles;
    int gp;  // query heads per workgroup (a power of two dividing G)
    uint32_t w_magic;  // p % window == ring_slot(p, window, w_magic, w_shift)
    int w_shift;
    float c;  // scale * log2(e)
    // Key-range split (not the ping-pong and key-halves kernels): n_split > 1 writes each
    // split's unnormalized o and its (m, l) to part_o / part_ml for
    // prefill_merge_kernel.
    int n_split;
    float* part_o;   // [n_split][t][H][hd]
    float* part_ml;  // [n_split][t][H][2]
};

// How attn_prefill_wide_kernel runs a call: query heads and tokens of a
// workgroup, and whether in its form for few rows.
struct WidePlan {
    int gp, tokens;
    bool few;
};

// Keys the call's last query sees at most (attn_decode.hip).
int decode_max_vis(const lmx_attn_params* p);

constexpr float kRescaleSlack = 8.f;  // log2 units a running max may lag by

// attn.wgsl:52-66
__device__ __forceinline__ int vis_lo(int pos, int w) { return (w && pos + 1 > w) ? pos + 1 - w : 0; }
__device__ __forceinline__ int vis_hi(int pos, int w, int bidi, int end) {
    if (!bidi) return pos;
    return w ? min(end, pos + w - 1) : end;
}

// Q fragments as values defined here, not the registers of their loads (an
// f16 query's conversions fold away): otherwise the waitcnt pass counts Q's
// loads as possibly pending inside the key loop and puts vmcnt(n) waits
// between the score MFMAs, which drain the K/V prefetch of later tiles.
template <int N>
__device__ __forceinline__ void settle_q(f16x8 (&qf)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(qf[i]));
}

// s_waitcnt vmcnt(0) as an instruction the compiler's waitcnt pass sees
// (inline assembly it does not): every load issued before it is complete.
__device__ __forceinline__ void drain_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

}  // namespace lmx
