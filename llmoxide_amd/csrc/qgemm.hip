// GEMM on gfx950 matrix cores: Y[t][r] = sum_k W[r][k] X[t][k] for a batch of
// tokens and a weight matrix in ggml's on-disk formats Q4_K, Q6_K, Q8_0, F16
// or BF16, read once per launch.
//
// Replaces the reference's prefill GEMM (gemm_q6k in gemm.wgsl:93-95 and
// gemm_q6k.metal:50, chosen from 16 tokens: crates/gpu/src/lib.rs:1039-1046,
// 1083) and computes what its CPU reference dot_row computes
// (crates/gguf/src/quant.rs:187-271), to fp32 accuracy:
//
//   The block formats: qgemm.hpp.
//   x, scaled (below), is split into f16 x_hi + x_lo, and all products run on
//   v_mfma_f32_32x32x16_f16 with fp32 accumulation.  The integer scales go
//   into the weight operand, where the vector unit pays for them once a weight instead of once a token: sc_g q of Q4_K is at most 945
//   and exact in f16; of Q6_K it is at most 4096 and exact as f16(sc_g q) plus
//   a remainder (third product: remainder times x_hi).  Only d, one a
//   super-block of 256, is applied to the fp32 sums (of a bf16 row, the power
//   of two that brought 256 / KQ of its weights into f16's range).  Q4_K's offsets are one
//   more MFMA a super-block: the m_g against the group sums of the scaled x
//   (hi and lo, times 1/16: at most 2^15).  Q8_0's d has 11 bits of its own, so its
//   group sums are scaled in fp32.
//
//   Range: before the split, each token's x is multiplied by a power of two
//   2^k_t (exact).  Its first nonzero chunk sets k_t so that the chunk's
//   largest |x| lands in [2^11, 2^12); a later chunk whose scaled |x| reach
//   2^14 lowers it to do the same.  So no scaled value comes near f16's 65504,
//   and |x - x_hi - x_lo| is at most 2^-22 |x| for every x down to 2^-14 of
//   the largest met, and 2^-36 of that largest below: f16's subnormals begin
//   at 2^-14, so a residual keeps its 11 bits only from a scaled |x| of 2^-3
//   up.  (Left unscaled, x of rms 0.006 cost 2.9e-6 of the result, 0.1 2.1e-7;
//   the matvec costs 1.0e-7 to 2.7e-7, this 1.2e-7 to 1.9e-7 at any rms.)  Every
//   partial sum of a token is in one scaled domain: when a chunk lowers k_t,
//   the token's accumulated y is first multiplied by the (exact) ratio, and
//   the store multiplies by 2^-k_t.  Infinities: see qgemm_kernel.
//
// A workgroup of eight waves owns 32 TT tokens x 32 RT WR rows and walks K in
// chunks of 256.  x goes through LDS, two buffers of swizzled f16 hi / lo
// rows: each wave loads, splits and stores TM / 8 tokens of the next chunk
// beside its MFMAs, its loads a chunk ahead of that.  A chunk's raw weight
// bytes come from memory straight to LDS, in 16-byte pieces that cover each
// row's block (whole lines; 2- and 4-byte loads of the 2-byte aligned fields
// kept the address unit busy for longer than the MFMAs); each wave reads the
// bytes of its own k range (KQ = 8 / WR ranges a chunk) into registers, and
// decodes them there into MFMA operands, each weight once a workgroup.  The
// KQ partial sums meet in LDS at the end.
//
// Measured (in_dim 4096, us a call; before: 64 x 128 tiles with one wave kind
// per stage for the block formats, four tokens a launch for dense rows):
// 16 tokens x 4096 rows Q4_K 81 -> 25, Q6_K 116 -> 29, Q8_0 94 -> 22, bf16
// 103 -> 25; 500 x 1024 rows 83 -> 40, 120 -> 39, 99 -> 34, 2577 -> 36; 64 x
// 4096 rows bf16 433 -> 36.  What bounds it: a workgroup's chunks come one after
// the other, each a round trip (its x and W loads are a chunk ahead; 1.5 us at
// 32 tokens) or x's staging (2.1 us a chunk at 64), with the vector unit busy 57
// to 65% of the time and the matrix pipe 3 to 14%.
#include <algorithm>
#include <climits>

#include "lds_dma.hpp"
#include "qgemm.hpp"

namespace lmx {

template <int TY>
constexpr bool g_dense() { return TY == kGF16 || TY == kGBF16; }

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

constexpr int kGK = 256;  // k per chunk: a K-quant super-block, eight Q8_0 blocks

// Bytes of a chunk of a row, the 16-byte pieces that cover it at its largest
// misalignment (blocks of Q4_K are 16-byte aligned, the others 2-byte), and
// the pieces' stride in LDS: odd, so that 16 rows of one piece meet all banks.
template <int TY>
struct GTraits;
template <> struct GTraits<kGQ4K> { static constexpr int bytes = 144, pieces = 9, stride = 9; };
template <> struct GTraits<kGQ6K> { static constexpr int bytes = 210, pieces = 14, stride = 15; };
template <> struct GTraits<kGQ8_0> { static constexpr int bytes = 272, pieces = 18, stride = 19; };
template <> struct GTraits<kGF16> { static constexpr int bytes = 512, pieces = 32, stride = 33; };
template <> struct GTraits<kGBF16> { static constexpr int bytes = 512, pieces = 32, stride = 33; };

struct GemmArgs {
    const uint8_t* w;
    const float* x;
    float* y;
    int rows, in_dim, n_tok;
    size_t row_bytes, w_bytes;
};

// max(|a|, |b|, c) as one instruction (fmaxf first quiets each operand).
__device__ __forceinline__ float absmax3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// Largest x over the wave's 64 lanes (x >= 0).
__device__ __forceinline__ float wave_max64(float x) {
    x = fmaxf(x, dpp<0xB1>(x));   // quad_perm [1,0,3,2]
    x = fmaxf(x, dpp<0x4E>(x));   // quad_perm [2,3,0,1]
    x = fmaxf(x, dpp<0x141>(x));  // row_half_mirror
    x = fmaxf(x, dpp<0x140>(x));  // row_mirror
    const int b = __builtin_bit_cast(int, x);
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0));
    const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32));
    const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
    return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

__device__ __forceinline__ f16x2 as_h2(uint32_t x) { return __builtin_bit_cast(f16x2, x); }
__device__ __forceinline__ uint32_t lds_u16(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }
// N dwords at a 2-byte aligned LDS address.
template <int N>
__device__ __forceinline__ void lds_words(const uint8_t* p, uint32_t (&o)[N]) {
    const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 2);
    const uint32_t* b = reinterpret_cast<const uint32_t*>(p - sh);
    uint32_t raw[N + 1];
#pragma unroll
    for (int i = 0; i <= N; ++i) raw[i] = b[i];
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], sh);
}
// Four small unsigned integers (bytes) as f16 + 1024, in the order 0 2 1 3 in
// which x is stored (masks instead of byte moves).
__device__ __forceinline__ void bytes_1024(uint32_t q, f16x2& a, f16x2& b) {
    a = as_h2((q & 0x00FF00FFu) | 0x64006400u);
    b = as_h2(((q >> 8) & 0x00FF00FFu) | 0x64006400u);
}
__device__ __forceinline__ f16x2 pk_fma(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }

// An infinity or NaN as +-65504.
__device__ __forceinline__ f16x2 finite2(f16x2 x) {
    const f16x2 hi = {(f16)65504.f, (f16)65504.f}, lo = {(f16)-65504.f, (f16)-65504.f};
    return __builtin_elementwise_min(__builtin_elementwise_max(x, lo), hi);
}

// A wave's share of a chunk of one weight row: its raw bytes, read from LDS
// once, and the operand of each of its k-steps.  KQ ranges a chunk; lane half
// hh holds 8 weights a step.
//   Q4_K  range = pair of sub-blocks (KQ 4) or one (KQ 8); the half's 16 quant
//         bytes; steps: low nibbles of bytes 0-7, 8-15, then the high ones
//   Q6_K  range = half h, l in [16 lq, + 16) of every quarter k (KQ 4) or of
//         quarters 2 kn, 2 kn + 1 (KQ 8); the half's 8 l; a step per quarter,
//         which is one scale group
//   Q8_0  range = two blocks (KQ 4) or one; the half's 16 weights of each
template <int TY, int KQ>
struct WFrag;

template <int KQ>
struct WFrag<kGQ4K, KQ> {
    static constexpr int NK = 16 / KQ;
    uint32_t hdr[4], q[4];
    __device__ __forceinline__ void load(const uint8_t* blk, int kq, int hh) {
        const uint4 h = *reinterpret_cast<const uint4*>(blk);
        const uint4 v = *reinterpret_cast<const uint4*>(blk + 16 + 32 * (KQ == 4 ? kq : kq >> 1) + 16 * hh);
        hdr[0] = h.x; hdr[1] = h.y; hdr[2] = h.z; hdr[3] = h.w;
        q[0] = v.x; q[1] = v.y; q[2] = v.z; q[3] = v.w;
    }
    __device__ static __forceinline__ int k_of(int s, int kq, int hh) {
        return KQ == 4 ? 64 * kq + 32 * (s >> 1) + 16 * hh + 8 * (s & 1) : 32 * kq + 16 * hh + 8 * s;
    }
    // 6-bit scale and min of sub-block j, quant.rs:33-47
    __device__ __forceinline__ uint32_t scale(int j) const {
        const int s = 8 * (j & 3);
        const uint32_t b0 = (hdr[1] >> s) & 0xFF, b2 = (hdr[3] >> s) & 0xFF;
        return j < 4 ? b0 & 63 : (b2 & 0xF) | ((b0 >> 6) << 4);
    }
    __device__ __forceinline__ f16x8 step(int s, int kq) const {
        const int j = KQ == 4 ? 2 * kq + (s >> 1) : kq;  // sub-block
        const int hi = 4 * (j & 1);
        const f16 sc = (f16)(float)scale(j);
        const f16x2 s2 = {sc, sc}, n2 = f16x2{(f16)-1024.f, (f16)-1024.f} * s2;
        f16x8 o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t v = q[2 * (s & 1) + i] >> hi;
            // (1024 + q) sc - 1024 sc, exact
            const f16x2 a = pk_fma(as_h2((v & 0x000F000Fu) | 0x64006400u), s2, n2);
            const f16x2 b = pk_fma(as_h2(((v >> 8) & 0x000F000Fu) | 0x64006400u), s2, n2);
            o[4 * i] = a[0]; o[4 * i + 1] = a[1]; o[4 * i + 2] = b[0]; o[4 * i + 3] = b[1];
        }
        return o;
    }
    __device__ __forceinline__ float d() const { return (float)as_h2(hdr[0])[0]; }
    __device__ __forceinline__ float dmin() const { return (float)as_h2(hdr[0])[1]; }
    __device__ __forceinline__ f16x8 mins() const {
        f16x8 m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t b1 = (hdr[2] >> (8 * j)) & 0xFF, b2 = (hdr[3] >> (8 * j)) & 0xFF;
            m[j] = (f16)(float)(b1 & 63);
            m[j + 4] = (f16)(float)((b2 >> 4) | ((b1 >> 6) << 4));
        }
        return m;
    }
};

template <int KQ>
struct WFrag<kGQ6K, KQ> {
    static constexpr int NK = 16 / KQ;
    uint32_t la[2], lb[2], h[2], sc[2], dd;
    __device__ __forceinline__ void load(const uint8_t* blk, int kq, int hh) {
        const int half = KQ == 4 ? kq >> 1 : kq >> 2, lq = KQ == 4 ? kq & 1 : (kq >> 1) & 1;
        const int l0 = 16 * lq + 8 * hh;
        lds_words<2>(blk + 64 * half + l0, la);
        lds_words<2>(blk + 64 * half + 32 + l0, lb);
        lds_words<2>(blk + 128 + 32 * half + l0, h);
        lds_words<2>(blk + 192 + 8 * half, sc);
        dd = lds_u16(blk + 208);
    }
    __device__ static __forceinline__ int quarter(int s, int kq) { return KQ == 4 ? s : 2 * (kq & 1) + s; }
    __device__ static __forceinline__ int k_of(int s, int kq, int hh) {
        const int half = KQ == 4 ? kq >> 1 : kq >> 2, lq = KQ == 4 ? kq & 1 : (kq >> 1) & 1;
        return 128 * half + 32 * quarter(s, kq) + 16 * lq + 8 * hh;
    }
    // hi + lo = sc q, both exact
    __device__ __forceinline__ void step(int s, int kq, f16x8& hi, f16x8& lo) const {
        const int k = quarter(s, kq), lq = KQ == 4 ? kq & 1 : (kq >> 1) & 1;
        const int g = 2 * k + lq;
        const f16 c = (f16)(float)(int8_t)((g < 4 ? sc[0] : sc[1]) >> (8 * (g & 3)));
        const f16x2 c2 = {c, c}, off = {(f16)-1056.f, (f16)-1056.f};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t ql = ((k & 1) ? lb[i] : la[i]) >> (4 * (k >> 1));
            const uint32_t q = (ql & 0x0F0F0F0Fu) | (((h[i] >> (2 * k)) << 4) & 0x30303030u);
            f16x2 a, b;
            bytes_1024(q, a, b);
            a += off;
            b += off;
            const f16x2 ah = a * c2, bh = b * c2;
            const f16x2 al = pk_fma(a, c2, -ah), bl = pk_fma(b, c2, -bh);
            hi[4 * i] = ah[0]; hi[4 * i + 1] = ah[1]; hi[4 * i + 2] = bh[0]; hi[4 * i + 3] = bh[1];
            lo[4 * i] = al[0]; lo[4 * i + 1] = al[1]; lo[4 * i + 2] = bl[0]; lo[4 * i + 3] = bl[1];
        }
    }
    __device__ __forceinline__ float d() const { return (float)as_h2(dd)[0]; }
};

template <int KQ>
struct WFrag<kGQ8_0, KQ> {
    static constexpr int NK = 16 / KQ, NB = NK / 2;
    uint32_t q[NB][4], dd[NB];
    __device__ __forceinline__ void load(const uint8_t* blk, int kq, int hh) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const uint8_t* p = blk + 34 * (NB * kq + b);
            dd[b] = lds_u16(p);
            lds_words<4>(p + 2 + 16 * hh, q[b]);
        }
    }
    __device__ static __forceinline__ int k_of(int s, int kq, int hh) {
        return 32 * (NB * kq + (s >> 1)) + 16 * hh + 8 * (s & 1);
    }
    __device__ __forceinline__ f16x8 step(int s) const {
        const f16x2 off = {(f16)-1152.f, (f16)-1152.f};
        f16x8 o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            f16x2 a, b;
            bytes_1024(q[s >> 1][2 * (s & 1) + i] ^ 0x80808080u, a, b);  // q + 128
            a += off;
            b += off;
            o[4 * i] = a[0]; o[4 * i + 1] = a[1]; o[4 * i + 2] = b[0]; o[4 * i + 3] = b[1];
        }
        return o;
    }
    __device__ __forceinline__ float d(int b) const { return (float)as_h2(dd[b])[0]; }
};

// Dense rows: range = 256 / KQ consecutive weights.  bf16 becomes f16 times a
// power of two that brings the range's largest finite weight into [2^14, 2^15):
// exact for weights down to 2^-31 of it, 2^-39 of it below.
template <int TY, int KQ>
struct DFrag {
    static constexpr int NK = 16 / KQ;
    uint4 raw[NK];
    int sc;
    __device__ static __forceinline__ int k_of(int s, int kq, int hh) { return 16 * (NK * kq + s) + 8 * hh; }
    // left: weights of the chunk that lie inside the row
    __device__ __forceinline__ void load(const uint8_t* row, int kq, int hh, int left) {
        u16x2 top = {0, 0};  // largest magnitudes (bit patterns order as their values)
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            const int k = k_of(s, kq, hh);
            raw[s] = k < left ? *reinterpret_cast<const uint4*>(row + 2 * k) : uint4{0u, 0u, 0u, 0u};
        }
        auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                const uint32_t w[4] = {raw[s].x, raw[s].y, raw[s].z, raw[s].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) f(__builtin_bit_cast(u16x2, w[i] & 0x7FFF7FFFu));
            }
        };
        sc = 0;
        if constexpr (TY == kGBF16) {
            each([&](u16x2 m) { top = __builtin_elementwise_max(top, m); });
            constexpr uint16_t inf = 0x7F80;
            if (__builtin_amdgcn_ballot_w64(max(top[0], top[1]) >= inf)) {  // the largest finite one, then
                top = u16x2{0, 0};
                each([&](u16x2 m) {
                    const u16x2 fin = {m[0] < inf ? m[0] : (uint16_t)0, m[1] < inf ? m[1] : (uint16_t)0};
                    top = __builtin_elementwise_max(top, fin);
                });
            }
            const float t = __builtin_bit_cast(float, (uint32_t)max(top[0], top[1]) << 16);
            const float m = fmaxf(t, shfl_xor(t, 32));
            if (m > 0.f) sc = 15 - __builtin_amdgcn_frexp_expf(m);
        }
    }
    __device__ __forceinline__ f16x8 step(int s) const {
        const uint32_t w[4] = {raw[s].x, raw[s].y, raw[s].z, raw[s].w};
        f16x8 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // pairs (0 1) (2 3) .. into the order 0 2 1 3
            f16 a, b;
            if constexpr (TY == kGBF16) {
                a = (f16)__builtin_amdgcn_ldexpf(__builtin_bit_cast(float, w[i] << 16), sc);
                b = (f16)__builtin_amdgcn_ldexpf(__builtin_bit_cast(float, w[i] & 0xFFFF0000u), sc);
            } else {
                a = as_h2(w[i])[0];
                b = as_h2(w[i])[1];
            }
            o[4 * (i >> 1) + (i & 1)] = a;
            o[4 * (i >> 1) + 2 + (i & 1)] = b;
        }
        return o;
    }
    __device__ __forceinline__ float d() const { return __builtin_amdgcn_ldexpf(1.f, -sc); }
};
template <int KQ>
struct WFrag<kGF16, KQ> : DFrag<kGF16, KQ> {};
template <int KQ>
struct WFrag<kGBF16, KQ> : DFrag<kGBF16, KQ> {};

template <int TY, int TT, int RT, int WR>
struct GemmLds {
    static constexpr int TM = 32 * TT, TN = 32 * RT * WR, KQ = 8 / WR;
    // x rows of 256 halfs, 16-byte pieces XORed with the row, hi and lo of two
    // chunks; also the partial sums at the end
    static constexpr int XB = TM * kGK;
    static constexpr int X = 2 * 2 * XB * 2, Y = KQ * TM * TN * 4;
    alignas(16) unsigned char xy[X > Y ? X : Y];
    alignas(16) unsigned char w[TN * GTraits<TY>::stride * 16 + 16];
    alignas(16) f16 xs[2][TY == kGQ4K ? TM * 16 : 8];  // x sums / 16: 8 hi, 8 lo
    alignas(16) float rs[2][TM];  // a token's scale ratio of this chunk
    alignas(16) int chg[2][8];    // per staging wave: some ratio is not 1
    int k[TM];  // a token's scale exponent after the last chunk
    int nan;    // some result is NaN
};

// INF: dense rows, with infinite x and weights kept apart from the split's 0
// (see qgemm_kernel).
template <int TY, int TT, int RT, int WR, bool INF>
__device__ __forceinline__ void qgemm_tile(const GemmArgs& a, GemmLds<TY, TT, RT, WR>& lds) {
    constexpr int TM = 32 * TT, TN = 32 * RT * WR, KQ = 8 / WR;
    constexpr int NK = 16 / KQ;  // k-steps of a wave per chunk
    constexpr int STR = GTraits<TY>::stride * 16, PC = GTraits<TY>::stride, NPC = GTraits<TY>::pieces;
    constexpr int NX = TM / 8;   // tokens a wave stages per chunk
    constexpr bool OFFSET = TY == kGQ4K;
    constexpr int XB = TM * kGK;
    auto& xy_s = lds.xy;
    auto& w_s = lds.w;
    auto& xs_s = lds.xs;
    auto& rs_s = lds.rs;
    auto& chg_s = lds.chg;
    auto& k_s = lds.k;
    auto xh = [&](int b) { return reinterpret_cast<f16*>(xy_s) + b * 2 * XB; };
    auto xl = [&](int b) { return xh(b) + XB; };

    const int n_tb = (a.n_tok + TM - 1) / TM;
    const int tb = blockIdx.x % n_tb, rb = blockIdx.x / n_tb;
    const int t0 = tb * TM, r0 = rb * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hh = lane >> 5;
    const int kq = wave % KQ, wr = wave / KQ;
    const int n_chunks = (a.in_dim + kGK - 1) / kGK;

    // ---- weights: piece p of the tile is piece p % PC of row p / PC.  Rows
    // past the matrix repeat its last one; a piece that would reach past the
    // matrix is put together from its 2-byte words.
    auto fetch_w = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < (TN * PC + 511) / 512; ++i) {
            const int n = wave + 8 * i, p = n * 64 + lane;
            const int row = p / PC, c = p % PC;
            if (row < TN && c < NPC) {
                const size_t at = (size_t)min(r0 + row, a.rows - 1) * a.row_bytes + (size_t)ch * GTraits<TY>::bytes;
                const size_t off = (at & ~(size_t)15) + 16 * c;
                if (TY == kGQ4K || off + 16 <= a.w_bytes) {  // (a Q4_K row is whole pieces)
                    dma16_lane(a.w + off, lds_addr(w_s) + n * 1024);
                } else {
#pragma unroll 1
                    for (int u = 0; u < 8; ++u)
                        *reinterpret_cast<uint16_t*>(w_s + p * 16 + 2 * u) =
                            off + 2 * u + 2 <= a.w_bytes ? *reinterpret_cast<const uint16_t*>(a.w + off + 2 * u) : 0;
                }
            }
        }
    };
    // ---- x: token wave * NX + u, floats 4 lane .. + 3 of the chunk
    f32x4 rx[NX];
    // running scale exponents; kNone, which no chunk sets (the smallest
    // denormal sets 12 + 148): no nonzero x yet
    constexpr int kNone = 1000;
    int kx[NX];
#pragma unroll
    for (int u = 0; u < NX; ++u) kx[u] = kNone;
    auto load_x = [&](int ch) __attribute__((always_inline)) {
        const int k = ch * kGK + 4 * lane;
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            // tokens past the batch repeat its last one and are not stored
            const int tok = min(t0 + wave * NX + u, a.n_tok - 1);
            rx[u] = *reinterpret_cast<const f32x4*>(a.x + (size_t)tok * a.in_dim + min(k, a.in_dim - 4));
        }
    };
    int ones = 0;  // bit b: buffer b's ratios of this wave's tokens are 1 (uniform)
    // One token's floats to hi / lo rows, and (Q4_K) its group sums.
    auto emit = [&](int b, int u, const f32x4& v) __attribute__((always_inline)) {
        const int tok = wave * NX + u;
        // hi once (pinned: the residual is taken against these very
        // registers); in the order 0 2 1 3
        f16x2 h0 = {(f16)v[0], (f16)v[2]}, h1 = {(f16)v[1], (f16)v[3]};
        if constexpr (INF) h0 = finite2(h0), h1 = finite2(h1);  // an infinite x: all residual (inf - inf is NaN)
        asm("" : "+v"(h0), "+v"(h1));
        const f16x4 hi = {h0[0], h0[1], h1[0], h1[1]};
        const f16x4 lo = {(f16)(v[0] - (float)h0[0]), (f16)(v[2] - (float)h0[1]), (f16)(v[1] - (float)h1[0]),
                          (f16)(v[3] - (float)h1[1])};
        const int at = tok * kGK + (((lane >> 1) ^ (tok & 15)) << 3) + 4 * (lane & 1);
        *reinterpret_cast<f16x4*>(xh(b) + at) = hi;
        *reinterpret_cast<f16x4*>(xl(b) + at) = lo;
        if constexpr (OFFSET) {
            // the sum of each group of 32: eight lanes hold its floats; lane 8 g
            // stores the hi part, lane 8 g + 1 the lo part
            const float sx = sum8((v[0] + v[1]) + (v[2] + v[3])) * 0.0625f;
            const f16 h = (f16)sx;
            const f16 l = (f16)(sx - (float)h);
            if ((lane & 7) < 2) xs_s[b][tok * 16 + 8 * (lane & 1) + (lane >> 3)] = lane & 1 ? l : h;
        }
    };
    auto stash_x = [&](int b, int ch) __attribute__((always_inline)) {
        if ((TY == kGQ8_0 || g_dense<TY>()) && ch * kGK + 4 * lane >= a.in_dim) {  // K may end inside a chunk
#pragma unroll
            for (int u = 0; u < NX; ++u) rx[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // nothing changes while no scaled |x| reaches 2^14 (a NaN passes through
        // as it is; before a token's first nonzero x its scale takes any to inf)
        f32x4 v[NX];
        float top = 0.f;
        auto scale = [&](int u) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[u][j] = __builtin_amdgcn_ldexpf(rx[u][j], kx[u]);
        };
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            scale(u);
            top = absmax3(v[u][2], v[u][3], absmax3(v[u][0], v[u][1], top));
        }
        if (__builtin_amdgcn_ballot_w64(top >= 16384.f) == 0) {
            if (!(ones >> b & 1)) {
                if (lane < NX) rs_s[b][wave * NX + lane] = 1.f;
                if (lane == 0) chg_s[b][wave] = 0;
                ones |= 1 << b;
            }
        } else {
            int changed = 0;
#pragma unroll
            for (int u = 0; u < NX; ++u) {
                float m = wave_max64(absmax3(rx[u][2], rx[u][3], absmax3(rx[u][0], rx[u][1], 0.f)));
                if (m > 3.402823466e38f) {  // (uniform) the largest finite one, then
                    m = 0.f;
#pragma unroll
                    for (int j = 0; j < 4; ++j) m = fmaxf(m, fabsf(rx[u][j]) <= 3.402823466e38f ? fabsf(rx[u][j]) : 0.f);
                    m = wave_max64(m);
                }
                int kn = kx[u];
                if (m > 0.f && __builtin_amdgcn_ldexpf(m, kn) >= 16384.f)
                    kn = 12 - __builtin_amdgcn_frexp_expf(m);
                // (y is 0 or not finite before the first nonzero x; a ratio
                // below 2^-126 leaves nothing of a finite y, and must not be 0
                // beside an infinite one)
                const float ratio = kx[u] == kNone ? 1.f : __builtin_amdgcn_ldexpf(1.f, max(kn - kx[u], -126));
                kx[u] = kn;
                changed |= ratio != 1.f;
                if (lane == 0) rs_s[b][wave * NX + u] = ratio;
                scale(u);
            }
            if (lane == 0) chg_s[b][wave] = changed;
            ones &= ~(1 << b);
        }
#pragma unroll
        for (int u = 0; u < NX; ++u) emit(b, u, v[u]);
    };

    f32x16 y[TT][RT];
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int n = 0; n < RT; ++n)
#pragma unroll
            for (int j = 0; j < 16; ++j) y[i][n][j] = 0.f;

    fetch_w(0);
    load_x(0);
    stash_x(0, 0);
    if (n_chunks > 1) load_x(1);
    for (int ch = 0; ch < n_chunks; ++ch) {
        const int b = ch & 1;
        // the chunk's bytes; this wave's x loads, issued after them, may still
        // be in flight
        if (ch > 0 && ch + 1 < n_chunks) wait_dma<NX>();
        else wait_dma<0>();
        __syncthreads();  // chunk ch is in LDS
        WFrag<TY, KQ> w[RT];
#pragma unroll
        for (int n = 0; n < RT; ++n) {
            const int row = (wr * RT + n) * 32 + l32;
            uint32_t sh = 0;
            if constexpr (TY != kGQ4K && !g_dense<TY>())
                sh = (uint32_t)((size_t)min(r0 + row, a.rows - 1) * a.row_bytes + (size_t)ch * GTraits<TY>::bytes) & 15;
            if constexpr (g_dense<TY>()) w[n].load(w_s + row * STR, kq, hh, a.in_dim - ch * kGK);
            else w[n].load(w_s + row * STR + sh, kq, hh);
        }
        const int4 c0 = *reinterpret_cast<const int4*>(&chg_s[b][0]), c1 = *reinterpret_cast<const int4*>(&chg_s[b][4]);
        const int chg = c0.x | c0.y | c0.z | c0.w | c1.x | c1.y | c1.z | c1.w;
        __syncthreads();  // the weight bytes are in registers
        if (ch + 1 < n_chunks) {
            stash_x(b ^ 1, ch + 1);  // (before the transfers: its wait for x would wait for them too)
            fetch_w(ch + 1);
            if (ch + 2 < n_chunks) load_x(ch + 2);
        }
        // token of register j: 8 (j / 4) + 4 hh + j % 4 of the tile's 32
        if (__builtin_amdgcn_readfirstlane(chg)) {
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 r = *reinterpret_cast<const f32x4*>(&rs_s[b][32 * i + 8 * g + 4 * hh]);
#pragma unroll
                    for (int n = 0; n < RT; ++n)
#pragma unroll
                        for (int j = 0; j < 4; ++j) y[i][n][4 * g + j] *= r[j];
                }
        }
        auto x_at = [&](const f16* xb, int i, int k) {
            return *reinterpret_cast<const f16x8*>(xb + (32 * i + l32) * kGK + (((k >> 3) ^ (l32 & 15)) << 3));
        };
        f32x16 acc[TT][RT];
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            const int k = WFrag<TY, KQ>::k_of(s, kq, hh);
            f16x8 ah[TT], al[TT];
#pragma unroll
            for (int i = 0; i < TT; ++i) {
                ah[i] = x_at(xh(b), i, k);
                al[i] = x_at(xl(b), i, k);
            }
            const bool first = TY == kGQ8_0 ? s % 2 == 0 : s == 0;
            if (first) {
#pragma unroll
                for (int i = 0; i < TT; ++i)
#pragma unroll
                    for (int n = 0; n < RT; ++n)
#pragma unroll
                        for (int j = 0; j < 16; ++j) acc[i][n][j] = 0.f;
            }
#pragma unroll
            for (int n = 0; n < RT; ++n) {
                f16x8 q, ql, qf;  // qf: beside x_lo
                if constexpr (TY == kGQ6K) w[n].step(s, kq, q, ql);
                else if constexpr (TY == kGQ4K) q = w[n].step(s, kq);
                else q = w[n].step(s);
                qf = q;
                if constexpr (INF)
#pragma unroll
                    for (int i = 0; i < 8; i += 2) {
                        const f16x2 f = finite2(f16x2{q[i], q[i + 1]});
                        qf[i] = f[0];
                        qf[i + 1] = f[1];
                    }
#pragma unroll
                for (int i = 0; i < TT; ++i) {
                    acc[i][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], q, acc[i][n], 0, 0, 0);
                    acc[i][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i], qf, acc[i][n], 0, 0, 0);
                    if constexpr (TY == kGQ6K)
                        acc[i][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], ql, acc[i][n], 0, 0, 0);
                }
            }
            if constexpr (TY == kGQ8_0) {
                if (s % 2 == 1) {  // a block is done
                    // blocks past the matrix (K a half chunk short) hold other bytes
                    const bool in = ch * kGK + (k & ~31) < a.in_dim;
#pragma unroll
                    for (int n = 0; n < RT; ++n) {
                        const float d = in ? w[n].d(s / 2) : 0.f;
#pragma unroll
                        for (int i = 0; i < TT; ++i)
#pragma unroll
                            for (int j = 0; j < 16; ++j) y[i][n][j] = fmaf(d, acc[i][n][j], y[i][n][j]);
                    }
                }
            }
        }
        if constexpr (TY != kGQ8_0) {
#pragma unroll
            for (int n = 0; n < RT; ++n) {
                const float d = w[n].d();
#pragma unroll
                for (int i = 0; i < TT; ++i)
#pragma unroll
                    for (int j = 0; j < 16; ++j) y[i][n][j] = fmaf(d, acc[i][n][j], y[i][n][j]);
            }
        }
        if constexpr (OFFSET) {
            if (kq == ch % KQ) {  // the ranges take the chunks' offsets in turn
#pragma unroll
                for (int n = 0; n < RT; ++n) {
                    const f16x8 m = w[n].mins();
                    const float dm = -16.f * w[n].dmin();
#pragma unroll
                    for (int i = 0; i < TT; ++i) {
                        const f16x8 xs = *reinterpret_cast<const f16x8*>(&xs_s[b][(32 * i + l32) * 16 + 8 * hh]);
                        f32x16 z;
#pragma unroll
                        for (int j = 0; j < 16; ++j) z[j] = 0.f;
                        z = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs, m, z, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 16; ++j) y[i][n][j] = fmaf(dm, z[j], y[i][n][j]);
                    }
                }
            }
        }
    }

    // ---- the KQ partial sums, [range][token][row], through the x buffers;
    // each staging wave knows its tokens' final exponents
    __syncthreads();
    float* y_s = reinterpret_cast<float*>(xy_s);
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int n = 0; n < RT; ++n)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int tok = 32 * i + 8 * (j >> 2) + 4 * hh + (j & 3);
                y_s[(kq * TM + tok) * TN + (wr * RT + n) * 32 + l32] = y[i][n][j];
            }
    if (lane == 0)
#pragma unroll
        for (int u = 0; u < NX; ++u) k_s[wave * NX + u] = kx[u] == kNone ? 0 : kx[u];
    if (tid == 0) lds.nan = 0;
    __syncthreads();
#pragma unroll
    for (int i = tid; i < TM * TN; i += 512) {
        const int tok = i / TN, row = i % TN;
        if (t0 + tok >= a.n_tok || r0 + row >= a.rows) continue;
        float v = y_s[i];
#pragma unroll
        for (int q = 1; q < KQ; ++q) v += y_s[q * TM * TN + i];
        a.y[(size_t)(t0 + tok) * a.rows + r0 + row] = __builtin_amdgcn_ldexpf(v, -k_s[tok]);
        if (g_dense<TY>() && !INF && v != v) lds.nan = 1;
    }
}

// The split gives NaN where an infinite x or a dense row's infinite weight
// makes a product infinite (inf - inf in the residual, 0 times inf beside an
// x that f16 holds).  The block formats' matvec does so too; the dense one
// gives inf.  So a dense tile with a NaN among its results is done again with
// both kept finite in one of the two products: the same sums elsewhere.
// (Testing for them in the first pass cost 3 to 8% of every call.)  An x that
// is 0 in f16 once scaled, 2^-36 of the token's largest, still counts as 0.
template <int TY, int TT, int RT, int WR>
__global__ __launch_bounds__(512, 1) void qgemm_kernel(GemmArgs a) {
    __shared__ GemmLds<TY, TT, RT, WR> lds;
    qgemm_tile<TY, TT, RT, WR, false>(a, lds);
    if constexpr (g_dense<TY>()) {
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(lds.nan)) qgemm_tile<TY, TT, RT, WR, true>(a, lds);
    }
}

template <int TY, int TT, int RT, int WR>
static void launch(const GemmArgs& a, hipStream_t st) {
    constexpr int TM = 32 * TT, TN = 32 * RT * WR;
    const long grid = ((long)a.n_tok + TM - 1) / TM * ((a.rows + TN - 1) / TN);
    hipLaunchKernelGGL((qgemm_kernel<TY, TT, RT, WR>), dim3((unsigned)grid), dim3(512), 0, st, a);
}

// Tiles.  Up to 32 tokens: 32 x 32, or 32 x 64 where those still make a
// workgroup for every CU (fewer rows raise the share of x's staging, which
// every workgroup of a token block repeats).  Dense rows beside more tokens: 64
// x 32, whose x leaves LDS for no more.  Block formats beside more: 64 tokens x
// 32, 64 or 128 (qgemm_big.hip) rows.  A CU holds one workgroup, so a call
// takes as many rounds as its grid has times 256, each about as long whatever
// is in it.  us a round at in_dim 4096 (1024): 64 x 32 Q4_K 41 (16), Q6_K 40
// (16), Q8_0 34 (14); 64 x 64 50 (20), 51 (20), 46 (18); 64 x 128 65 (23), 84
// (29), 71 (23), and where the last token block is not whole 84 (27), 118 (37),
// 98 (33).  The least rounds times that is taken; from 256 workgroups of 64 x
// 128 on those always are.  us a call, 64 x 128 everywhere / 64 x 64 wherever it
// made 256 workgroups / now: Q4_K 64 tokens x 12288 x 4096 65 / 79 / 49, 512 x
// 3000 x 4096 68 / 95 / 66; Q6_K 128 x 6000 x 4096 84 / 76 / 50, 512 x 3000 x
// 4096 86 / 96 / 87, 400 x 3000 x 4096 121 / 96 / 96.
constexpr long kCus = 256;
static long blocks(const GemmArgs& a, int tm, int tn) {
    return ((long)a.n_tok + tm - 1) / tm * ((a.rows + tn - 1) / tn);
}
// Rows of a block format's tile of 64 tokens.
static int tile_rows(const GemmArgs& a, uint32_t type) {
    if (blocks(a, 64, 128) >= kCus) return 128;
    // in hundredths of a 64 x 32 round
    const int big = a.n_tok % 64 ? (type == kGQ4K ? 200 : 290) : type == kGQ4K ? 160 : 205;
    const int mid = type == kGQ4K ? 122 : type == kGQ6K ? 128 : 135;
    auto rounds = [&](int tn) { return (blocks(a, 64, tn) + kCus - 1) / kCus; };
    const long c32 = rounds(32) * 100, c64 = rounds(64) * mid;
    if (std::min(c32, c64) > big) return 128;
    return c64 < c32 ? 64 : 32;
}
template <int TY>
static void launch_type(const GemmArgs& a, int tn, hipStream_t st) {
    if (a.n_tok <= 32) {
        if (blocks(a, 32, 64) >= kCus) launch<TY, 1, 1, 2>(a, st);
        else launch<TY, 1, 1, 1>(a, st);
    } else if (!g_dense<TY>() && tn == 64) {
        if constexpr (!g_dense<TY>()) launch<TY, 2, 1, 2>(a, st);
    } else {
        launch<TY, 2, 1, 1>(a, st);
    }
}

// qgemm_big.hip
lmx_status qgemm_big(const lmx_qmv_desc* d, const void* w, const float* x, float* y, hipStream_t st);

// y [n_tok, rows] = W x: one launch, W read once from HBM (each of the
// token blocks of a row block reads it from L2 or the last-level cache after
// the first).
lmx_status qgemm(const lmx_qmv_desc* d, const void* w, const float* x, float* y, hipStream_t st) {
    size_t bb = 0, be = 0;
    switch (d->type) {
        case kGQ4K: bb = 144; be = 256; break;
        case kGQ6K: bb = 210; be = 256; break;
        case kGQ8_0: bb = 34; be = 32; break;
        case kGF16: case kGBF16: bb = 2; be = 1; break;
        default: return LMX_E_UNSUPPORTED;
    }
    if (d->in_dim % (be == 1 ? 64 : 128) || d->in_dim % be) return LMX_E_SHAPE;
    GemmArgs a{};
    a.w = static_cast<const uint8_t*>(w);
    a.x = x;
    a.y = y;
    a.rows = (int)d->rows;
    a.in_dim = (int)d->in_dim;
    a.n_tok = (int)d->n_tok;
    a.row_bytes = (size_t)d->in_dim / be * bb;
    a.w_bytes = a.row_bytes * d->rows;
    if (((long)d->n_tok + 31) / 32 * (((long)d->rows + 31) / 32) > INT32_MAX) return LMX_E_SHAPE;
    const int tn = be > 1 && d->n_tok > 32 ? tile_rows(a, d->type) : 32;
    if (tn == 128) return qgemm_big(d, w, x, y, st);
    (void)hipGetLastError();
    switch (d->type) {
        case kGF16: launch_type<kGF16>(a, tn, st); break;
        case kGBF16: launch_type<kGBF16>(a, tn, st); break;
        case kGQ4K: launch_type<kGQ4K>(a, tn, st); break;
        case kGQ6K: launch_type<kGQ6K>(a, tn, st); break;
        default: launch_type<kGQ8_0>(a, tn, st); break;
    }
    LMX_CHECK_LAUNCH();
    return LMX_OK;
}

}  // namespace lmx
