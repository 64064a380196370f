// Tiled attention for long batches at head_dim 256 and 512 on gfx950 MFMA.
//
// The same products as attn_prefill_kernel (S^T = K Q^T, O^T += V^T P^T on
// v_mfma_f32_32x32x16_f16, online softmax in fp32 with a lazy rescale, P in
// f16), shared out differently, because at these head sizes one wave cannot
// hold a query block's Q and output and still leave a second wave room on its
// SIMD.  A workgroup is eight waves, two per SIMD; WPR = head_dim / 128 of
// them share a block of 32 query rows:
//
//   scores   wave (kb, dq) forms S^T of 32 of the tile's 64 keys (block kb)
//            over 256 of the head's dims (part dq, of one or two); at
//            head_dim 512 the two parts trade halves of their partial scores
//            through LDS, so each finishes 16 keys
//   softmax  each wave exponentiates only the scores it finished and leaves
//            its P as MFMA operand fragments in LDS
//   output   every wave multiplies all 64 keys' P by its own 128 dims of V
//
// So a wave holds 64 registers of output and 64 of Q (128 with an fp32
// query's f16 residual) at both head sizes.  A workgroup's rows are (token,
// head) pairs of gp heads that share a kv head, tokens outermost: 16 heads
// make 64 rows out of 4 tokens, whose causal ranges nearly coincide.
//
// K and V tiles go from memory straight to LDS (no registers), key-major,
// their 16-byte chunks XOR-swizzled by row so that both the score operand
// reads (32 rows of one chunk) and the transposing V reads
// (ds_read_b64_tr_b16, 4 rows of 64 bytes per half wave) spread over all
// banks.  At head_dim 256 two stages of each fit the LDS; at 512 one, K being
// refilled once the scores are done and V once the output step is.  Q comes
// in and the output leaves through the same LDS in whole rows: as MFMA
// operands a load or store instruction touches 16 bytes of each of 32 rows,
// and the address unit takes 64 cycles for it instead of 16 (8 us a workgroup
// for an fp32 query, 4 us for its output).
//
// Measured against the one-wave-per-SIMD kernel this replaces (fp32 / f16
// queries, us a call): head_dim 512, 16 heads on one kv head, 2048 tokens
// 979 / 391 -> 149 / 124; 4096 tokens 3792 / 1482 -> 520 / 430 (531 / 640
// TFLOP/s); head_dim 256, 16 heads on 8, window 1024, 1999 tokens at 3001
// 92 / 79 -> 78 / 60; 4096 tokens, no window 305 / 228 -> 235 / 186.  What
// bounds it: with the transfers skipped a head_dim 512 call takes two thirds
// of the time, without the MFMAs as long; the transfers move 10.5 TB/s of tiles
// over all CUs (head_dim 512, 4096 f16-query tokens: 33 thousand of 128 KB in
// 404 us), and overlap little of the scores and softmax.  Tried
// and no faster: the two waves of a SIMD half a tile apart (ping-pong; at 512
// it halves the tile and lost 25%), transfers dealt out between the MFMAs.
#include <climits>

#include "attn_prefill.hpp"
#include "lds_dma.hpp"

namespace lmx {

// LIN: key row p lives at cache row p (see attn_prefill_kernel).
// FEW: the workgroup's rows are at most few_rows(HD), one row block.  Q then
// leaves the first tile's LDS free, whose transfers go out with Q's instead of
// after it, and the other row blocks' waves only move data.  us a call of 9
// tokens, head_dim 256, 16 heads on 8, position 0, the kernel this file
// replaces / not FEW / FEW: fp32 queries 11.0 / 14.1 / 10.8, f16 8.5 / 10.6 /
// 8.3; head_dim 512, f16 9.7 / 10.8 / 8.3.
template <int HD>
constexpr int few_rows() { return HD == 256 ? 32 : 16; }
template <typename QT, int HD, bool LIN, bool FEW>
__global__ __launch_bounds__(512, 1) void attn_prefill_wide_kernel(PrefillArgs a) {
    static_assert(HD == 256 || HD == 512, "two or four waves a row block");
    constexpr bool kQlo = sizeof(QT) == 4;  // fp32 queries carry an f16 residual (qk_tile)
    constexpr bool kTight = kQlo;      // Q and its residual leave few registers for operand reads
    constexpr int BN = 64;             // keys per tile
    constexpr int WPR = HD / 128;      // waves per row block
    constexpr int RB = 8 / WPR;        // 32-row blocks
    constexpr int BM = 32 * RB;        // rows per workgroup
    constexpr int DS = WPR / 2;        // parts the scores' dims are split into
    constexpr int QD = HD / DS;        // dims of a part
    constexpr int KSTEPS = QD / 16;
    constexpr int NS = 16 / DS;        // scores a lane finishes
    constexpr int PS = 2 / DS;         // 16-key P fragments they make
    constexpr int STG = DS == 1 ? 2 : 1;
    constexpr int ROWB = HD * 2;       // bytes of a tile row
    constexpr int NDMA = BN * ROWB / 1024 / 8;  // transfers a wave issues per tile
    // K stages, then V stages; Q before the key loop (fp32: all of it, f16:
    // the V half) and the output after it
    constexpr int TILE = BN * HD;
    __shared__ __attribute__((aligned(1024))) f16 KV_s[2 * STG * TILE];
    auto K_st = [&](int st) { return &KV_s[st * TILE]; };
    auto V_st = [&](int st) { return &KV_s[(STG + st) * TILE]; };
    __shared__ __attribute__((aligned(16))) f16 P_s[RB * 4 * 64 * 8];  // [row block][k-step][lane][8]
    __shared__ __attribute__((aligned(16))) float X_s[DS == 2 ? 8 * 2 * 64 * 4 : 4];  // traded partial scores
    __shared__ __attribute__((aligned(16))) float M_s[8][32];  // per wave and row: a max, then the row sums
    __shared__ __attribute__((aligned(16))) int F_s[8];        // a wave asks for the exact path

    // ---- which kv head, heads, query tile and key split.  XCD x = b % 8 takes
    // whole kv heads when they divide evenly over the XCDs, else XCDs share
    // one and deal its tiles out in turn, so that each gets heavy and light
    // ones; surplus workgroups of the rounded grid leave at once.
    const int gp = a.gp, hgroups = a.G / gp, n_split = a.n_split;
    const int per_kvh = a.n_qtiles * hgroups * n_split;
    const int b = blockIdx.x;
    int kvh, idx;
    if (a.Hkv % 8 == 0) {
        kvh = (b % 8) * (a.Hkv / 8) + b / 8 / per_kvh;
        idx = b / 8 % per_kvh;
    } else if (8 % a.Hkv == 0) {
        const int share = 8 / a.Hkv;
        kvh = b % 8 / share;
        idx = b / 8 * share + b % 8 % share;
        if (idx >= per_kvh) return;
    } else {
        kvh = b % a.Hkv;
        idx = b / a.Hkv;
    }
    // (scalar: the divisions run on the vector unit, and what is derived from
    // their results there would stay there, the transfers' row pointers too)
    auto scalar = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    kvh = scalar(kvh);
    const int qt = scalar(a.n_qtiles - 1 - idx / (hgroups * n_split));  // heaviest first
    const int sp = scalar(idx % n_split), hg = scalar(idx / n_split % hgroups);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hh = lane >> 5;
    const int rb = wave / WPR, j4 = wave % WPR;  // row block; 128-dim part of the output
    const int kb = j4 & 1, dq = j4 >> 1;         // score block and dim part
    const int t = a.n_tokens, base = a.base_pos, w = a.window;
    const int end = base + t - 1;
    const int tpw = scalar((FEW ? few_rows<HD>() : BM) / gp), tpb = scalar(32 / gp);  // tokens of the workgroup, of a row block
    const int q0 = qt * tpw, qb0 = q0 + rb * tpb;

    // ---- this lane's row: token qb0 + l32 / gp, head l32 % gp of the group.
    // Rows past the batch repeat its last token and are not stored.
    const int tok = qb0 + l32 / gp;
    const bool qvalid = tok < t;
    const int qrow = qvalid ? tok : t - 1;
    const int h = kvh * a.G + hg * gp + l32 % gp;
    const int my_lo = vis_lo(base + qrow, w), my_hi = vis_hi(base + qrow, w, a.bidi, end);

    // ---- key ranges: the workgroup's (a row block does all of its tiles, masked
    // where it has no keys: its waves would wait for the others' at the barriers)
    const int wg_lo = vis_lo(base + q0, w);
    const int wg_hi = vis_hi(base + min(q0 + tpw, t) - 1, w, a.bidi, end);
    // keys every query of the row block sees
    const int bk_lo_max = vis_lo(base + min(qb0 + tpb, t) - 1, w);
    const int bk_hi_min = vis_hi(base + min(qb0, t - 1), w, a.bidi, end);

    const int cur_begin = (!LIN && a.k_cur) ? base : INT_MAX;
    const int kvb = a.kv_dim * 2;
    // The row of position p (uniform).
    auto row_of = [&](const f16* cache, const f16* cur, int p) -> const char* {
        const char* src = reinterpret_cast<const char*>(cache);
        if constexpr (!LIN) {
            if (p >= cur_begin) {
                src = reinterpret_cast<const char*>(cur);
                p -= base;
            } else if (w) {
                p = ring_slot(p, w, a.w_magic, a.w_shift);
            }
        }
        return src + (size_t)p * kvb + kvh * ROWB;
    };
    // A tile's rows to LDS: row r at r * ROWB, its chunk c at position
    // c ^ swz(r): for K r & 15 (32 rows of one chunk meet all banks), for V
    // (r & 3) * 4 (the 64-byte pieces of 4 rows do).  Rows outside the
    // workgroup's range, which are masked for every query, repeat its first
    // or last row: the reads stay inside the caches.
    auto fetch = [&](const f16* cache, const f16* cur, int kt, const f16* dst, bool is_v) {
        const uint32_t lds = lds_addr(dst) + wave * (NDMA * 1024);
        // the lane's chunk offset before the transfer's own swizzle bits
        uint32_t c16 = (HD == 512 ? lane : l32 ^ (is_v ? hh << 2 : hh)) << 4;
        opaque(c16);
        auto swz = [&](int r0) { return (uint32_t)((is_v ? (r0 & 3) << 2 : r0 & 15) << 4); };
        const int row0 = wave * (BN / 8);
        bool plain = kt >= wg_lo && kt + BN - 1 <= wg_hi;  // whole and side by side in one buffer
        if constexpr (!LIN)
            plain = plain && (kt >= cur_begin || (kt + BN <= cur_begin &&
                                                  (!w || ring_slot(kt, w, a.w_magic, a.w_shift) + BN <= w)));
        if (plain) {
            const char* src = uniform_ptr(row_of(cache, cur, kt) + (size_t)row0 * kvb);
            const uint32_t second = HD == 256 && hh ? kvb : 0;  // two rows a transfer
#pragma unroll
            for (int i = 0; i < NDMA; ++i) {
                dma16(src, (c16 ^ swz(row0 + (HD == 512 ? i : 2 * i))) + second, lds + i * 1024);
                src += HD == 512 ? kvb : 2 * kvb;
            }
        } else {
#pragma unroll 1
            for (int i = 0; i < NDMA; ++i) {
                const int r0 = row0 + (HD == 512 ? i : 2 * i);
#pragma unroll
                for (int u = 0; u < (HD == 512 ? 1 : 2); ++u) {
                    const char* row = row_of(cache, cur, max(wg_lo, min(wg_hi, kt + r0 + u)));
                    if (HD == 512 || hh == u) dma16(row, c16 ^ swz(r0), lds + i * 1024);
                }
            }
        }
    };

    float m_run = -1e30f, l_run = 0.f;
    f32x16 o[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[nb][i] = 0.f;

    // ---- operand addresses (halfs) at k-step / block 0; a swizzled step is an
    // XOR of bits the rest leaves clear.  Score rows: key 32 kb + l32 (part 1
    // of head_dim 512 swaps the block's 16-key halves), chunk 2 ks + hh of
    // the part; V: lane (i = lane & 15) addresses key
    // 16 ks + 4 hh + i / 4, dims 16 (lane >> 4 & 1) + 4 (i & 3) of a 32-dim
    // block nb, and receives dim 16 (..) + i of those four keys.
    const int k_at0 = (kb * 32 + (l32 ^ (16 * dq))) * HD + dq * QD + ((hh ^ (l32 & 15)) << 3);
    const int v_key = 4 * hh + ((lane >> 2) & 3);
    const int v_at0 = v_key * HD + j4 * 128 + ((v_key & 3) << 5) + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;

    // This workgroup's split: chunk sp of the tiles covering [wg_lo, wg_hi].
    const int kt_all = wg_lo / BN * BN;
    const int n_t_all = (wg_hi - kt_all) / BN + 1;
    const int cs = scalar((n_t_all + n_split - 1) / n_split);
    const int kt_begin = kt_all + sp * cs * BN;
    const int n_t = max(0, min(cs, n_t_all - sp * cs));
    // ---- Q as the B operand (lane: 8 dims 16 ks + 8 hh of its row), out of
    // LDS; an fp32 query as hi and residual, scaled per row as in
    // attn_prefill_kernel (at head_dim 512 per part: each scales its own sums
    // back)
    const int gp_shift = __builtin_ctz(gp);
    constexpr int ROWQ = HD * (int)sizeof(QT);
    const int nq = FEW ? scalar(min(tpw, t - q0) * gp) : BM;  // rows
    f16* Q_s = kQlo ? K_st(0) : V_st(0);
    if constexpr (FEW) {  // beside the first tile: the second stage of V, or X_s
        static_assert(HD == 256 || !kQlo, "16 rows of f16 fill X_s");
        Q_s = HD == 256 ? V_st(1) : reinterpret_cast<f16*>(X_s);
        static_assert(few_rows<HD>() * ROWQ <= (HD == 256 ? TILE * 2 : (int)sizeof(X_s)), "Q's rows fit there");
    } else if (!kQlo && n_t > 0) {
        fetch(a.k, a.k_cur, kt_begin, K_st(0), false);
    }
    constexpr int NQ = BM * ROWQ / 1024 / 8;  // transfers a wave issues for BM rows
#pragma unroll 4
    for (int i = 0; i < (FEW ? (nq * ROWQ + 1023) / 1024 - wave : 8 * NQ); i += 8) {
        const int n = FEW ? wave + i : wave * NQ + i / 8;
        const int at = n * 1024 + lane * 16, r = at / ROWQ, c = at % ROWQ / 16;
        const int qt_r = min(q0 + (r >> gp_shift), t - 1), h_r = kvh * a.G + hg * gp + (r & (gp - 1));
        dma16_lane(reinterpret_cast<const char*>(a.q) + ((size_t)qt_r * a.H + h_r) * a.q_stride * sizeof(QT) +
                       ((c ^ (r & 15)) << 4),
                   lds_addr(Q_s) + n * 1024);
    }
    if (FEW && n_t > 0) {
        fetch(a.k, a.k_cur, kt_begin, K_st(0), false);
        fetch(a.v, a.v_cur, kt_begin, V_st(0), true);
        wait_dma<2 * NDMA>();  // Q: the tile took that many transfers or more
    } else {
        wait_dma<0>();
    }
    __syncthreads();
    f16x8 qf[KSTEPS], ql[kQlo ? KSTEPS : 1];
    float c_sc = a.c;
    {
        // (FEW: rows past the batch, and the idle waves', read its last token's)
        const int r = FEW && rb * 32 + l32 >= nq ? nq - gp + l32 % gp : rb * 32 + l32;
        const char* qrow_s = reinterpret_cast<const char*>(Q_s) + r * ROWQ;
        auto chunk = [&](int c) { return qrow_s + ((c ^ (r & 15)) << 4); };
        if constexpr (!kQlo) {
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks)
                qf[ks] = *reinterpret_cast<const f16x8*>(chunk(dq * (QD / 8) + 2 * ks + hh));
        } else {
            f32x4 x[2 * KSTEPS];
#pragma unroll
            for (int i = 0; i < 2 * KSTEPS; ++i)
                x[i] = *reinterpret_cast<const f32x4*>(chunk(dq * (QD / 4) + 4 * (i / 2) + 2 * hh + i % 2));
            float m = 0.f;
#pragma unroll
            for (int i = 0; i < 2 * KSTEPS; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) m = fmaxf(m, fabsf(x[i][j]));
            m = fmaxf(m, shfl_xor(m, 32)) * fabsf(a.c);
            const int S = (m > 0.f && m <= 3.402823466e38f) ? 15 - __builtin_amdgcn_frexp_expf(m) : 0;
            const float qc = a.c * __builtin_amdgcn_ldexpf(1.f, S);
            c_sc = __builtin_amdgcn_ldexpf(1.f, -S);
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) {
                float y[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    // one rounding of x c 2^S, seen by hi and residual alike
                    y[j] = x[2 * ks + j / 4][j % 4] * qc;
                    asm volatile("" : "+v"(y[j]));
                    qf[ks][j] = (f16)y[j];
                }
                asm volatile("" : "+v"(qf[ks]));
#pragma unroll
                for (int j = 0; j < 8; ++j) ql[ks][j] = (f16)(y[j] - (float)qf[ks][j]);
            }
            settle_q(ql);
        }
        settle_q(qf);
    }
    if constexpr (!FEW) __syncthreads();  // Q is in registers: its LDS is the tiles'
    if (!FEW && n_t > 0) {
        if (kQlo) fetch(a.k, a.k_cur, kt_begin, K_st(0), false);
        fetch(a.v, a.v_cur, kt_begin, V_st(0), true);
    }

    const bool act = !FEW || rb == 0;
    for (int it = 0; it < n_t; ++it) {
        const int kt = kt_begin + it * BN;
        const int stage = STG == 2 ? it & 1 : 0;
        const bool more = it + 1 < n_t;
        wait_dma<0>();    // this tile (one stage: its K; V follows below)
        __syncthreads();  // and every wave is done with the tile before
        if constexpr (STG == 2) {
            if (more) {
                fetch(a.k, a.k_cur, kt + BN, K_st(stage ^ 1), false);
                fetch(a.v, a.v_cur, kt + BN, V_st(stage ^ 1), true);
            }
        } else if (it > 0) {
            fetch(a.v, a.v_cur, kt, V_st(0), true);
        }

        // ---- scores, minus mb once scaled
        float mb = m_run > -1e29f ? m_run : 0.f;
        float sv[NS];
        {
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.f;
            const f16* Ks = K_st(stage);
            if (act) {
                constexpr int D = kTight ? 3 : 4;  // operand reads ahead
                int k_tile = k_at0;
                opaque(k_tile);
                auto rd = [&](int ks) {
                    int k_at = k_tile;
                    if (kTight) opaque(k_at);
                    return *reinterpret_cast<const f16x8*>(&Ks[(k_at ^ ((ks & 7) << 4)) + (ks >> 3) * 128]);
                };
                f16x8 ka[KSTEPS];
#pragma unroll
                for (int ks = 0; ks < D; ++ks) ka[ks] = rd(ks);
                __builtin_amdgcn_sched_group_barrier(0x100, D, 0);
#pragma unroll
                for (int ks = 0; ks < KSTEPS; ++ks) {
                    if (ks + D < KSTEPS) ka[ks + D] = rd(ks + D);
                    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[ks], qf[ks], s, 0, 0, 0);
                    if constexpr (kQlo) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[ks], ql[ks], s, 0, 0, 0);
                    if (ks + D < KSTEPS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, kQlo ? 2 : 1, 0);
                }
            }
            if constexpr (DS == 2) {
                // each part finishes the 16 keys in its registers 0-7 and
                // hands over registers 8-15, which the other finishes
#pragma unroll
                for (int g = 0; g < 2 && act; ++g) {
                    f32x4 x;
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = s[8 + 4 * g + i] * c_sc;
                    *reinterpret_cast<f32x4*>(&X_s[((wave * 2 + g) * 64 + lane) * 4]) = x;
                }
                __syncthreads();  // K is free
                if (more) fetch(a.k, a.k_cur, kt + BN, K_st(0), false);
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const f32x4 x = *reinterpret_cast<const f32x4*>(&X_s[(((wave ^ 2) * 2 + g) * 64 + lane) * 4]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) sv[4 * g + i] = fmaf(s[4 * g + i], c_sc, x[i]) - mb;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) sv[i] = fmaf(s[i], c_sc, -mb);
            }
        }
        // sv[i] is key kt + 32 kb + 16 dq + 8 (i / 4) + 4 hh + i % 4
        if (!(kt >= bk_lo_max && kt + BN - 1 <= bk_hi_min)) {
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const int key = kt + 32 * kb + 16 * dq + 8 * (i / 4) + 4 * hh + i % 4;
                if (key < my_lo || key > my_hi) sv[i] = -INFINITY;
            }
        }

        // ---- softmax with a lazy rescale, as in attn_prefill_kernel; the
        // test is the workgroup's, since the row block's waves rescale together
        constexpr float kSlackP = 256.f;  // 2^kRescaleSlack
        static_assert(kRescaleSlack == 8.f, "kSlackP is 2^kRescaleSlack");
        f16x8 pf[PS];
        auto make_p = [&]() {
#pragma unroll
            for (int st = 0; st < PS; ++st) {
#pragma unroll
                for (int j = 0; j < 8; ++j) pf[st][j] = (f16)fast_exp2(sv[8 * st + j]);
                // k-step 2 kb + dq + st of the tile
                *reinterpret_cast<f16x8*>(&P_s[((rb * 4 + 2 * kb + dq + st) * 64 + lane) * 8]) = pf[st];
            }
        };
        bool ask = false;
        if (act) {
            make_p();
            f16x2 pm = {pf[0][0], pf[0][1]};
#pragma unroll
            for (int st = 0; st < PS; ++st)
#pragma unroll
                for (int j = 0; j < 8; j += 2) pm = __builtin_elementwise_max(pm, f16x2{pf[st][j], pf[st][j + 1]});
            const float pmax = fmaxf((float)pm[0], (float)pm[1]);
            ask = !(pmax <= kSlackP);
            if (__builtin_amdgcn_ballot_w64(m_run < -1e29f) != 0) {  // a row's first keys set its max
                float mt = sv[0];
#pragma unroll
                for (int i = 1; i < NS; ++i) mt = fmaxf(mt, sv[i]);
                ask = ask || (m_run < -1e29f && mt > -INFINITY);
            }
        }
        const int asks = __builtin_amdgcn_ballot_w64(ask) != 0;
        if (lane == 0) F_s[wave] = asks;
        if constexpr (STG == 1) {
            // V of this tile; K of the next may still be in flight
            if (more) wait_dma<NDMA>();
            else wait_dma<0>();
        }
        __syncthreads();  // P and V are there
        const int4 f0 = *reinterpret_cast<const int4*>(&F_s[0]), f1 = *reinterpret_cast<const int4*>(&F_s[4]);
        const int any = f0.x | f0.y | f0.z | f0.w | f1.x | f1.y | f1.z | f1.w;
        if (__builtin_amdgcn_readfirstlane(any)) {
            float mt = sv[0];
#pragma unroll
            for (int i = 1; i < NS; ++i) mt = fmaxf(mt, sv[i]);
            mt = fmaxf(mt, shfl_xor(mt, 32)) + mb;
            if (hh == 0) M_s[wave][l32] = mt;
            __syncthreads();
            float mn = m_run;
#pragma unroll
            for (int i = 0; i < WPR; ++i) mn = fmaxf(mn, M_s[rb * WPR + i][l32]);
            const float corr = fast_exp2(m_run - mn);
            m_run = mn;
            l_run *= corr;
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[nb][i] *= corr;
            const float shift = (mn > -1e29f ? mn : 0.f) - mb;
#pragma unroll
            for (int i = 0; i < NS; ++i) sv[i] -= shift;
            if (act) make_p();
            __syncthreads();
        }
        if (!act) continue;
        const f16x2 one2 = {(f16)1.f, (f16)1.f};
#pragma unroll
        for (int st = 0; st < PS; ++st)
#pragma unroll
            for (int j = 0; j < 8; j += 2)
                l_run = __builtin_amdgcn_fdot2(f16x2{pf[st][j], pf[st][j + 1]}, one2, l_run, false);

        // ---- O^T += V^T P^T over the tile's four k-steps, dims 128 j4 ..
        const f16* Vs = V_st(stage);
        typedef __fp16 tr_h4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
        typedef __attribute__((address_space(3))) tr_h4 lds_h4;
        auto rdp = [&](int ks) { return *reinterpret_cast<const f16x8*>(&P_s[((rb * 4 + ks) * 64 + lane) * 8]); };
        int v_tile = v_at0;
        opaque(v_tile);
        auto rdv = [&](int q) {
            int v_at = v_tile;
            if (kTight) opaque(v_at);
            const int ks = q >> 2, nb = q & 3;
            const f16* p = &Vs[(v_at ^ (nb << 5)) + ks * 16 * HD];
            const f16x4 v0 = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)p));
            const f16x4 v1 = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)(p + 8 * HD)));
            return f16x8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        };
        constexpr int PD = kTight ? 2 : 3;  // operands ahead
        f16x8 va[16], pb[4];
        pb[0] = rdp(0);
#pragma unroll
        for (int q = 0; q < PD; ++q) va[q] = rdv(q);
        __builtin_amdgcn_sched_group_barrier(0x100, 1 + 2 * PD, 0);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            if (q + PD < 16) va[q + PD] = rdv(q + PD);
            if (q % 4 == 1 && q / 4 + 1 < 4) pb[q / 4 + 1] = rdp(q / 4 + 1);
            o[q & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[q], pb[q >> 2], o[q & 3], 0, 0, 0);
            if (q + PD < 16) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            if (q % 4 == 1 && q / 4 + 1 < 4) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
    }

    // ---- row sums over the row block's waves, then normalize (a split's
    // partial stays as accumulated) and store: o[nb][i] is dim
    // 128 j4 + 32 nb + 8 (i / 4) + 4 hh + i % 4 of row 32 rb + l32
    const float l_own = l_run + shfl_xor(l_run, 32);
    __syncthreads();  // the last tile and exact path's maxima are read
    if (hh == 0) M_s[wave][l32] = l_own;
    __syncthreads();
    float l_tot = 0.f;
#pragma unroll
    for (int i = 0; i < WPR; ++i) l_tot += M_s[rb * WPR + i][l32];
    const bool part = n_split > 1;
    if (part && act && qvalid && hh == 0 && j4 == 0)
        *reinterpret_cast<f32x2*>(a.part_ml + 2 * (((size_t)sp * t + qrow) * a.H + h)) = f32x2{m_run, l_tot};
    const float inv = part ? 1.f : 1.f / l_tot;
    char* O_s = reinterpret_cast<char*>(KV_s);
    constexpr int ROWO = HD * 4;
    static_assert(BM * ROWO <= (int)sizeof(KV_s), "output rows fit the tiles' LDS");
    {
        const int r = rb * 32 + l32;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = 32 * j4 + 8 * nb + 2 * g + hh;
                *reinterpret_cast<f32x4*>(O_s + r * ROWO + ((c ^ (r & 15)) << 4)) =
                    f32x4{o[nb][4 * g] * inv, o[nb][4 * g + 1] * inv, o[nb][4 * g + 2] * inv, o[nb][4 * g + 3] * inv};
            }
    }
    __syncthreads();
    float* dst = part ? a.part_o + (size_t)sp * t * a.H * HD : a.out;
    constexpr int NO = BM * ROWO / 1024 / 8;
#pragma unroll 4
    for (int i = 0; i < (FEW ? nq * ROWO / 1024 - wave : 8 * NO); i += 8) {
        const int at = (FEW ? wave + i : wave * NO + i / 8) * 1024 + lane * 16;
        const int r = at / ROWO, c = at % ROWO / 16;
        const int row_t = q0 + (r >> gp_shift), row_h = kvh * a.G + hg * gp + (r & (gp - 1));
        f32x4 y = *reinterpret_cast<const f32x4*>(O_s + r * ROWO + ((c ^ (r & 15)) << 4));
        if (row_t >= t) continue;
        const size_t row = (size_t)row_t * a.H + row_h;
        if (a.gate && !part) y = gate_sigmoid4(y, a.gate + row * a.gate_stride + 4 * c);
        *reinterpret_cast<f32x4*>(dst + row * HD + 4 * c) = y;
    }
}

// Heads that share a workgroup's rows, its tokens, and which form it takes.
// The heads: the largest power of two that divides the kv group, up to the 32
// rows of a block.  A short call over few keys takes the FEW form with as few
// heads as make one workgroup of its tokens, as long as the CUs hold all
// workgroups at once.  The lines (us a call, not FEW / FEW): 64 heads on 8,
// head_dim 256, f16, 32 tokens at position 900 25.4 / 21.5, at 16000 62 / 101;
// 128 heads, 80 tokens at 900 38 / 58; head_dim 512, f16, 48 heads on 3, 17
// tokens at 300 21.4 / 17.1, at 900 25.6 / 27.3; 64 heads on 8, 48 tokens at 900
// 32 / 37.
WidePlan prefill_wide_plan(const lmx_attn_params* p, lmx_dtype q_dt) {
    const int hd = (int)p->head_dim, t = (int)p->n_tokens, H = (int)p->n_heads, G = H / (int)p->n_kv_heads;
    const int few = hd == 256 ? few_rows<256>() : q_dt == LMX_F16 ? few_rows<512>() : 0;
    const int most = hd == 512 ? 32 : q_dt == LMX_F16 ? 96 : 64, keys = hd == 512 ? 512 : 1024;
    bool small = few && t <= most && decode_max_vis(p) <= keys;
    int few_gp = 1, gp = 1;
    while (2 * few_gp * t <= few && G % (2 * few_gp) == 0) few_gp *= 2;
    while (gp < 32 && G % (2 * gp) == 0) gp *= 2;
    small = small && (t * few_gp + few - 1) / few * (H / few_gp) < 256;
    if (small) gp = few_gp;
    if (const int v = tuning().prefill_gp; v > 0 && G % v == 0) gp = v;
    if (few && (gp * t <= few || (small && gp <= few))) return {gp, few / gp, true};
    return {gp, (hd == 512 ? 64 : 128) / gp, false};
}

// a: as prefill_fwd fills it, with gp, n_qtiles and n_split for this kernel.
lmx_status prefill_wide(const PrefillArgs& a, int hd, lmx_dtype q_dt, bool lin, bool few, hipStream_t st) {
    const long per_kvh = (long)a.n_qtiles * (a.G / a.gp) * a.n_split;
    long nblk = per_kvh * a.Hkv;
    if (a.Hkv % 8 && 8 % a.Hkv == 0) {
        const long share = 8 / a.Hkv;
        nblk = (per_kvh + share - 1) / share * 8;
    }
    if (nblk > INT_MAX) return LMX_E_SHAPE;
    const dim3 grid((unsigned)nblk);
#define LMX_WDL(QT, HDV, FEW)                                                                                   \
    do {                                                                                                        \
        if (lin) hipLaunchKernelGGL((attn_prefill_wide_kernel<QT, HDV, true, FEW>), grid, dim3(512), 0, st, a); \
        else hipLaunchKernelGGL((attn_prefill_wide_kernel<QT, HDV, false, FEW>), grid, dim3(512), 0, st, a);    \
    } while (0)
#define LMX_WD(QT, HDV)                    \
    do {                                   \
        if (few) LMX_WDL(QT, HDV, true);   \
        else LMX_WDL(QT, HDV, false);      \
    } while (0)
    if (q_dt == LMX_F16) {
        if (hd == 256) LMX_WD(f16, 256);
        else LMX_WD(f16, 512);
    } else {
        if (hd == 256) LMX_WD(float, 256);
        else LMX_WDL(float, 512, false);
    }
#undef LMX_WD
#undef LMX_WDL
    return LMX_OK;
}

}  // namespace lmx
