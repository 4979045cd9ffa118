// Time attention for gfx950, bf16 / fp16, 64-wide heads: the ring kernel of Timestral's rows and of the
// Chronos-2 rows that no persistent kernel takes.
//
// Same contracts as time_attention_lp.hip (Chronos-2's Chronos2Kernels.rope + timeAttention,
// Chronos2Kernels.java:87-116, 118-464; Timestral's TimestralKernels.rope + timeAttention + gate,
// TimestralKernels.java:71-100, 102-278, 572-578; oracles CpuChronos2.java:175-228, 284-304 and
// CpuTimestral.java:156-161, 190-259): the rotation by each token's own table row, in fp32, rounded to the
// storage type; fp32 scores, softmax and sums.
//
// Work split: a workgroup of NW waves covers 32 * NW consecutive queries of one (row, head), and NW
// (4 .. 8) is the row's, chosen so that its 32-query tiles fill the workgroups (time_attention_lpr_launch). The
// 64-key blocks some query of the workgroup sees stream through a ring of three LDS slots: one computed, one
// rotated, one arriving by direct-to-LDS loads. A block is eight units of 8 keys. A unit's loads, its
// table rows and its rotation in place belong to one wave, so a block needs one barrier, and all loads of a wave have a
// block's compute to arrive in. V is never touched by VALU code: the PV operand V^T is read with
// ds_read_b64_tr_b16. Rows past the row's last key are zeroed where the rotation passes them.
//
// The softmax is time_attention_lp.hip's on 32-key halves: the key mask and the running max ride in an extra
// MFMA step, P = exp2(S) rounded to T, v_dot2 row sums, and a wave-uniform slow path for stale maxima. The mask of a
// block that every query of a wave sees alike (below the causal diagonal; all of Chronos-2's) is one scalar word.
//
// What bounds it: the latency of a block's step (4 waves per SIMD; at Timestral's 64 x 1,025 tokens, gate on, VALU 43% and
// MFMA 18% of the cycles, LDS 21%). There 0.298 ms, 0.408 on the streaming kernel, whose workgroups of 128 queries staged
// every block through registers (fp16 0.300 against 0.463); with its last part of one query as any other part 0.323.
// Chronos-2: 90 x 197 0.039 (0.056), 383 x 245 0.170 (0.258), 64 x 577 0.128 (0.158 on the row-wide kernel).
// 5 .. 7 waves ran slower than 8 with idle ones (units of 8 keys then fall unevenly: 64 x
// 1,025 on 7 waves 0.389); requesting the first blocks ahead of the validity scan cost short rows 8%.
#include "jc_common.hpp"
#include "jc_kernels.hpp"
#include "lp_common.hpp"
#include "lp_stream.hpp"
#include "time_mask.hpp"

namespace jc {
namespace {

using namespace lp;

constexpr int kDH = 64;
constexpr int kQ = 32;     // queries per wave
constexpr int kKB = 64;    // keys per block
constexpr int kHalf = 32;  // keys per softmax step
constexpr int kUnits = 8;  // units of 8 keys per block
constexpr int kSlots = 3;
constexpr int kMaxTokens = 4096;
constexpr int kHand = 35 * kWave;  // floats a wave of a split tile hands over: O^T, its reference, its sum, whether it has any

struct alignas(16) RingLds {
    uint16_t kv[kSlots][2][kKB * kDH];  // [slot][K | V][swz(key, chunk)]
    uint64_t mask[kMaxTokens / kKB];    // per 64-key block: key validity bits
};

// 16 bytes per lane from base + off to lds_base + 16 * lane (M0 holds the wave-uniform LDS address)
__device__ __forceinline__ void dma16s(const void* base, uint32_t off, const void* lds_base) {
    const uint32_t m0 = (uint32_t)(size_t)(__attribute__((address_space(3))) const void*)lds_base;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(m0) : "memory", "m0");
}

template <typename T, int NW, bool ROPE, bool TS>
__global__ __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(4))) void time_attention_lpr(const TimeArgs a) {
    static_assert(kUnits % NW == 0, "every wave has as many units");
    constexpr int kU = kUnits / NW;  // units per wave
    typedef typename Lp<T>::x8 x8;
    typedef Enc<T> E;
    __shared__ RingLds lds;

    const T* __restrict__ qkv = static_cast<const T*>(a.qkv);
    const int n = a.n, inner = a.inner;
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane % 32, g = lane / 32;
    const uint32_t logical = xcd_remap(blockIdx.x, (uint32_t)a.rows * a.heads * a.qgroups);
    // a (row, head)'s last queries first: under a causal mask theirs is the longest stream
    const int part = a.qgroups - 1 - (int)(logical % a.qgroups);
    const uint32_t bh = logical / a.qgroups;
    const int h = bh % a.heads, r = bh / a.heads;
    TimeMask<TS> mask;
    mask.init(a, r);
    const int32_t* vrow = a.valid + (size_t)r * (TS ? a.enc : n);
    const size_t row0 = (size_t)r * n;
    const uint32_t stride = 3u * inner * 2u;  // bytes per token of qkv
    auto table_row = [&](int t) __attribute__((always_inline)) {
        return TS && a.pos ? min(max(a.pos[row0 + t], 0), a.table_rows - 1) : t;
    };

    // the wave's queries: lane (j, g) holds dims 16s + 8g .. of query q0 + j, so a RoPE pair sits in steps s, s + 2
    const bool lone = NW == 8 && n - part * NW * kQ <= kQ;  // a part of one tile
    const int q0 = (part * NW + (lone ? 0 : wave)) * kQ;
    const int nq = min(max(n - q0, 0), kQ);
    const int q = min(q0 + j, n - 1);
    u32x4 qraw[4];
    {
        const T* qp = qkv + (row0 + q) * 3 * inner + h * kDH + 8 * g;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            qraw[s] = *reinterpret_cast<const u32x4*>(qp + 16 * s);
            if (j >= nq) qraw[s] = u32x4{0u, 0u, 0u, 0u};
        }
    }
    floatx4 qc[2][2], qs[2][2];
    if (ROPE) {
        const float* tp = a.table + (size_t)table_row(q) * kDH + 8 * g;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                qc[s][u] = *reinterpret_cast<const floatx4*>(tp + 16 * s + 4 * u);
                qs[s][u] = *reinterpret_cast<const floatx4*>(tp + 16 * s + 4 * u + kDH / 2);
            }
    }

    const int nblk = (n + kKB - 1) / kKB;

    // ---- the stream -------------------------------------------------------------------------
    const char* kbase = reinterpret_cast<const char*>(qkv + row0 * 3 * inner + inner + h * kDH);
    const char* vbase = kbase + 2 * (size_t)inner;
    const int lkey = lane / 8;                       // the lane's key of a unit
    const int lcp = (lane % 8) / 2, lhh = lane % 2;  // the lane's dims of the rotation: 8 lcp + 4 lhh .. and 32 up
    // K and V of the 8 keys from k on (into the LDS rows at kd and vd): requested, and
    // later rotated in place. Keys past the row's end are loaded from its last one and become zeros.
    auto load_unit = [&](int k, uint16_t* kd, uint16_t* vd) __attribute__((always_inline)) {
        const uint32_t off = (uint32_t)min(k + lkey, n - 1) * stride + 16u * ((lane % 8) ^ lkey);
        dma16s(kbase, off, kd);
        dma16s(vbase, off, vd);
    };
    auto unit_row = [&](int k) __attribute__((always_inline)) { return table_row(min(k + lkey, n - 1)); };
    auto load_table = [&](int row, floatx4& c, floatx4& s) __attribute__((always_inline)) {
        const float* tp = a.table + (size_t)row * kDH + 8 * lcp + 4 * lhh;
        c = *reinterpret_cast<const floatx4*>(tp);
        s = *reinterpret_cast<const floatx4*>(tp + kDH / 2);
    };
    const int rofs0 = swz(lkey, lcp) + 4 * lhh, rofs1 = swz(lkey, lcp + 4) + 4 * lhh;
    auto rotate_unit = [&](int k, uint16_t* kd, uint16_t* vd, floatx4 c, floatx4 s) __attribute__((always_inline)) {
        if (ROPE) {
            const floatx4 x = widen4<T>(*reinterpret_cast<const u32x2*>(kd + rofs0));
            const floatx4 y = widen4<T>(*reinterpret_cast<const u32x2*>(kd + rofs1));
            *reinterpret_cast<u32x2*>(kd + rofs0) = narrow4<T>(x * c - y * s);
            *reinterpret_cast<u32x2*>(kd + rofs1) = narrow4<T>(y * c + x * s);
        }
        if (k + 8 > n && k + lkey >= n) {
            *reinterpret_cast<u32x2*>(kd + rofs0) = u32x2{0u, 0u};
            *reinterpret_cast<u32x2*>(kd + rofs1) = u32x2{0u, 0u};
            *reinterpret_cast<u32x2*>(vd + rofs0) = u32x2{0u, 0u};
            *reinterpret_cast<u32x2*>(vd + rofs1) = u32x2{0u, 0u};
        }
    };

    // the wave's units of a block: unit wave + i NW
    floatx4 tc[kU] = {}, ts[kU] = {};  // the table rows of the block being loaded
    int trow[kU];            // the table rows' indexes of the block after it
    auto unit = [&](int i) __attribute__((always_inline)) { return 8 * (wave + i * NW); };
    auto load_kv = [&](int b, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kU; i++)
            load_unit(b * kKB + unit(i), &lds.kv[slot][0][unit(i) * kDH], &lds.kv[slot][1][unit(i) * kDH]);
    };
    auto load_rows = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kU; i++)
            if (ROPE) trow[i] = unit_row(b * kKB + unit(i));
    };
    auto load_tables = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kU; i++)
            if (ROPE) load_table(trow[i], tc[i], ts[i]);
    };
    auto rotate = [&](int b, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kU; i++)
            rotate_unit(b * kKB + unit(i), &lds.kv[slot][0][unit(i) * kDH], &lds.kv[slot][1][unit(i) * kDH], tc[i], ts[i]);
    };

    for (int b = wave; b < nblk; b += NW) {
        const uint64_t bits = __ballot(mask.key_valid(vrow, b * kKB + lane));
        if (lane == 0) lds.mask[b] = bits;
    }
    __syncthreads();
    const uint64_t need = __ballot(lane < nblk && mask.any_allowed(lds.mask[lane], lane * kKB, part * NW * kQ,
                                                                   min((part + 1) * NW * kQ, n) - 1));
    auto next_block = [&](int after) __attribute__((always_inline)) {
        const uint64_t rest = after + 1 >= 64 ? 0ull : need & (~0ull << (after + 1));
        return rest ? (int)__builtin_ctzll(rest) : nblk;
    };
    int b0 = lone ? nblk : next_block(-1);
    int b1 = b0 < nblk ? next_block(b0) : nblk;
    int b2 = b1 < nblk ? next_block(b1) : nblk;
    if (b0 < nblk) {
        load_kv(b0, 0);
        load_rows(b0);
        load_tables();
    }
    if (b1 < nblk) {
        load_kv(b1, 1);
        load_rows(b1);
    }

    // Q operands: rotated, scaled by qscale (log2(e) times the score scale), rounded to T
    x8 qreg[4];
    {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            floatx4 x[2], y[2];
            widen8<T>(qraw[s], x[0], x[1]);
            widen8<T>(qraw[s + 2], y[0], y[1]);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if (ROPE) {
                    const floatx4 rx = x[u] * qc[s][u] - y[u] * qs[s][u], ry = y[u] * qc[s][u] + x[u] * qs[s][u];
                    x[u] = rx;
                    y[u] = ry;
                }
                x[u] *= a.qscale;
                y[u] *= a.qscale;
            }
            qreg[s] = __builtin_bit_cast(x8, narrow8<T>(x[0], x[1]));
            qreg[s + 2] = __builtin_bit_cast(x8, narrow8<T>(y[0], y[1]));
        }
    }
    wait_vm<0>();
    if (b0 < nblk) rotate(b0, 0);
    if (b1 < nblk) load_tables();
    if (b2 < nblk) load_rows(b2);
    lds_barrier();

    floatx16 o_acc[2] = {floatx16{0}, floatx16{0}};
    // softmax state of query j (equal in lanes j and j+32), as in time_attention_lp.hip
    float m_tot = 0.f, m_mfma = 0.f, resid = 0.f, l_run = 0.f;
    bool has_ref = false, any_resid = false;
    uint32_t qx0 = g == 0 ? E::kBigQ : 0u;

    // element offsets of the lane's operand rows in a 32-key half: K's chunk of step s at kofs ^ 16 s, the
    // transposing reads of V's 32-dim tile t at vofs ^ 32 t
    const int kofs = swz(j, g);
    const int vkey = 4 * g + (lane % 16) / 4;
    const int vofs = swz(vkey, 2 * ((lane / 16) % 2) + (lane % 4) / 2) + 4 * (lane % 2);
    // one 32-key half: S^T, P, the row sum check (and slow path), PV
    auto half_block = [&](const uint16_t* kb, const uint16_t* vb, uint32_t allowed, uint32_t kmask, bool uniform)
                          __attribute__((always_inline)) {
        const bool lane_keys = allowed != 0;
        floatx16 s_acc = floatx16{0};
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const x8 kv = __builtin_bit_cast(x8, *reinterpret_cast<const u32x4*>(&kb[kofs ^ (16 * s)]));
            s_acc = Lp<T>::mfma(kv, qreg[s], s_acc);
        }
        const uint32_t kx0 = g == 0 ? (((kmask >> j) & 1u) ? E::kLive : E::kDead) : 0u;
        s_acc = Lp<T>::mfma(__builtin_bit_cast(x8, u32x4{kx0, 0u, 0u, 0u}),
                            __builtin_bit_cast(x8, u32x4{qx0, 0u, 0u, 0u}), s_acc);
        // reg rho in lane (j, g) holds key 32sb + 8*(rho/4) + 4g + rho%4 of the block
        if (!uniform) {
            const uint32_t w = allowed >> (4 * g);
#pragma unroll
            for (int rho = 0; rho < 16; rho++)
                if (!((w >> (8 * (rho / 4) + rho % 4)) & 1u)) s_acc[rho] = -INFINITY;
        }
        x8 p[2];
        auto exps = [&](float shift) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                floatx4 lo, hi;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    lo[u] = fast_exp2(s_acc[8 * c + u] - shift);
                    hi[u] = fast_exp2(s_acc[8 * c + 4 + u] - shift);
                }
                p[c] = __builtin_bit_cast(x8, narrow8<T>(lo, hi));
            }
        };
        auto row_sum = [&]() __attribute__((always_inline)) {
            float acc = 0.f;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const u32x4 w = __builtin_bit_cast(u32x4, p[c]);
#pragma unroll
                for (int d = 0; d < 4; d++) acc = E::dot2(w[d], acc);
            }
            return pair_sum(acc);
        };
        if (!any_resid) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                floatx4 lo, hi;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    lo[u] = fast_exp2(s_acc[8 * c + u]);
                    hi[u] = fast_exp2(s_acc[8 * c + 4 + u]);
                }
                p[c] = __builtin_bit_cast(x8, narrow8<T>(lo, hi));
            }
        } else {
            exps(resid);
        }
        float lb = row_sum();
        const bool bad = !(lb <= kSumHi) || (!has_ref && lane_keys && !(lb >= kSumLo));
        if (__any(bad)) {
            float mx = s_acc[0];
#pragma unroll
            for (int rho = 1; rho < 16; rho++) mx = fmaxf(mx, s_acc[rho]);
            mx = pair_max(mx);
            const float s_max = m_mfma + mx;
            float m_new = !lane_keys ? m_tot : (has_ref ? fmaxf(m_tot, s_max) : s_max);
            const uint32_t bm = to_bits<T>(fminf(fmaxf(-m_new, -E::kMax), E::kMax));
            const float m_enc = -from_bits<T>(bm);
            if (fabsf(m_new) <= E::kMax) m_new = m_enc;  // keep the reference exactly encodable
            exps(m_new - m_mfma);
            lb = row_sum();
            if (has_ref) {
                const float alpha = fast_exp2(m_tot - m_new);
                o_acc[0] *= alpha;
                o_acc[1] *= alpha;
                l_run *= alpha;
            }
            m_tot = m_new;
            m_mfma = m_enc;
            resid = m_tot - m_mfma;
            any_resid = __any(resid != 0.f);
            qx0 = g == 0 ? (E::kBigQ | (bm << 16)) : 0u;
        }
        l_run += lb;
        has_ref = has_ref || lane_keys;
        // O^T += V^T P^T, 16 keys per MFMA
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const uint16_t* vp = vb + 16 * c * kDH + (vofs ^ (32 * t));
                const u32x2 v0 = read_tr(vp), v1 = read_tr(vp + 8 * kDH);
                o_acc[t] = Lp<T>::mfma(__builtin_bit_cast(x8, u32x4{v0[0], v0[1], v1[0], v1[1]}), p[c], o_acc[t]);
            }
        }
    };

    // the wave's queries are all the encoder's, or all the decoder's
    const bool all_enc = q0 + nq <= a.enc, all_dec = q0 >= a.enc;
    // the keys of block b that the lane's query sees, and whether every query of the wave sees them `alike`
    auto visible = [&](int b, bool& alike) __attribute__((always_inline)) {
        const int k0 = b * kKB;
        const uint64_t word = lds.mask[b];
        const uint64_t sword = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)word) |
                               ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(word >> 32)) << 32);
        // without a look at the lanes: whole blocks before the first query, after the last one of a known row's,
        // and the encoder's as the decoder sees them
        alike = !TS || (all_enc && (k0 + kKB <= q0 || (mask.known && k0 >= q0 + kQ && k0 + kKB <= a.enc))) ||
                (all_dec && k0 + kKB <= a.enc);
        if (!TS || alike) return TS && all_dec ? sword & bits_below(a.ll, k0) : sword;
        uint64_t allowed = mask.allowed(sword, k0, q0 + j);
        // lanes past the last query take lane 0's keys so they never decide a wave-wide branch
        const uint64_t ref = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)allowed) |
                             ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(allowed >> 32)) << 32);
        return j >= nq ? ref : allowed;
    };

    if (lone) {
        // One tile for the whole workgroup: instead of seven waves that only stage, six waves take every sixth
        // 32-key half each, stage it for themselves in a sixth of the ring, without a barrier, and add up at the end.
        constexpr int kSplit = 6, kPiece = kHalf * kDH;  // elements of a half block of K or V
        static_assert(kSplit * 2 * kPiece <= kSlots * 2 * kKB * kDH, "the waves' areas");
        static_assert((kSplit - 1) * kHand * 2 <= kSlots * 2 * kKB * kDH, "the handed over results");
        uint16_t* ring = &lds.kv[0][0][0];
        uint16_t* kd = ring + wave * 2 * kPiece;
        uint16_t* vd = kd + kPiece;
        for (int hb = wave; wave < kSplit && hb * kHalf < n; hb += kSplit) {
            const int b = hb / 2, k = hb * kHalf;
            if (!((need >> b) & 1ull)) continue;
            bool alike;
            const uint64_t allowed = visible(b, alike);
            const uint32_t a32 = hb % 2 ? (uint32_t)(allowed >> 32) : (uint32_t)allowed;
            if (!__any(a32 != 0)) continue;
#pragma unroll
            for (int i = 0; i < kHalf / 8; i++) load_unit(k + 8 * i, kd + 8 * i * kDH, vd + 8 * i * kDH);
#pragma unroll
            for (int i = 0; i < kHalf / 8; i += 2) {
                floatx4 c0{}, c1{}, s0{}, s1{};
                if (ROPE) {
                    load_table(unit_row(k + 8 * i), c0, s0);
                    load_table(unit_row(k + 8 * i + 8), c1, s1);
                }
                wait_vm<0>();
                rotate_unit(k + 8 * i, kd + 8 * i * kDH, vd + 8 * i * kDH, c0, s0);
                rotate_unit(k + 8 * i + 8, kd + 8 * (i + 1) * kDH, vd + 8 * (i + 1) * kDH, c1, s1);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            half_block(kd, vd, a32, alike ? a32 : ~0u, alike);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        lds_barrier();
        float* hand = reinterpret_cast<float*>(ring) + lane;
        if (wave > 0 && wave < kSplit) {
            float* mine = hand + (wave - 1) * kHand;
#pragma unroll
            for (int i = 0; i < 32; i++) mine[i * kWave] = o_acc[i / 16][i % 16];
            mine[32 * kWave] = m_tot;
            mine[33 * kWave] = l_run;
            mine[34 * kWave] = has_ref ? 1.f : 0.f;
        }
        lds_barrier();
        if (wave > 0) return;
        for (int w = 0; w < kSplit - 1; w++) {
            const float* p = hand + w * kHand;
            const float m2 = p[32 * kWave];
            const bool ref2 = p[34 * kWave] != 0.f;
            const float m = has_ref && ref2 ? fmaxf(m_tot, m2) : (has_ref ? m_tot : m2);
            const float f1 = has_ref ? fast_exp2(m_tot - m) : 0.f, f2 = ref2 ? fast_exp2(m2 - m) : 0.f;
            l_run = l_run * f1 + p[33 * kWave] * f2;
#pragma unroll
            for (int i = 0; i < 32; i++) o_acc[i / 16][i % 16] = o_acc[i / 16][i % 16] * f1 + p[i * kWave] * f2;
            m_tot = m;
            has_ref = has_ref || ref2;
        }
    }

    auto compute = [&](int b, int slot) __attribute__((always_inline)) {
        bool alike;
        const uint64_t allowed = visible(b, alike);
#pragma unroll
        for (int sb = 0; sb < 2; sb++) {
            const uint32_t a32 = sb ? (uint32_t)(allowed >> 32) : (uint32_t)allowed;
            if (__any(a32 != 0))
                half_block(&lds.kv[slot][0][sb * kHalf * kDH], &lds.kv[slot][1][sb * kHalf * kDH], a32, alike ? a32 : ~0u, alike);
        }
    };

    int slot = 0;
    while (b0 < nblk) {
        const int s1 = slot == kSlots - 1 ? 0 : slot + 1, s2 = s1 == kSlots - 1 ? 0 : s1 + 1;
        wait_vm<0>();
        if (b1 < nblk) rotate(b1, s1);
        const int b3 = b2 < nblk ? next_block(b2) : nblk;
        if (b2 < nblk) {
            load_kv(b2, s2);
            load_tables();
        }
        if (b3 < nblk) load_rows(b3);
        if (nq > 0) compute(b0, slot);
        lds_barrier();
        b0 = b1;
        b1 = b2;
        b2 = b3;
        slot = s1;
    }

    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
    const size_t at = (row0 + q) * inner + h * kDH + 8 * g;
    // Lanes (j, 0) and (j, 1) trade halves of each 16-dim run (v_permlane32_swap), so each holds 8 consecutive
    // dims 32t + 16p + 8g ..
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            floatx4 d0, d4;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(o_acc[t][8 * p + u] * inv),
                                                                 __float_as_uint(o_acc[t][8 * p + 4 + u] * inv), false, false);
                d0[u] = __uint_as_float(sw[0]);
                d4[u] = __uint_as_float(sw[1]);
            }
            if (j < nq) {
                if (a.gate) {
                    // the output gate: att * sigmoid(g) (CpuTimestral.java:156-161)
                    floatx4 g0, g4;
                    widen8<T>(*reinterpret_cast<const u32x4*>(static_cast<const T*>(a.gate) + at + 32 * t + 16 * p), g0, g4);
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        d0[u] *= __builtin_amdgcn_rcpf(1.f + fast_exp2(-g0[u] * kLog2e));
                        d4[u] *= __builtin_amdgcn_rcpf(1.f + fast_exp2(-g4[u] * kLog2e));
                    }
                }
                *reinterpret_cast<u32x4*>(static_cast<T*>(a.out) + at + 32 * t + 16 * p) = narrow8<T>(d0, d4);
            }
        }
}

template <typename T, int NW, bool TS>
hipError_t launch_nw(TimeArgs a, hipStream_t stream) {
    const dim3 grid((uint32_t)((uint64_t)a.rows * a.heads * a.qgroups)), block(NW * kWave);
    if (a.table) hipLaunchKernelGGL((time_attention_lpr<T, NW, true, TS>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((time_attention_lpr<T, NW, false, TS>), grid, block, 0, stream, a);
    return hipGetLastError();
}

template <typename T, bool TS>
hipError_t launch_lpr(TimeArgs a, hipStream_t stream) {
    // A workgroup of 4 waves costs 0.6 of one of 8 (all of a row's parts, 256 x 512 tokens: 0.41 against 0.35 ms; 300 x
    // 161 0.114 against 0.095), and 8 waves split a last part of one tile. So 4 waves for up to 4 tiles and for 10 .. 12
    // (1,000 x 65 0.134 against 0.171, 250 x 300 0.202 against 0.215), else 8 (64 x 577 0.128 against 0.136).
    const int tiles = (a.n + kQ - 1) / kQ;
    const int parts4 = (tiles + 3) / 4, parts8 = (tiles + 7) / 8;
    const bool four = tiles % 8 != 1 && 3 * parts4 < 5 * parts8;
    a.qgroups = four ? parts4 : parts8;
    return four ? launch_nw<T, 4, TS>(a, stream) : launch_nw<T, 8, TS>(a, stream);
}

}  // namespace

// Rows of one tile stay on the streaming kernel's 2-wave workgroups (2,000 x 32 tokens 0.177 against 0.469 ms, 2,000 x
// 33 0.194 against 0.177).
bool time_attention_lpr_fits(const TimeArgs& a, int dh) { return dh == kDH && a.q_begin == 0 && a.n > kQ; }

hipError_t time_attention_lpr_launch(const TimeArgs& a, bool ts, bool fp16, hipStream_t stream) {
    if (fp16) return ts ? launch_lpr<_Float16, true>(a, stream) : launch_lpr<_Float16, false>(a, stream);
    return ts ? launch_lpr<__bf16, true>(a, stream) : launch_lpr<__bf16, false>(a, stream);
}

}  // namespace jc
