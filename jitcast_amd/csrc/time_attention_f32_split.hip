// Time attention for gfx950: the FP32 path of Chronos-2 and Timestral for 64-wide heads, on fp16 MFMA
// (time_attention_f32.hip takes the other widths).
//
// The contract is time_attention_f32.hip's (Chronos2Kernels.java:87-116, 118-464; TimestralKernels.java:71-100,
// 102-278, 572-578): RoPE at each token's table row, the time mask (time_mask.hpp), fp32 scores, softmax,
// sums and results, the optional sigmoid gate. Every fp32 product of K Q^T and P V is made of three fp16
// MFMA products: x = hi + lo with hi = fp16(x), lo = fp16(x - hi), a.b = a_hi.b_hi + a_hi.b_lo + a_lo.b_hi
// (fp16 products are exact in fp32; the lo.lo product left out is at most 2^-22 of a.b). The pairs hold
// values scaled by powers of two: a query by its own largest magnitude, the (row, head)'s keys and its values
// by the largest of the first block that holds a nonzero one (to [2, 4), so lo is accurate to 2^-25 there and
// hi has a factor of 2^14 of headroom), P by 2^10. The scales leave with the softmax's multiply-add and the
// output's factor. A value past the headroom becomes an infinity; queries whose results are not finite are
// computed again on fp32 MFMA (f32_rows.hpp), so no finite value is out of range and infinities and NaN
// come out as they would there.
//
// Work split: a workgroup of 4 waves takes 128 consecutive queries of one (row, head), a wave 32. Keys
// stream through LDS in blocks of 32, double-buffered; blocks no query of the workgroup can see are skipped.
// Each block is loaded, rotated and split once per workgroup, the next one's loads issued above the
// current one's MFMAs.
// LDS: K rows of 64 dims (128 bytes per part), 16-byte chunk c of key r at c ^ ((r >> 1) & 7); V^T rows of
// 32 keys (64 bytes per part), chunk c of dim r at c ^ ((r >> 2) & 3), the keys of a 16-key group in
// the order that S^T's registers hold them: 16-lane read and write phases hit distinct banks.
//
// MFMA layouts (v_mfma_f32_32x32x16_f16: A lane i+32g = A[i][8g..8g+7], B lane j+32g = B[8g..8g+7][j],
// D lane j+32g reg r = D[8(r/4) + 4g + r%4][j]):
//   S^T[key][q] = K Q^T    step s contracts dims 16s + 8g ..: the RoPE pair (e, e + 32) sits in one lane
//   O^T[e][q] += V^T P^T   step c contracts the 16 keys 16c ..; lane (j, g) holds keys 16c + 8a + 4g + u in
//                          S^T's registers 8c + 4a + u, so P never leaves registers
//
// What bounds it: the MFMA and VALU pipes of a SIMD, which overlap by about half. 256 x 513 tokens x 12
// heads (half-row left padding): 0.85 ms, 183 TFLOP/s of fp32 products mask-aware (on fp32 MFMA 1.54 ms, 101);
// MFMA busy 28% of the cycles, VALU 60%. Timed variants at 512 tokens, no padding (0.94 ms on that box): the
// hi.hi products alone 0.71, no staging 0.70. Two query tiles per wave (a block staged once for 256
// queries, 2 waves per SIMD) ran 0.83 there but 0.89 against 0.87 at 513 and 0.74 against 0.66 at
// Timestral's 64 x 1,025; 2 waves per workgroup 1.07 at 513. Error against 64 bits 4.6e-7 (7.3e-7
// on fp32 MFMA).
// One query's softmax state lives in lanes j and j+32; the reference max moves only when a score passes it
// by 2^5, which P's 2^10 and fp16's range allow.
#include "f32_rows.hpp"
#include "jc_common.hpp"
#include "jc_kernels.hpp"
#include "lp_common.hpp"
#include "time_mask.hpp"

namespace jc {
namespace {

using lp::make_rsrc;

constexpr int kDH = 64, kKB = 32, kQ = 32;
constexpr int kWaves = 4;
constexpr int kMaxTokens = 4096;
constexpr float kPScale = 1024.f;  // P's scale, 2^10 (in the exponent's argument it would cost 3 bits of it)
constexpr int kPExp = 10;
constexpr float kLazy = 5.f;       // the reference max moves past 2^5: P stays within 2^15
constexpr int kTarget = 1;         // scaled maxima lie in [2^1, 2^2)

template <bool TS>
struct alignas(16) SplitLds {
    uint16_t k[2][2][kKB * kDH];  // [buffer][hi, lo]
    uint16_t v[2][2][kDH * kKB];
    uint64_t mask[kMaxTokens / kMaskBlock];  // per 64-key word: key validity bits
    float red[2][kWaves];                    // the waves' maxima of K and V
    int32_t pos[TS ? kMaxTokens : 1];        // table row of every token of the row (Timestral)
};

// the exponent field of 2^(kTarget - floor(log2 m)) for m > 0, where its inverse is normal too
__device__ __forceinline__ int scale_field(float m) {
    return min(max(254 + kTarget - (int)(__float_as_uint(m) >> 23), 2), 252);
}
__device__ __forceinline__ float field_float(int f) { return __uint_as_float((uint32_t)f << 23); }

// |v| where it is finite, else 0
__device__ __forceinline__ float finite_abs(float v) {
    const float m = fabsf(v);
    return m < INFINITY ? m : 0.f;
}
__device__ __forceinline__ float max4(float m, floatx4 v) {
#pragma unroll
    for (int u = 0; u < 4; u++) m = fmaxf(m, finite_abs(v[u]));
    return m;
}

// x * s as a pair: s a power of two
struct Pair {
    _Float16 hi, lo;
};
__device__ __forceinline__ Pair split_scaled(float x, float s) {
    const _Float16 hi = (_Float16)__builtin_fmaf(x, s, 0.f);
    return Pair{hi, (_Float16)__builtin_fmaf(x, s, -(float)hi)};
}

// X3 (Chronos-2; the JC_F16X3 layer): out is the O projection's A operand, fp16 rows of 3 * inner values
// [hi | hi | lo] (the three-term split of each fp32 output value), so the layer needs no separate split pass.
// A layer of 48 x 133 tokens (768 wide, 12 heads): 0.949 ms with its time attention on fp32 MFMA, 0.928 here.
template <bool ROPE, bool TS, bool X3>
__global__ __launch_bounds__(kWaves * kWave, 3) void time_attention_f32_split(const TimeArgs a) {
    __shared__ SplitLds<TS> lds;
    const float* __restrict__ qkv = static_cast<const float*>(a.qkv);
    const int n = a.n, inner = a.inner;
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane % 32, g = lane / 32;
    const uint32_t logical = xcd_remap(blockIdx.x, (uint32_t)a.rows * a.heads * a.qgroups);
    const int qg = logical % a.qgroups, bh = logical / a.qgroups;
    const int h = bh % a.heads, r = bh / a.heads;
    TimeMask<TS> mask;
    mask.init(a, r);
    const int32_t* vrow = a.valid + (size_t)r * (TS ? a.enc : n);
    const size_t row0 = (size_t)r * n;

    // The wave's queries are requested first, so their latency overlaps the validity scan. Lane (j, g)
    // holds dims 16s + 8g .. +7 of query q0 + j for s < 4.
    const int q0 = (qg * kWaves + wave) * kQ;
    const int nq = min(max(n - q0, 0), kQ);
    floatx4 qa[8], qc[4], qs[4];
    if (j < nq) {
        const int q = q0 + j;
        const float* qp = qkv + (row0 + q) * 3 * inner + h * kDH + 8 * g;
        int trow = q;
        if (TS && ROPE && a.pos) trow = min(max(a.pos[row0 + q], 0), a.table_rows - 1);
#pragma unroll
        for (int s = 0; s < 8; s++) qa[s] = *reinterpret_cast<const floatx4*>(qp + 16 * (s / 2) + 4 * (s % 2));
        if (ROPE) {
            const float* tp = a.table + (size_t)trow * kDH + 8 * g;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                qc[s] = *reinterpret_cast<const floatx4*>(tp + 16 * (s / 2) + 4 * (s % 2));
                qs[s] = *reinterpret_cast<const floatx4*>(tp + kDH / 2 + 16 * (s / 2) + 4 * (s % 2));
            }
        }
    }

    // key validity of every 64-key word of the row, and (Timestral) every token's table row
    const int nwords = (n + kMaskBlock - 1) / kMaskBlock;
    for (int w = wave; w < nwords; w += kWaves) {
        const uint64_t bits = __ballot(mask.key_valid(vrow, w * kMaskBlock + (int)lane));
        if (lane == 0) lds.mask[w] = bits;
    }
    if (TS) {
        for (int t = tid; t < n; t += kWaves * kWave)
            lds.pos[t] = a.pos ? min(max(a.pos[row0 + t], 0), a.table_rows - 1) : t;
    }
    __syncthreads();
    // 64-key words any query of the workgroup can see (the same in every wave)
    const int qlo = qg * kWaves * kQ, qhi = min(qlo + kWaves * kQ, n) - 1;
    const uint64_t need = __ballot((int)lane < nwords && mask.any_allowed(lds.mask[lane], lane * kMaskBlock, qlo, qhi));
    const int nblk = (n + kKB - 1) / kKB;
    auto next_block = [&](int after) {
        const int b = after + 1, w = b * kKB / kMaskBlock;
        const uint64_t rest = (b >= nblk || w >= 64) ? 0ull : need & (~0ull << w);
        if (!rest) return nblk;
        const int wn = (int)__builtin_ctzll(rest);
        return wn == w ? b : wn * kMaskBlock / kKB;
    };

    // Q operands: rotated, scaled to the query's own largest magnitude, as pairs
    halfx8 qh[4], ql[4];
    int q_exp = 0;  // the query's scale exponent
    {
        float m = 0.f;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            floatx4 x = floatx4{0.f, 0.f, 0.f, 0.f}, y = x;
            if (j < nq) {
                x = qa[s];
                y = qa[s + 4];
                if (ROPE) {
                    x = qa[s] * qc[s] - qa[s + 4] * qs[s];
                    y = qa[s + 4] * qc[s] + qa[s] * qs[s];
                }
            }
            qa[s] = x;
            qa[s + 4] = y;
#pragma unroll
            for (int u = 0; u < 4; u++) m = fmaxf(m, fmaxf(fabsf(x[u]), fabsf(y[u])));
        }
        if (__any(m == INFINITY)) {  // the largest finite one
            m = 0.f;
#pragma unroll
            for (int s = 0; s < 8; s++) m = max4(m, qa[s]);
        }
        m = pair_max(m);
        const int f = m > 0.f ? scale_field(m) : 127;
        q_exp = f - 127;
        const float sc = field_float(f);
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const Pair p = split_scaled(qa[2 * s + u / 4][u % 4], sc);
                qh[s][u] = p.hi;
                ql[s][u] = p.lo;
            }
    }

    // Staging, an eighth of a block per wave of K and of V: key kl = 8 wave + lane / 8, dims ke .. ke+3 and
    // ke+32 .., with the cos and sin of the pairs; and dim `lane` of keys vk + {0..3, 8..11}.
    const uint32_t stride_b = 12u * inner;
    floatx4 kx[2], kcs[2], vx[2];  // the next block in flight: K, its cos and sin, V
    const uint32_t ke = 4 * (lane % 8), kl = 8 * wave + lane / 8;
    const uint32_t off_k = kl * stride_b + 4 * ke;
    const int vk = 16 * (wave / 2) + 4 * (wave % 2);
    auto load = [&](int b) __attribute__((always_inline)) {
        const int k0 = b * kKB;
        const float* kp = qkv + (row0 + k0) * 3 * inner + inner + h * kDH;
        const uint32_t left = (uint32_t)(n - k0) * stride_b - (uint32_t)(inner + h * kDH) * 4u;
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(kp, left);  // keys past n read as 0
        const __amdgpu_buffer_rsrc_t rv = make_rsrc(kp + inner, left - (uint32_t)inner * 4u);
        const __amdgpu_buffer_rsrc_t rt = make_rsrc(a.table, (uint32_t)(TS ? a.table_rows : n) * kDH * 4u);
        kx[0] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rk, off_k, 0, 0));
        kx[1] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rk, off_k + kDH * 2, 0, 0));
        if (ROPE) {
            const int key = k0 + kl;
            const uint32_t row = TS ? (key < n ? (uint32_t)lds.pos[key] : 0u) : (uint32_t)key;
            const uint32_t ot = row * (kDH * 4) + 4 * ke;
            kcs[0] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rt, ot, 0, 0));
            kcs[1] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rt, ot + kDH * 2, 0, 0));
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            // the range check takes the scalar offset in; a key past n reads the last one's value (its P is 0)
            const int key = min(vk + 8 * (e / 4) + e % 4, n - 1 - k0);
            vx[e / 4][e % 4] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, lane * 4, (uint32_t)key * stride_b, 0));
        }
    };
    int k_field = 0, v_field = 0;  // the scales' exponent fields, 0 while every value was zero (uniform)
    float sk = 1.f, sv = 1.f;
    auto store = [&](int buf) __attribute__((always_inline)) {
        if (k_field == 0 || v_field == 0) {
            float mk = 0.f, mv = 0.f;
            mk = max4(max4(mk, kx[0]), kx[1]);
            mv = max4(max4(mv, vx[0]), vx[1]);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                mk = fmaxf(mk, __shfl_xor(mk, off));
                mv = fmaxf(mv, __shfl_xor(mv, off));
            }
            if (lane == 0) {
                lds.red[0][wave] = mk;
                lds.red[1][wave] = mv;
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < kWaves; w++) {
                mk = fmaxf(mk, lds.red[0][w]);
                mv = fmaxf(mv, lds.red[1][w]);
            }
            mk = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(mk)));
            mv = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(mv)));
            if (k_field == 0 && mk > 0.f) sk = field_float(k_field = scale_field(mk));
            if (v_field == 0 && mv > 0.f) sv = field_float(v_field = scale_field(mv));
            __syncthreads();  // red is free again
        }
        floatx4 x = kx[0], y = kx[1];
        if (ROPE) {
            x = kx[0] * kcs[0] - kx[1] * kcs[1];
            y = kx[1] * kcs[0] + kx[0] * kcs[1];
        }
        halfx4 h0, l0, h1, l1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const Pair p = split_scaled(x[e], sk), q = split_scaled(y[e], sk);
            h0[e] = p.hi;
            l0[e] = p.lo;
            h1[e] = q.hi;
            l1[e] = q.lo;
        }
        const uint32_t ch = ke / 8, sw = (kl >> 1) & 7;
        const uint32_t o0 = kl * kDH + ((ch ^ sw) << 3) + (ke & 4);
        const uint32_t o1 = kl * kDH + (((ch + 4) ^ sw) << 3) + (ke & 4);
        *reinterpret_cast<halfx4*>(&lds.k[buf][0][o0]) = h0;
        *reinterpret_cast<halfx4*>(&lds.k[buf][1][o0]) = l0;
        *reinterpret_cast<halfx4*>(&lds.k[buf][0][o1]) = h1;
        *reinterpret_cast<halfx4*>(&lds.k[buf][1][o1]) = l1;
        halfx8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const Pair p = split_scaled(vx[e / 4][e % 4], sv);
            hi[e] = p.hi;
            lo[e] = p.lo;
        }
        const uint32_t ov = lane * kKB + (((uint32_t)wave ^ ((lane >> 2) & 3)) << 3);
        *reinterpret_cast<halfx8*>(&lds.v[buf][0][ov]) = hi;
        *reinterpret_cast<halfx8*>(&lds.v[buf][1][ov]) = lo;
    };

    int kb = next_block(-1);
    if (kb < nblk) {
        load(kb);
        store(0);
    }
    __syncthreads();

    floatx16 o_acc[2] = {floatx16{0}, floatx16{0}};
    float m_run = -INFINITY, l_run = 0.f;
    int buf = 0;
    // Settle every prologue load here: the compiler cannot prove that the divergent Q loads were consumed
    // on all paths and would otherwise wait for the block's prefetch (vmcnt(0)) ahead of its MFMAs.
    __builtin_amdgcn_s_waitcnt(0);
    while (kb < nblk) {
        const int next = next_block(kb);
        if (next < nblk) load(next);
        // keep the prefetch above the block's MFMAs (the scheduler would sink it to its use)
        __builtin_amdgcn_sched_barrier(0);

        // the keys of this block the lane's query may see (bit i = key kb*32 + i)
        const int k0 = kb * kKB;
        const uint32_t allowed = (uint32_t)(mask.allowed(lds.mask[k0 / kMaskBlock], k0 & ~(kMaskBlock - 1), q0 + j) >>
                                            (k0 % kMaskBlock));
        if (nq > 0 && __any(j < nq && allowed != 0)) {
            floatx16 s = floatx16{0};
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const uint32_t o = j * kDH + (((uint32_t)(2 * t + g) ^ ((j >> 1) & 7)) << 3);
                const halfx8 kh = *reinterpret_cast<const halfx8*>(&lds.k[buf][0][o]);
                const halfx8 kx = *reinterpret_cast<const halfx8*>(&lds.k[buf][1][o]);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[t], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kx, qh[t], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[t], s, 0, 0, 0);
            }
            if (__any(j < nq && allowed != ~0u)) {
                // reg rho of lane (j, g) is key 8 (rho / 4) + 4g + rho % 4 of the block
                const uint32_t al = allowed >> (4 * g);
#pragma unroll
                for (int rho = 0; rho < 16; rho++)
                    if (!((al >> (8 * (rho / 4) + rho % 4)) & 1u)) s[rho] = -INFINITY;
            }
            // score times log2(e): s * c, with the scales of q and K taken off (at least the smallest normal
            // float, so a masked -inf stays -inf)
            const float c = fmaxf(__builtin_amdgcn_ldexpf(a.qscale, -(q_exp + (k_field ? k_field - 127 : 0))), 0x1p-126f);
            float mx = fmaxf(s[0], s[1]);
#pragma unroll
            for (int rho = 2; rho < 16; rho++) mx = fmaxf(mx, s[rho]);
            mx = pair_max(mx) * c;
            if (__any(mx > m_run + kLazy)) {
                const float m_new = fmaxf(m_run, mx);
                const float alpha = m_run == -INFINITY ? 0.f : fast_exp2(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
                o_acc[0] *= alpha;
                o_acc[1] *= alpha;
            }
            const float m_use = m_run == -INFINITY ? 0.f : m_run;
            halfx8 ph[2], pl[2];
            float rs = 0.f;
#pragma unroll
            for (int rho = 0; rho < 16; rho++) {
                const float p = fast_exp2(__builtin_fmaf(s[rho], c, -m_use));
                rs += p;
                const Pair pp = split_scaled(p, kPScale);
                ph[rho / 8][rho % 8] = pp.hi;
                pl[rho / 8][rho % 8] = pp.lo;
            }
            l_run += rs;
#pragma unroll
            for (int kc = 0; kc < 2; kc++)
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const uint32_t row = 32 * t + j;
                    const uint32_t o = row * kKB + (((uint32_t)(2 * kc + g) ^ ((row >> 2) & 3)) << 3);
                    const halfx8 vh = *reinterpret_cast<const halfx8*>(&lds.v[buf][0][o]);
                    const halfx8 vx = *reinterpret_cast<const halfx8*>(&lds.v[buf][1][o]);
                    o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[kc], o_acc[t], 0, 0, 0);
                    o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vx, ph[kc], o_acc[t], 0, 0, 0);
                    o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[kc], o_acc[t], 0, 0, 0);
                }
        }
        if (next < nblk) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
        kb = next;
    }

    // O^T reg 4q + u of lane (j, g) is dim 32t + 8q + 4g + u of query j. With the gate, o / l * sigmoid(g) is
    // one division by l (1 + e^-g) (CpuTimestral.java:156-161).
    const float l = pair_sum(l_run);
    const bool seen = l > 0.f && l < INFINITY;
    const float inv = seen ? 1.f / l : l == 0.f ? 0.f : NAN;
    const int oe = -(kPExp + (v_field ? v_field - 127 : 0));
    const size_t at = (row0 + q0 + j) * inner + h * kDH + 4 * g;
    const float* gp = a.gate && j < nq ? static_cast<const float*>(a.gate) + at : nullptr;
    float bad = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (gp) {
                const floatx4 gv = *reinterpret_cast<const floatx4*>(gp + 32 * t + 8 * q);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const float o = __builtin_amdgcn_ldexpf(o_acc[t][4 * q + u], oe);
                    const float d = 1.f + fast_exp2(-gv[u] * kLog2e);
                    o_acc[t][4 * q + u] = seen ? (d == INFINITY ? 0.f * o : o / (l * d)) : o * inv;
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; u++) o_acc[t][4 * q + u] = __builtin_amdgcn_ldexpf(o_acc[t][4 * q + u] * inv, oe);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) bad = __builtin_fmaf(o_acc[t][4 * q + u], 0.f, bad);
        }
    const uint64_t again64 = __ballot(j < nq && bad != bad);
    const uint32_t again = (uint32_t)again64 | (uint32_t)(again64 >> 32);  // bit i = query q0 + i
    const bool store_it = j < nq && !((again >> j) & 1u);
    if constexpr (X3) {
        // Lanes (j, 0) and (j, 1) trade halves of each 16-dim run (v_permlane32_swap), so each holds 8
        // consecutive dims 32t + 16p + 8g ..: each piece of the split goes out as one 16-byte store.
        _Float16* orow = static_cast<_Float16*>(a.out) + (row0 + q0 + j) * 3 * inner + h * kDH;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int p = 0; p < 2; p++) {
                floatx4 d0, d4;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(o_acc[t][8 * p + u]),
                                                                     __float_as_uint(o_acc[t][8 * p + 4 + u]), false, false);
                    d0[u] = __uint_as_float(sw[0]);
                    d4[u] = __uint_as_float(sw[1]);
                }
                if (store_it) store_split_row8(orow, inner, 32 * t + 16 * p + 8 * g, d0, d4);
            }
    } else if (store_it) {
        float* op = static_cast<float*>(a.out) + at;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<floatx4*>(op + 32 * t + 8 * q) =
                    floatx4{o_acc[t][4 * q], o_acc[t][4 * q + 1], o_acc[t][4 * q + 2], o_acc[t][4 * q + 3]};
    }
    if (again) {
        auto trow = [&](int t) { return TS ? lds.pos[t] : t; };
        for (int half = 0; half < 2; half++)
            if ((again >> (16 * half)) & 0xffffu)
                f32_rows<ROPE, TS, X3>(a, mask, lds.mask, trow, r, h, q0 + 16 * half, again >> (16 * half), lane);
    }
}

template <bool TS, bool X3>
hipError_t launch_split(TimeArgs a, hipStream_t stream) {
    a.qgroups = (a.n + kWaves * kQ - 1) / (kWaves * kQ);
    const dim3 grid((uint32_t)((uint64_t)a.rows * a.heads * a.qgroups)), block(kWaves * kWave);
    if (a.table) hipLaunchKernelGGL((time_attention_f32_split<true, TS, X3>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((time_attention_f32_split<false, TS, X3>), grid, block, 0, stream, a);
    return hipGetLastError();
}

}  // namespace

hipError_t time_attention_f32_split_launch(const TimeArgs& a, bool ts, hipStream_t stream) {
    return ts ? launch_split<true, false>(a, stream) : launch_split<false, false>(a, stream);
}

hipError_t time_attention_f32_x3_launch(const TimeArgs& a, int dh, hipStream_t stream) {
    if (dh != 64) return hipErrorInvalidValue;
    return launch_split<false, true>(a, stream);
}

}  // namespace jc
