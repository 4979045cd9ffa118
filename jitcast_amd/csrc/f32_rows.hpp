// fp32 time attention of up to 16 queries of one (row, head) by one wave on fp32 MFMA, straight from
// memory: no LDS of its own, no barriers. time_attention_f32_split.hip computes again with it the queries
// whose results on fp16 pairs are not finite.
//
// Same contract as the kernel around it (time_mask.hpp, RoPE at the token's table row, the optional
// gate). Operand layouts of v_mfma_f32_16x16x4f32 (A lane i+16kk = A[i][kk], B lane j+16kk = B[kk][j],
// D lane j+16g reg r = D[4g+r][j]):
//   S^T[key][q] = K Q^T   step (m, u) contracts dim 16m + 4kk + u, so a lane holds 4 consecutive dims
//                         per m (one 16-byte load) and the RoPE pair of dim e < 32, e + 32, sits in
//                         the same lane (m and m + 2): the rotation is lane-local.
//   O^T[e][q] += V^T P^T  step c contracts keys 4kk + c, whose P^T is S^T's reg c in the same lane;
//                         V^T comes per lane as V[key][16t + i].
// Keys stream in 16-key tiles; a tile is loaded, then used (this path is for rare values, so nothing
// is prefetched and the registers stay below the surrounding kernel's).
#pragma once

#include "jc_common.hpp"
#include "jc_kernels.hpp"

namespace jc {

// Queries q0 + i (i < 16, below n) with bit i of `write` set are stored. words[b]: the validity word of
// key block b (64 keys); trow(t): the RoPE table row of token t.
template <bool ROPE, bool TS, bool X3, typename Trow>
__device__ __forceinline__ void f32_rows(const TimeArgs& a, const TimeMask<TS>& mask, const uint64_t* words, Trow trow,
                                         int r, int h, int q0, uint32_t write, int lane) {
    constexpr int kDH = 64, kT = 16;
    const int n = a.n, inner = a.inner;
    const int i = lane % 16, kk = lane / 16;  // also (j, g) of the accumulator layouts
    const size_t ts = 3 * (size_t)inner;      // floats per token of qkv
    const float* base = static_cast<const float*>(a.qkv) + (size_t)r * n * ts + h * kDH;

    // dims 16m + 4kk .. +3 of a token's vector at p, rotated at its table row
    auto load = [&](const float* p, int t, floatx4* v) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 4; m++) v[m] = *reinterpret_cast<const floatx4*>(p + 16 * m + 4 * kk);
        if (ROPE) {
            const float* tab = a.table + (size_t)trow(t) * kDH + 4 * kk;
#pragma unroll
            for (int m = 0; m < 2; m++) {
                const floatx4 c = *reinterpret_cast<const floatx4*>(tab + 16 * m);
                const floatx4 s = *reinterpret_cast<const floatx4*>(tab + kDH / 2 + 16 * m);
                const floatx4 x = v[m], y = v[m + 2];
                v[m] = x * c - y * s;
                v[m + 2] = y * c + x * s;
            }
        }
    };
    const int q = min(q0 + i, n - 1);
    floatx4 qv[4];
    load(base + (size_t)q * ts, q, qv);
#pragma unroll
    for (int m = 0; m < 4; m++) qv[m] *= a.qscale;

    float m_run = -INFINITY, l_run = 0.f;
    floatx4 o[4];
#pragma unroll
    for (int t = 0; t < 4; t++) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int kt = 0; kt < (n + kT - 1) / kT; kt++) {
        const int b = kt * kT / kMaskBlock, k0 = b * kMaskBlock;
        const uint32_t see = (uint32_t)(mask.allowed(words[b], k0, q) >> (kt * kT - k0)) & 0xffffu;
        if (!__any(see != 0)) continue;
        const int key = min(kT * kt + i, n - 1);
        floatx4 kr[4];
        load(base + (size_t)key * ts + inner, key, kr);
        floatx4 s = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < 4; m++) {
#pragma unroll
            for (int u = 0; u < 4; u++) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[m][u], qv[m][u], s, 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < 4; c++) s[c] = ((see >> (4 * kk + c)) & 1u) ? s[c] : -INFINITY;  // key 16kt + 4kk + c
        const float mx = quad_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
        const float m_new = fmaxf(m_run, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = fast_exp2(m_run - m_use);
        m_run = m_new;
#pragma unroll
        for (int c = 0; c < 4; c++) s[c] = fast_exp2(s[c] - m_use);
        l_run = l_run * alpha + (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            o[t] *= alpha;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int vkey = min(kT * kt + 4 * kk + c, n - 1);
                const float v = base[(size_t)vkey * ts + 2 * inner + 16 * t + i];
                o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, s[c], o[t], 0, 0, 0);
            }
        }
    }

    // O^T reg r of lane (j, g) in dim tile t is dim 16t + 4g + r of query q0 + j
    const float l = quad_sum(l_run);
    if (q0 + i < n && ((write >> i) & 1u)) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
        const size_t at = ((size_t)r * n + q0 + i) * inner + h * kDH + 4 * kk;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            floatx4 v = o[t] * inv;
            if (a.gate) {
                const floatx4 gv = *reinterpret_cast<const floatx4*>(static_cast<const float*>(a.gate) + at + 16 * t);
#pragma unroll
                for (int u = 0; u < 4; u++) v[u] *= 1.f / (1.f + fast_exp2(-gv[u] * kLog2e));
            }
            if constexpr (X3) {  // [hi | hi | lo] rows, each value's three-term split
                store_split_row(static_cast<_Float16*>(a.out) + ((size_t)r * n + q0 + i) * 3 * inner, inner,
                                h * kDH + 4 * kk + 16 * t, v);
            } else {
                *reinterpret_cast<floatx4*>(static_cast<float*>(a.out) + at + 16 * t) = v;
            }
        }
    }
}

}  // namespace jc
