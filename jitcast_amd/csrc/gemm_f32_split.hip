// The fp32 GEMM on fp16 MFMA: C[m, n] (+)= act(A[m, :k] . W[n, :k] + b[n]) with fp32 operands, sums
// and results (Kernels.gemm's flags and epilogue order, Kernels.java:50-103), every product made of
// three fp16 MFMA products instead of one fp32 one: fp16 MFMA runs 16 times as fast as fp32 MFMA.
//
// Operands. A value v of a row becomes x = v * 2^p, hi = fp16(x) and lo = fp16(x - hi), both rounded
// to nearest, and a.w becomes a_hi.w_hi + a_hi.w_lo + a_lo.w_hi (fp16 products are exact in fp32).
// 2^p is the row's own power of two (one per row of A and per row of W): the row's first stage of 32
// columns that holds a nonzero value is brought to a maximum in [4, 8), so lo is accurate to 2^-25 where
// the row's values are around 1 to 8 (a value's own fp32 rounding there) and hi has a factor of 2^13 of
// headroom. The split depends on the row's values alone, not on its place or its neighbours. A value
// past the headroom becomes an infinity, and results that are not finite are computed again on fp32
// MFMA, 32 x 32 tile by tile, from the operands themselves, each element on its own account: no finite
// value is out of range, and infinities and NaN among the operands come out as they would there.
//
// Tiling: a workgroup owns a BM x BN tile of C, a wave TM x TN MFMA tiles of 32 x 32
// (v_mfma_f32_32x32x16_f16: A lane i+32g = A[i][8g..8g+7], B lane j+32g = B[8g..8g+7][j], D lane
// j+32g reg r = D[8(r/4) + 4g + r%4][j]). K advances 32 at a time through two LDS stages; a stage
// holds hi and lo of BM and BN rows, 64 bytes per row and part, chunk c (8 values) of row r at
// position c ^ ((r >> 2) & 3), so that the 16 lanes of a read phase (16 rows, one chunk) and of a
// write phase (4 rows, 4 chunks) hit distinct banks. fp32 values arrive in registers by buffer loads
// (rows past m or n and columns past k read as zero through the range check), are split there and
// written to the stage that the MFMAs are not reading: one conversion per value and tile, two VALU
// instructions each (v_fma_mixlo/mixhi_f16), issued between the MFMAs.
//
// What bounds it: MFMA, at the clock that power allows. 65,472 x 768 x 3,072: 0.82 ms, 377 TFLOP/s of
// fp32 products, 1.13 PFLOP/s executed (hipBLASLt's fp32 kernels 2.13 ms, 145; its plain fp16 GEMM
// reaches 1.42 PFLOP/s on this card); MFMA pipes busy 71% of 1.25 M cycles (0 LDS bank conflicts).
// With the conversion ahead of the MFMAs instead of between them it took 0.87 ms. 34,580 rows:
// 2,304 x 768 0.381 ms (hipBLASLt 0.985), 768 x 768 0.147 (0.363), 3,072 x 768 0.505 (1.262), 768 x
// 3,072 0.477 (1.212). Error against 64 bits (2-norm, N(0, 1) times N(0, 0.02)): 3.2e-7 at k = 768, 6.2e-7
// at k = 3,072; fp32 MFMA 5.0e-7 and 7.0e-7 to 9.9e-7 (a k-step adds 16 products before it rounds).
//
// W as split rows (JC_F16X3 layers: pairs made once by jc_split_f16x3, unscaled) skips W's half of the conversion:
// a layer of 34,580 rows whose GEMMs all run so 2.40 ms, with fp32 W 2.45.
#include <type_traits>

#include "jc_common.hpp"
#include "jc_kernels.hpp"
#include "lp_common.hpp"

namespace jc {
namespace {

using namespace lp;

constexpr int kSK = 32;                          // k values per stage
constexpr uint32_t kOutOfRange = 0x80000000u;    // a buffer offset past every range: reads 0
constexpr int kTarget = 2;                       // a row's first stage is scaled to a maximum in [2^2, 2^3)

template <int BM, int BN>
struct alignas(16) SplitLds {
    uint16_t a[2][2][BM * kSK];  // [stage][hi, lo]
    uint16_t w[2][2][BN * kSK];
    int32_t ea[BM], ew[BN];  // minus the rows' scale exponents
};

// element offset of chunk c of row r within one part of a stage
__device__ __forceinline__ uint32_t sswz(uint32_t r, uint32_t c) { return r * kSK + ((c ^ ((r >> 2) & 3)) << 3); }

__device__ __forceinline__ void split_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// One operand's stage in flight: NI items of 8 consecutive values per thread, item i = row
// tid / 4 + i * STEP, chunk tid % 4. sc: the row's scale 2^p, 0 while all its values were zero.
template <int NI, int STEP>
struct Operand {
    floatx4 x0[NI], x1[NI];
    float sc[NI];
    bool pending;  // some row of the wave has no scale yet (the same in every lane)

    __device__ __forceinline__ void init() {
        pending = true;
#pragma unroll
        for (int i = 0; i < NI; i++) sc[i] = 0.f;
    }
    // Stage st of the rows at p (`rows` of them, k values each): one descriptor per item, its base at the
    // stage's first value, so the lane's offset never changes. Nothing is in range past the last stage,
    // nor in the second half of a last stage of 16 values.
    __device__ __forceinline__ void load(const float* p, int rows, uint32_t row_bytes, uint32_t tid, int st, int stages, int k) {
        const uint32_t half = (st == stages - 1 && (k & 16)) ? kOutOfRange : 0u;
        const uint32_t t = tid;
        const uint32_t o = ((t / 4) * row_bytes + 32u * (t % 4)) | (t << 30 & half);
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int left = st < stages ? rows - i * STEP : 0;
            const uint32_t bytes = left > 0 ? (uint32_t)(left - 1) * row_bytes + (uint32_t)(k - st * kSK) * 4u : 0u;
            const char* base = reinterpret_cast<const char*>(p) + (size_t)i * STEP * row_bytes + (size_t)st * kSK * 4;
            const __amdgpu_buffer_rsrc_t rs = make_rsrc(base, bytes);
            x0[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
            x1[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, o + 16, 0, 0));
        }
    }
    // Gives a scale to the rows whose first nonzero values are in this stage (the stages before were
    // zero, so the accumulators hold nothing of the row yet).
    __device__ __forceinline__ void set_scales() {
        if (!pending) return;
        bool unset = false;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            float m = 0.f;
#pragma unroll
            for (int u = 0; u < 4; u++) m = fmaxf(m, fmaxf(fabsf(x0[i][u]), fabsf(x1[i][u])));
            m = fmaxf(m, quad_perm<0xB1>(m));  // the row's four chunks: lanes 4r .. 4r + 3
            m = fmaxf(m, quad_perm<0x4E>(m));
            if (sc[i] == 0.f && m > 0.f) {
                // the exponent field of 2^(kTarget - floor(log2 m)), where its inverse is normal too
                const int f = min(max(254 + kTarget - (int)(__float_as_uint(m) >> 23), 2), 252);
                sc[i] = __uint_as_float((uint32_t)f << 23);
            }
            unset |= sc[i] == 0.f;
        }
        pending = __any(unset);
    }
    template <int N>
    __device__ __forceinline__ void store(uint16_t (&part)[2][N], uint32_t tid, int i0 = 0, int i1 = NI) {
        const uint32_t t = tid;
#pragma unroll
        for (int i = i0; i < i1; i++) {
            halfx8 hi, lo;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float v = u < 4 ? x0[i][u & 3] : x1[i][u & 3];
                hi[u] = (_Float16)__builtin_fmaf(v, sc[i], 0.f);
                lo[u] = (_Float16)__builtin_fmaf(v, sc[i], -(float)hi[u]);
            }
            const uint32_t o = sswz(t / 4, t % 4) + i * STEP * kSK;  // STEP is a multiple of 16 rows
            *reinterpret_cast<halfx8*>(&part[0][o]) = hi;
            *reinterpret_cast<halfx8*>(&part[1][o]) = lo;
        }
    }
    __device__ __forceinline__ void finish(int32_t* e, uint32_t tid) const {
        if (tid % 4) return;
#pragma unroll
        for (int i = 0; i < NI; i++) e[tid / 4 + i * STEP] = sc[i] != 0.f ? 127 - (int)(__float_as_uint(sc[i]) >> 23) : 0;
    }
};

// W's rows as jc_split_f16x3 wrote them ([hi | lo | hi], 3k fp16 values; the third part is not read): the pairs
// pass to the stage as they are, with no scale. The interface is Operand's.
template <int NI, int STEP>
struct SplitOperand {
    halfx8 hi[NI], lo[NI];

    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ void load(const _Float16* p, int rows, uint32_t row_bytes, uint32_t tid, int st, int stages, int k) {
        const uint32_t half = (st == stages - 1 && (k & 16)) ? kOutOfRange : 0u;
        const uint32_t t = tid;
        const uint32_t o = ((t / 4) * row_bytes + 16u * (t % 4)) | (t << 30 & half);
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int left = st < stages ? rows - i * STEP : 0;
            const uint32_t bytes = left > 0 ? (uint32_t)(left - 1) * row_bytes + (uint32_t)(k - st * kSK) * 2u : 0u;
            const char* base = reinterpret_cast<const char*>(p) + (size_t)i * STEP * row_bytes + (size_t)st * kSK * 2;
            hi[i] = __builtin_bit_cast(halfx8, __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(base, bytes), o, 0, 0));
            lo[i] = __builtin_bit_cast(halfx8, __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(base + (size_t)k * 2, bytes), o, 0, 0));
        }
    }
    __device__ __forceinline__ void set_scales() {}
    template <int N>
    __device__ __forceinline__ void store(uint16_t (&part)[2][N], uint32_t tid, int i0 = 0, int i1 = NI) {
        const uint32_t t = tid;
#pragma unroll
        for (int i = i0; i < i1; i++) {
            const uint32_t o = sswz(t / 4, t % 4) + i * STEP * kSK;
            *reinterpret_cast<halfx8*>(&part[0][o]) = hi[i];
            *reinterpret_cast<halfx8*>(&part[1][o]) = lo[i];
        }
    }
    __device__ __forceinline__ void finish(int32_t* e, uint32_t tid) const {
        if (tid % 4) return;
#pragma unroll
        for (int i = 0; i < NI; i++) e[tid / 4 + i * STEP] = 0;
    }
};

// XW: g.w holds split rows (SplitOperand) instead of fp32 ones.
template <bool XW, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM * WN * kWave, 2) void gemm_f32_split(const GemmArgs g, uint32_t tiles_n, uint32_t total,
                                                                    int vec) {
    constexpr int kThreads = WM * WN * kWave;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr int kStep = kThreads / 4, NA = BM / kStep, NW = BN / kStep;
    static_assert(BM % kStep == 0 && BN % kStep == 0 && BM <= kThreads && BN <= kThreads, "whole items");
    constexpr int kCols = 32 * TN;  // columns of a wave's block
    static_assert(sizeof(float) * 32 * kCols * WM * WN <= sizeof(uint16_t) * 4 * (BM + BN) * kSK, "epilogue staging");
    __shared__ SplitLds<BM, BN> lds;
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t j = lane % 32, hg = lane / 32;
    const int wm = wave / WN, wn = wave % WN;
    const uint32_t tile = xcd_remap(blockIdx.x, total);
    const int m0 = (int)(tile / tiles_n) * BM, n0 = (int)(tile % tiles_n) * BN;
    const int stages = (g.k + kSK - 1) / kSK;

    using WT = std::conditional_t<XW, _Float16, float>;
    const size_t ldw = (XW ? 3 : 1) * (size_t)g.k;  // a row of W, in its own elements
    const float* pa = g.a + (size_t)m0 * g.lda;
    const WT* pw = reinterpret_cast<const WT*>(g.w) + (size_t)n0 * ldw;
    const int rows_a = min(BM, g.m - m0), rows_w = min(BN, g.n - n0);
    Operand<NA, kStep> oa;
    std::conditional_t<XW, SplitOperand<NW, kStep>, Operand<NW, kStep>> ow;
    oa.init();
    ow.init();
    const uint32_t a_row = (uint32_t)g.lda * 4u, w_row = (uint32_t)(ldw * sizeof(WT));
    oa.load(pa, rows_a, a_row, tid, 0, stages, g.k);
    ow.load(pw, rows_w, w_row, tid, 0, stages, g.k);
    floatx16 acc[TM][TN];
#pragma unroll
    for (int ti = 0; ti < TM; ti++)
#pragma unroll
        for (int tj = 0; tj < TN; tj++) acc[ti][tj] = floatx16{0};
    oa.set_scales();
    oa.store(lds.a[0], tid);
    oa.load(pa, rows_a, a_row, tid, 1, stages, g.k);
    ow.set_scales();
    ow.store(lds.w[0], tid);
    ow.load(pw, rows_w, w_row, tid, 1, stages, g.k);
    split_barrier();

    for (int st = 0; st < stages; st++) {
        const int buf = st & 1;
        halfx8 ah[TM], al[TM], wh[TN], wl[TN];
        auto read_a = [&](int kk, int part, halfx8* v) __attribute__((always_inline)) {
            const uint32_t l = lane, o = sswz(32 * TM * wm + l % 32, 2 * kk + l / 32);
#pragma unroll
            for (int ti = 0; ti < TM; ti++)
                v[ti] = *reinterpret_cast<const halfx8*>(&lds.a[buf][part][o + 32 * ti * kSK]);
        };
        auto read_w = [&](int kk, int part, halfx8* v) __attribute__((always_inline)) {
            const uint32_t l = lane, o = sswz(kCols * wn + l % 32, 2 * kk + l / 32);
#pragma unroll
            for (int tj = 0; tj < TN; tj++)
                v[tj] = *reinterpret_cast<const halfx8*>(&lds.w[buf][part][o + 32 * tj * kSK]);
        };
        // one term's TM x TN MFMAs, with what else this phase holds spread between them
        auto products = [&](const halfx8* av, const halfx8* wv) __attribute__((always_inline)) {
#pragma unroll
            for (int ti = 0; ti < TM; ti++)
#pragma unroll
                for (int tj = 0; tj < TN; tj++)
                    acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[ti], wv[tj], acc[ti][tj], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TM * TN; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 16 / (TM * TN) + 1, 0);  // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        read_a(0, 0, ah);
        read_w(0, 1, wl);
        // Three phases per k-step, one per term, each reading the next phase's operands; ah is free after
        // the second, so the third can read the next k-step's. The next stage's A (loaded a stage ago) is
        // split into the other buffer beside the first k-step, its W beside the second.
        oa.set_scales();
        read_w(0, 0, wh);
        oa.store(lds.a[buf ^ 1], tid, 0, (NA + 1) / 2);
        products(ah, wl);
        read_a(0, 1, al);
        oa.store(lds.a[buf ^ 1], tid, (NA + 1) / 2, NA);
        products(ah, wh);
        read_a(1, 0, ah);
        read_w(1, 1, wl);
        oa.load(pa, rows_a, a_row, tid, st + 2, stages, g.k);
        products(al, wh);
        ow.set_scales();
        read_w(1, 0, wh);
        ow.store(lds.w[buf ^ 1], tid, 0, (NW + 1) / 2);
        products(ah, wl);
        read_a(1, 1, al);
        ow.store(lds.w[buf ^ 1], tid, (NW + 1) / 2, NW);
        products(ah, wh);
        ow.load(pw, rows_w, w_row, tid, st + 2, stages, g.k);
        products(al, wh);
        split_barrier();
    }
    oa.finish(lds.ea, tid);
    ow.finish(lds.ew, tid);
    split_barrier();

    // Epilogue, 32 rows of the wave's block at a time: unscale in the accumulator layout, recompute
    // tiles with a value that is not finite, then through the wave's own part of the (now free)
    // stages, so that each lane stores 16 bytes of one row. Bias, activation, accumulate, in
    // Kernels.gemm's order.
    float* ep = reinterpret_cast<float*>(&lds.a[0][0][0]) + wave * (32 * kCols);
    constexpr int kQuads = kCols / 4, kRows = kWave / kQuads;  // lanes per row, rows per instruction
    const int er = lane / kQuads, ec = 4 * (lane % kQuads);
    const int col0 = n0 + kCols * wn + ec;
    floatx4 b4 = floatx4{0.f, 0.f, 0.f, 0.f};
    if (g.flags & kGemmBias) {
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (col0 + u < g.n) b4[u] = g.bias[col0 + u];
    }
    const bool accumulate = g.flags & kGemmAccumulate;
    const bool whole = vec && m0 + BM <= g.m && n0 + BN <= g.n;
#pragma unroll
    for (int ti = 0; ti < TM; ti++) {
        const int rb = 32 * TM * wm + 32 * ti;  // the block's first row within the tile
        int4 ea[4];
#pragma unroll
        for (int q = 0; q < 4; q++) ea[q] = *reinterpret_cast<const int4*>(&lds.ea[rb + 8 * q + 4 * hg]);
#pragma unroll
        for (int tj = 0; tj < TN; tj++) {
            const int cb = kCols * wn + 32 * tj;
            const int ew = lds.ew[cb + j];
            float bad = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int e = (r % 4 == 0 ? ea[r / 4].x : r % 4 == 1 ? ea[r / 4].y : r % 4 == 2 ? ea[r / 4].z : ea[r / 4].w) + ew;
                acc[ti][tj][r] = __builtin_amdgcn_ldexpf(acc[ti][tj][r], e);
                bad = __builtin_fmaf(acc[ti][tj][r], 0.f, bad);
            }
            if (__any(bad != bad)) {
                // on fp32 MFMA from the operands themselves: lane (i, hg) contracts k = 8q + 4hg + u
                // with step u
                const float* ta = g.a + (size_t)min(m0 + rb + j, g.m - 1) * g.lda + 4 * hg;
                const WT* tw = reinterpret_cast<const WT*>(g.w) + (size_t)min(n0 + cb + j, g.n - 1) * ldw + 4 * hg;
                floatx16 t = floatx16{0};
                for (int q = 0; q < g.k; q += 8) {
                    const floatx4 av = *reinterpret_cast<const floatx4*>(ta + q);
                    floatx4 wv;
                    if constexpr (XW) {
#pragma unroll
                        for (int u = 0; u < 4; u++) wv[u] = (float)tw[q + u] + (float)tw[g.k + q + u];
                    } else {
                        wv = *reinterpret_cast<const floatx4*>(tw + q);
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++) t = __builtin_amdgcn_mfma_f32_32x32x2f32(av[u], wv[u], t, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float v = acc[ti][tj][r];
                    acc[ti][tj][r] = v - v == 0.f ? v : t[r];
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int R = 8 * (r / 4) + 4 * hg + r % 4;
                ep[R * kCols + ((32 * tj + j) ^ (TN > 1 ? (R & 4) << 3 : 0))] = acc[ti][tj][r];
            }
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
        floatx4 vv[32 / kRows];
#pragma unroll
        for (int q = 0; q < 32 / kRows; q++) {
            const int R = kRows * q + er;
            vv[q] = *reinterpret_cast<const floatx4*>(&ep[R * kCols + (ec ^ (TN > 1 ? (R & 4) << 3 : 0))]);
        }
        auto finish = [&](floatx4 v) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                v[u] += b4[u];
                if (g.flags & kGemmSilu) v[u] = v[u] / (1.f + __expf(-v[u]));
                if (g.flags & kGemmRelu) v[u] = (v[u] > 0.f || v[u] != v[u]) ? v[u] : 0.f;
            }
            return v;
        };
        if (whole) {
            float* cp = g.c + (size_t)(m0 + rb + er) * g.ldc + col0;
            if (accumulate) {
                floatx4 cv[32 / kRows];
#pragma unroll
                for (int q = 0; q < 32 / kRows; q++)
                    cv[q] = *reinterpret_cast<const floatx4*>(cp + (size_t)(kRows * q) * g.ldc);
#pragma unroll
                for (int q = 0; q < 32 / kRows; q++)
                    *reinterpret_cast<floatx4*>(cp + (size_t)(kRows * q) * g.ldc) = finish(vv[q]) + cv[q];
            } else {
#pragma unroll
                for (int q = 0; q < 32 / kRows; q++)
                    *reinterpret_cast<floatx4*>(cp + (size_t)(kRows * q) * g.ldc) = finish(vv[q]);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 32 / kRows; q++) {
                const floatx4 v = finish(vv[q]);
                const int row = m0 + rb + kRows * q + er;
                if (row >= g.m) continue;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (col0 + u >= g.n) break;
                    float* cp = g.c + (size_t)row * g.ldc + col0 + u;
                    *cp = accumulate ? v[u] + *cp : v[u];
                }
            }
        }
        // this block's reads are issued before the next block's writes (LDS keeps a wave's order)
        asm volatile("" ::: "memory");
    }
}

template <bool XW, int BM, int BN, int WM, int WN>
hipError_t launch_split(const GemmArgs& g, hipStream_t stream) {
    const uint32_t tn = (uint32_t)((g.n + BN - 1) / BN);
    const uint64_t total = (uint64_t)((g.m + BM - 1) / BM) * tn;
    const int vec = g.ldc % 4 == 0 && (size_t)g.c % 16 == 0;
    hipLaunchKernelGGL((gemm_f32_split<XW, BM, BN, WM, WN>), dim3((uint32_t)total), dim3(WM * WN * kWave), 0, stream, g, tn,
                       (uint32_t)total, vec);
    return hipGetLastError();
}

// The three tile sizes, and the time of one round of each (all CUs holding a tile, 1, 2 or 4 a CU) per
// 768 values of k, in microseconds: 256 x 256 76, 128 x 128 47 (34 while half the slots are empty),
// 64 x 64 35 (24). The smallest product of rounds and time wins: the large tiles read each operand
// fewer times and split it less often, the small ones fill the chip on few rows.
struct Tiling {
    int bm, slots;
    float full, half;
};
constexpr Tiling kTilings[3] = {{256, 256, 76.f, 76.f}, {128, 512, 47.f, 34.f}, {64, 1024, 35.f, 24.f}};

float tiling_us(const GemmArgs& g, int cfg) {
    const Tiling& t = kTilings[cfg];
    const uint64_t tiles = (uint64_t)((g.m + t.bm - 1) / t.bm) * (uint64_t)((g.n + t.bm - 1) / t.bm);
    const uint64_t rounds = (tiles + t.slots - 1) / t.slots;
    return (float)rounds * (tiles <= (uint64_t)t.slots / 2 ? t.half : t.full) * (float)g.k / 768.f;
}

int best_tiling(const GemmArgs& g) {
    int best = 0;
    for (int c = 1; c < 3; c++)
        if (tiling_us(g, c) < tiling_us(g, best)) best = c;
    return best;
}

template <bool XW>
hipError_t launch_best(const GemmArgs& g, hipStream_t stream) {
    switch (best_tiling(g)) {
        case 0: return launch_split<XW, 256, 256, 2, 4>(g, stream);
        case 1: return launch_split<XW, 128, 128, 2, 2>(g, stream);
        default: return launch_split<XW, 64, 64, 2, 2>(g, stream);
    }
}

}  // namespace

bool gemm_f32_split_fits(const GemmArgs& g) { return g.lda < (1 << 21) && g.k < (1 << 21); }

bool gemm_f32_split_w_fits(const GemmArgs& g) { return g.lda < (1 << 21) && g.k < (1 << 20); }

float gemm_f32_split_us(const GemmArgs& g) { return tiling_us(g, best_tiling(g)); }

hipError_t gemm_f32_split_launch(const GemmArgs& g, hipStream_t stream) { return launch_best<false>(g, stream); }

hipError_t gemm_f32_split_w_launch(const GemmArgs& g, hipStream_t stream) { return launch_best<true>(g, stream); }

}  // namespace jc
