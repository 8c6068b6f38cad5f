// The fp32 matrix tile on bf16 MFMA that the fp32 GEMM family (gemm_f32.hip) and
// the convolution (conv2d.hip) share.
#pragma once

#include "common.h"

#include <type_traits>

namespace mb {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

enum { BL_KN = 0, BL_NK = 1 };                           // B is [K][N] or [N][K]
enum { EPI_STORE = 0, EPI_RESID = 1, EPI_SWIGLU = 2 };   // C = acc | acc + R | silu(acc) acc2

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }

// ---- fp32 product on bf16 MFMA: every operand as the sum of three bf16 terms ----
// v = h + m + l with h = bf16(v), m = bf16(v - h), l = bf16(v - h - m): 3 x 8
// significant bits hold all 24 of v, so the three terms add up to v exactly,
// unless they leave bf16's range.  The last bit of v = 2^e (1 + ...) has weight
// 2^(e - 23), and bf16 holds multiples of 2^-133, so below 2^-110 the low terms
// would lose bits; every operand is therefore multiplied by SPLIT_SCALE first
// (exact), which lifts the last bit of the smallest fp32 number, 2^-149, to
// 2^-133, and the sums are divided by SPLIT_SCALE^2 at the end (one rounding,
// where the result is subnormal).  What that costs at the other end: a value
// of 2^112 or a sum of 2^96 and more overflows, and is computed otherwise (see
// split_tile).
// A product a b is then the six term products of order 2^0 (ah bh), 2^-9 (ah
// bm, am bh) and 2^-18 (am bm, ah bl, al bh) relative to it; the three left
// out (am bl, al bm, al bl) are below 2^-26, under the rounding of an fp32
// accumulation.  (The decomposition of Henry, Tang and Heinecke, "Leveraging
// the bfloat16 artificial intelligence datatype for higher-precision
// computations", 2019.)  Six v_mfma_f32_32x32x16_bf16 take 192 cycles where
// eight v_mfma_f32_32x32x2f32 take 512.
constexpr float SPLIT_SCALE = 0x1p16f;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct Split8 { u32x4 h, m, l; };   // eight values, one bf16 term of each in every half word

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ void split2(float a, float b, Split8& o, int p) {   // values 2 p, 2 p + 1
    a *= SPLIT_SCALE;
    b *= SPLIT_SCALE;
    const uint32_t h = pack_bf16(a, b);
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    const uint32_t m = pack_bf16(ra, rb);
    o.h[p] = h;
    o.m[p] = m;
    o.l[p] = pack_bf16(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
}
__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// One workgroup computes a 64 x 64 tile (SwiGLU: 64 x 32 of gate and of up)
// with four waves that divide K: unit u = k 16 u .. 16 u + 15 belongs to wave
// u % 4, and each wave multiplies the whole tile over its units, so the waves
// share nothing and the K loop has no barrier.  Per unit a wave
//  * fetches A (64 rows x 64 bytes, by the caller's dma_a) and B (16 k-rows x 256
//    bytes) by DMA into its own two LDS slots of 8 KB.  (Loaded straight into the MFMA layout, a
//    quad of lanes touches four rows of A: 20.7 us at 1024^3 on 17.7.)
//    16-byte chunk c of A row r sits in slot c ^ ((r / 4) % 4), so that 16
//    lanes reading 16 rows touch 16 distinct bank groups;
//  * reads unit t+2 into registers, splits unit t+1 (208 vector instructions)
//    and runs the 24 MFMAs of unit t in one straight-line block; a
//    v_mfma_f32_32x32x16_bf16 hides six of the split's instructions (a
//    16x16x32 two, and each one more costs four cycles).  32 of the 208 are
//    the scaling: 1024^3 14.4 -> 14.6 us, 2048^3 97.4 -> 99.2, 512 x 512 x 2048
//    20.8 -> 22.0, 32x56x56x64 3x3 convolution 55.8 -> 56.4 (a check of the
//    operands for small values would have to look at every element as well).
// 229 registers and 64 KB of LDS: two workgroups per CU, whose instructions
// interleave (one wave alone issues one per four to five cycles: 17.7 us at
// 1024^3) and whose first fetches and last sums overlap.  With eight waves per
// workgroup and one workgroup per CU: 15.4 us at 1024^3 and 27.0 at 2048 x
// 2048 x 256; as here 14.4 and 19.6 (17.8 and 24.5 on fp32 MFMA).  What
// bounds a long K is power: at 1024 x 1024 x 4096 zeros run in 35 us and
// uniform operands in 51 (without the split's instructions 40, without DMA 44).
// The operand layout in k is lane half h = k 4 h .. 4 h + 3 and 8 + 4 h ..
// 8 + 4 h + 3 of a unit, for A and B alike.  The waves' four partial tiles are
// added through LDS in wave order.
// Any shape and alignment: rows past M read row M - 1, and what lies past the
// end of an operand reads as zero (a raw buffer checks every dword); results
// past the output are not stored.  k past K is zero in B, and masked in A.
// The split cannot hold an infinity (inf - inf) nor what SPLIT_SCALE lifts past
// the largest number: a tile with a sum that is not finite is computed again by
// v_mfma_f32_32x32x2f32 from the unsplit, unscaled operands.  That second pass
// takes as long as a product on fp32 MFMA: 1024^3 with an infinity in one row of
// A 32.7 us (its row of tiles twice, the others waiting for it), 2048^3 with
// all sums past 2^96 222 us (99; 133 on fp32 MFMA alone).
// 1021 x 1531 x 2043: 47 us (138 with element-wise loads on fp32 MFMA); 2048^3
// 99 us (133); 1024 x 2048 x 4096 97 us (127); all launches back to back on one
// set of operands.
constexpr uint32_t SP_BAND = 4;          // tile-rows per XCD band (xcd_band_tile)
constexpr int SP_W = 4;                 // waves per workgroup
constexpr uint32_t SP_SLOT = 8192;       // one unit of A and B
constexpr uint32_t SP_WAVE = 2 * SP_SLOT;

struct SplitTile {
    const float *b, *b2, *r;   // B (and SwiGLU's second one), the residual
    float* c;
    uint32_t m, n, k, ldb, ldc, ldr;
    uint32_t m0, n0;           // the tile's first row and column
    float eps;
};

// dma_a(lds, u) issues the NA DMA instructions that land A's unit u (zeros past K
// or the next row's values, which are masked here) at `lds`.
template <int BL, int EPI, bool RMS, int NA, class DmaA>
__device__ __forceinline__ void split_tile(const SplitTile& g, DmaA dma_a) {
    constexpr bool DUAL = EPI == EPI_SWIGLU;
    __shared__ __attribute__((aligned(1024))) uint8_t L[SP_W * SP_WAVE];
    __shared__ float rss[SP_W][64];      // RMS: wave, row
    __shared__ uint32_t flag[SP_W];

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t li = lane & 31, lh = lane >> 5;
    const uint32_t m0 = g.m0, n0 = g.n0;
    const uint32_t M = g.m, N = g.n, K = g.k, ldb = g.ldb;
    const float *B = g.b, *B2 = DUAL ? g.b2 : g.b;
    float* C = g.c;
    auto extent = [](uint32_t rows, uint32_t ld, uint32_t cols) {   // bytes up to the last element
        return rows && cols ? ((rows - 1) * ld + cols) * 4 : 0;
    };
    const uint32_t b_bytes = BL == BL_KN ? extent(K, ldb, N) : extent(N, ldb, K);
    const i32x4 brs = dma_rsrc(B, b_bytes), b2rs = dma_rsrc(B2, b_bytes);

    // DMA instruction i of a unit: B^T rows 16 i + lane / 4, slot lane % 4; B k-rows 4 i + lane / 16 (DUAL: LDS row 8 (i % 2) + lane / 8 of
    // gate, then up; k-row r sits in row r ^ ((r / 4) % 2), so that the k-rows
    // of the two half-waves, r and r + 4, lie in opposite halves of the banks).
    // k-rows past K lie past the end of B, and are at most 15: under 2^32 bytes
    // together with K < 2^31 / (4 ldb) of them when K is 16 or more.  With K
    // below 16 a row of very many columns would wrap around, and takes an
    // out-of-range offset.
    uint32_t b_vo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t r = 16 * i + (lane >> 2), ch = (lane & 3) ^ (lane >> 4);
        if (BL == BL_NK) b_vo[i] = (min(n0 + r, N - 1) * ldb + 4 * ch) * 4;
        else if (DUAL) {
            const uint32_t p = 8 * (i & 1) + (lane >> 3);
            const uint32_t k = p ^ ((p >> 2) & 1);
            b_vo[i] = k < K ? (k * ldb + n0 + 4 * (lane & 7)) * 4 : 0x80000000u;
        } else {
            const uint32_t k = 4 * i + (lane >> 4);
            b_vo[i] = k < K ? (k * ldb + n0 + 4 * (lane & 15)) * 4 : 0x80000000u;
        }
    }
    // the wave takes units u = wave (mod SP_W), last first
    const uint32_t units = (K + 15) / 16;
    const uint32_t n = units > wave ? (units - wave + SP_W - 1) / SP_W : 0;
    const uint32_t u_top = wave + SP_W * (n - 1);   // (n > 0)
    const uint32_t l0 = lds_addr(L) + wave * SP_WAVE;
    auto dma = [&](uint32_t slot, uint32_t j) {   // the wave's j-th unit
        const uint32_t u = u_top - SP_W * j;
        const uint32_t b_so = BL == BL_NK ? u * 64 : u * 64 * ldb;
        dma_a(l0 + slot, u);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            dma16(DUAL && i >= 2 ? b2rs : brs, l0 + slot + 4096 + 1024 * i, b_vo[i], b_so);
    };

    struct Raw { float a[2][8], b[2][8]; };
    struct Ops { Split8 a[2], b[2]; };
    const uint8_t* lw = L + wave * SP_WAVE;
    const uint32_t sw = (li >> 2) & 3;
    const uint32_t a_rd[2] = {64 * li + 16 * (lh ^ sw), 64 * li + 16 * ((2 + lh) ^ sw)};
    const uint32_t b_rd = DUAL ? 4 * li : 1024 * lh + 8 * li;
    auto read = [&](Raw& r, uint32_t slot) {
        const uint8_t* s = lw + slot;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float4 v = *reinterpret_cast<const float4*>(s + a_rd[q] + 2048 * i);
                r.a[i][4 * q] = v.x; r.a[i][4 * q + 1] = v.y; r.a[i][4 * q + 2] = v.z; r.a[i][4 * q + 3] = v.w;
                if (BL == BL_NK) {
                    const float4 w = *reinterpret_cast<const float4*>(s + 4096 + a_rd[q] + 2048 * i);
                    r.b[i][4 * q] = w.x; r.b[i][4 * q + 1] = w.y; r.b[i][4 * q + 2] = w.z; r.b[i][4 * q + 3] = w.w;
                }
            }
        if (BL == BL_KN)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = 8 * (e >> 2) + (e & 3);
                if (DUAL) {
                    const uint32_t p = (k + 4 * lh) ^ lh;   // LDS row of k-row k + 4 lh
                    r.b[0][e] = *reinterpret_cast<const float*>(s + 4096 + 128 * p + b_rd);
                    r.b[1][e] = *reinterpret_cast<const float*>(s + 6144 + 128 * p + b_rd);
                } else {
                    const float2 v = *reinterpret_cast<const float2*>(s + 4096 + 256 * k + b_rd);
                    r.b[0][e] = v.x;
                    r.b[1][e] = v.y;
                }
            }
    };
    auto mask_top = [&](Raw& r) {   // the wave's first unit may end past K
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (u_top * 16 + 8 * (e >> 2) + 4 * lh + (e & 3) >= K)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    r.a[i][e] = 0.f;
                    if (BL == BL_NK) r.b[i][e] = 0.f;
                }
    };

    f32x16 acc[2][2];
    float ss[2];        // RMS: row sums of squares of the units multiplied so far,
    float ss_next[2];   // and of the unit split last (added when it is multiplied)
    auto split = [&](const Raw& r, Ops& o) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ss_next[i] = 0.f;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                split2(r.a[i][2 * p], r.a[i][2 * p + 1], o.a[i], p);
                split2(r.b[i][2 * p], r.b[i][2 * p + 1], o.b[i], p);
                if (RMS) ss_next[i] = fmaf(r.a[i][2 * p], r.a[i][2 * p],
                                           fmaf(r.a[i][2 * p + 1], r.a[i][2 * p + 1], ss_next[i]));
            }
        }
    };
    // keeps the terms where they are computed (the compiler would otherwise
    // move them behind the stage's branch, out of the MFMAs' shadow)
    auto pin = [](Ops& o) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            asm volatile("" : "+v"(o.a[i].h), "+v"(o.a[i].m), "+v"(o.a[i].l), "+v"(o.b[i].h),
                         "+v"(o.b[i].m), "+v"(o.b[i].l) :: "memory");
    };
    auto mfma = [&](const Ops& o) {
#pragma unroll
        for (int t = 0; t < 6; ++t)   // small terms first
#pragma unroll
            for (int ij = 0; ij < 4; ++ij) {
                const int i = ij >> 1, j = (ij & 1) ^ i;
                const Split8 &x = o.a[i], &y = o.b[j];
                acc[i][j] = mfma_bf16(t == 0 ? x.l : t == 2 || t == 3 ? x.m : x.h,
                                      t == 1 ? y.l : t == 2 || t == 4 ? y.m : y.h, acc[i][j]);
            }
    };
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ss[i] = 0.f;
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
        }
    };
    // The four waves' partials meet in LDS, each in its wave's own ring.
    // Wave w finishes 64 / SP_W rows of both column blocks.  `scaled`: the sums are
    // those of split operands; true in every thread, with nothing stored, if one of
    // the tile's is not finite.
    auto finish = [&](bool scaled) -> bool {
        auto part = [&](uint32_t w) { return reinterpret_cast<float*>(L + w * SP_WAVE); };
#pragma unroll
        for (int ij = 0; ij < 4; ++ij)
#pragma unroll
            for (int q = 0; q < 16; ++q) part(wave)[(16 * ij + q) * 64 + lane] = acc[ij >> 1][ij & 1][q];
        if (RMS) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float t = ss[i] + __shfl_xor(ss[i], 32);
                if (lh == 0) rss[wave][32 * i + li] = t;
            }
        }
        __syncthreads();
        constexpr int QN = 32 / SP_W;   // accumulator registers finished per wave and block
        const uint32_t i = wave / (SP_W / 2), q0 = QN * (wave % (SP_W / 2));
        float v[2][QN];
        bool odd = false;
#pragma unroll
        for (int q = 0; q < QN; ++q) {
            const uint32_t gr = m0 + 32 * i + 8 * ((q0 + q) >> 2) + 4 * lh + (q & 3);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t at = (32 * i + 16 * j + q0 + q) * 64 + lane;
                float t = part(0)[at];
#pragma unroll
                for (int w = 1; w < SP_W; ++w) t += part(w)[at];
                v[j][q] = t;
                const uint32_t gc = DUAL ? n0 + li : BL == BL_NK ? n0 + 32 * j + li : n0 + 2 * li + j;
                odd |= (gr < M) & (gc < N) & !(fabsf(t) <= 3.402823466e38f);
            }
        }
        if (scaled) {
            const bool any = __builtin_amdgcn_ballot_w64(odd) != 0;
            if (lane == 0) flag[wave] = any;
            __syncthreads();
            uint32_t f = 0;
#pragma unroll
            for (int w = 0; w < SP_W; ++w) f |= flag[w];
            if (f) return true;
        }
        // rows and columns past the output take an out-of-range offset
        auto rsrc = [](const float* p, uint32_t bytes) {
            return __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(p), 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000u);
        };
        // (from the tile's first row, so that C and R may pass 4 GB)
        const uint32_t rows = min(M - m0, 64u);
        const __amdgpu_buffer_rsrc_t crs = rsrc(C + (size_t)m0 * g.ldc, extent(rows, g.ldc, N));
        const __amdgpu_buffer_rsrc_t rrs =
            EPI == EPI_RESID ? rsrc(g.r + (size_t)m0 * g.ldr, extent(rows, g.ldr, N)) : crs;
#pragma unroll
        for (int q = 0; q < QN; ++q) {
            const uint32_t lr = 32 * i + 8 * ((q0 + q) >> 2) + 4 * lh + (q & 3), gr = m0 + lr;
            float sc = scaled ? 1.0f / (SPLIT_SCALE * SPLIT_SCALE) : 1.0f;
            if (RMS) {
                float t = 0.f;
#pragma unroll
                for (int w = 0; w < SP_W; ++w) t += rss[w][lr];
                sc *= rsqrtf(t / (float)K + g.eps);
            }
#pragma unroll
            for (int j = 0; j < (DUAL ? 1 : 2); ++j) {
                const uint32_t gc = DUAL ? n0 + li : BL == BL_NK ? n0 + 32 * j + li : n0 + 2 * li + j;
                const bool in = (gr < M) & (gc < N);
                float out = v[j][q] * sc;
                if (DUAL) out = silu_f(out) * (v[1][q] * sc);
                if (EPI == EPI_RESID)
                    out += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rrs, in ? (lr * g.ldr + gc) * 4 : 0x80000000u, 0, 0));
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(out), crs,
                                                      in ? (lr * g.ldc + gc) * 4 : 0x80000000u, 0, 0);
            }
        }
        return false;
    };

    clear();
    if (n > 0) {
        Raw r[2];
        Ops o[2];
        dma(0, 0);
        if (n > 1) {
            dma(SP_SLOT, 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA + 4) : "memory");   // unit 0 has landed
        } else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        read(r[0], 0);
        mask_top(r[0]);
        split(r[0], o[0]);
        pin(o[0]);
        if (n > 2) {
            dma(0, 2);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA + 4) : "memory");
        } else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        read(r[1], SP_SLOT);
        // stage t multiplies unit t, splits unit t + 1 and reads unit t + 2;
        // unit t + 1's slot (its reads have ended) takes unit t + 3
        auto stage = [&](auto c_, uint32_t t) {
            constexpr int c = decltype(c_)::value;
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            if (t + 3 < n) dma((c ^ 1) * SP_SLOT, t + 3);
            __builtin_amdgcn_sched_barrier(0);
            read(r[c], c * SP_SLOT);
            if (RMS) { ss[0] += ss_next[0]; ss[1] += ss_next[1]; }
            split(r[c ^ 1], o[c ^ 1]);
            mfma(o[c]);
            pin(o[c ^ 1]);
#pragma unroll
            for (int x = 0; x < 24; ++x) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        uint32_t t = 0;
        for (; t + 1 < n; t += 2) {
            stage(std::integral_constant<int, 0>{}, t);
            stage(std::integral_constant<int, 1>{}, t + 1);
        }
        if (t < n) stage(std::integral_constant<int, 0>{}, t);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the ring becomes the partial sums' place
    }
    if (!finish(true)) return;

    clear();
    __syncthreads();   // the partials are read: their LDS is free
    for (uint32_t t = 0; t < n; ++t) {
        Raw r;
        dma(0, t);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        read(r, 0);
        if (t == 0) mask_top(r);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (RMS) ss[i] = fmaf(r.a[i][e], r.a[i][e], ss[i]);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(r.a[i][e], r.b[j][e],
                                                                     acc[i][j], 0, 0, 0);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot's reads have ended
    }
    finish(false);
}

}  // namespace
}  // namespace mb
