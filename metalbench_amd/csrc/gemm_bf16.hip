// bf16 GEMM C[M][N] = bf16(A[M][K] @ B[K][N]), fp32 accumulation, on bf16 MFMA.
//
// No reference kernel: the reference has no bf16 (its dtype tables stop at
// f32/f16/i32/u32, reference mlx/scripts/mlx_helpers.py:83-89).  The spec is
// the reference's matmul (mlx/kernels/common/sqr_mm.py:10-11; registry
// helper mlx/kernels/common/registry.py:43-59: A@0, B@1, C@2, M@3, N@4, K@5)
// at bf16, rounded to bf16 (round to nearest even) once, from fp32.
//
// gfx950 design (MFMA bound: 2*M*N*K flops vs 2*(MK+KN+MN) bytes):
//  * workgroup tile 256x256, 4 waves in a 2x2 grid, each wave a 128x128
//    sub-tile (256 fp32 accumulators per lane, held in AccVGPRs); one
//    workgroup per CU, 1024 tiles at 8192^3 = exactly four rounds of 256 CUs;
//  * full tiles (the large_mm shape) take gemm_bf16_full_kernel further down:
//    8 x 8 v_mfma_f32_16x16x32_bf16 per wave and 32-deep k stage, both
//    operands global -> LDS by DMA (no staging registers, no LDS store
//    instructions) into rings that fill all 160 KB of LDS (A in 64-deep
//    slots of whole 128-byte lines, B in 32-deep slots), B transposed by the
//    LDS reads (ds_read_b64_tr_b16);
//  * other shapes take the cheapest of k_tiles: the same kernel with guarded
//    edges, gemm_bf16_tile_kernel (32 MB x 32 NB tiles), for a small C
//    gemm_bf16_kwave_kernel (16 MB x 16 NC tiles, K dealt to four waves), or, for a
//    large C of unaligned rows and a short K, gemm_bf16_kernel below.  A 256 x 256
//    tile leaves CUs idle below 256 tiles, and unaligned rows were loaded element
//    by element: 1000 x 3000 x 4096 159 -> 36 us, 1001 x 3001 x 4095 457 -> 71,
//    128 x 4096 x 4096 148 -> 15, 64 x 512 x 4096 142 -> 7.4;
//  * operands or results past 2 GB that are not full tiles, a C off a 4-byte boundary
//    likewise, more than 16 million columns with K < 128, and K = 0 take
//    gemm_bf16_kernel (4 x 4 v_mfma_f32_32x32x16_bf16 per wave), BK = 64 with an LDS
//    double buffer:
//    both operands stored K-contiguous, row pitch 72 bf16 (144 B), 2 x 2 x
//    36 KB = 144 KB of the 160 KB.  With that pitch the MFMA operand reads
//    (ds_read_b128 of 16 consecutive rows) and both store patterns below
//    touch distinct bank groups.  A is row-major [M][K], already
//    K-contiguous: 16-byte global loads go straight to LDS rows.  B is
//    row-major [K][N] (N-contiguous), but the MFMA B operand wants 8
//    consecutive k per lane: each lane loads an 8(k) x 8(n) block as eight
//    16-byte rows, transposes it in registers with 32 v_perm_b32 (pairing k
//    and k+1 halves into dwords) and stores eight K-contiguous 16-byte rows.
//    Global loads of stage s+1 are issued before the MFMAs of stage s, and
//    the LDS operand reads of k-step kk+1 are in flight during the MFMAs of kk.
//    Guarded loads (zero fill) and stores; K % 8 or N % 8 != 0 element-wise;
//  * XCD-aware tile order: hardware dispatches block b to XCD b % 8, so the
//    block id is remapped so that each XCD walks one band of GM = 4 tile-rows
//    in column order; the 32 tiles one XCD runs at a time share 4 A panels and
//    8 B panels in that XCD's L2.
#include "common.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace mb {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 256, BN = 256, BK = 64;
constexpr int PITCH = BK + 8;             // bf16 per LDS row (144 B)
constexpr int TILE_ELEMS = BM * PITCH;    // per operand per stage
constexpr int GM = 4;                     // tile-rows per XCD band

enum { MODE_GUARD = 1, MODE_ELEM = 2 };

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);   // quiet NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ void tile_coords(uint32_t b, uint32_t nblocks, uint32_t tiles_m,
                                            uint32_t tiles_n, uint32_t* tm, uint32_t* tn) {
    xcd_band_tile(b, nblocks, tiles_m, tiles_n, GM, tm, tn);
}

template <int MODE>
__global__ __launch_bounds__(256, 1)
void gemm_bf16_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                      uint16_t* __restrict__ C, uint32_t M, uint32_t N, uint32_t K,
                      uint32_t tiles_m, uint32_t tiles_n) {
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    uint16_t* As = smem;                       // [2][BM][PITCH]
    uint16_t* Bs = smem + 2 * TILE_ELEMS;      // [2][BN][PITCH]

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = tid >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1;
    uint32_t tm, tn;
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, &tm, &tn);
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t nstages = (K + BK - 1) / BK;

    // A loader: row = tid/8 + 32*i, 16-byte chunk = tid%8.
    // B loader: k-octet ko = tid%8, n-octet no = tid/8 (8 rows of 16 B each).
    const uint32_t a_row = tid >> 3, a_chunk = tid & 7;
    const uint32_t b_ko = tid & 7, b_no = tid >> 3;

    u32x4 ra[8], rb[8];

    auto load = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t gm = m0 + a_row + 32 * i, gk = k0 + 8 * a_chunk;
            const uint16_t* p = A + (size_t)gm * K + gk;
            if (MODE == MODE_GUARD) {
                ra[i] = (gm < M && gk < K) ? *reinterpret_cast<const u32x4*>(p) : u32x4{};
            } else {
                uint16_t e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = (gm < M && gk + j < K) ? p[j] : (uint16_t)0;
                ra[i] = u32x4{e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16,
                              e[4] | (uint32_t)e[5] << 16, e[6] | (uint32_t)e[7] << 16};
            }
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t gk = k0 + 8 * b_ko + r, gn = n0 + 8 * b_no;
            const uint16_t* p = B + (size_t)gk * N + gn;
            if (MODE == MODE_GUARD) {
                rb[r] = (gk < K && gn < N) ? *reinterpret_cast<const u32x4*>(p) : u32x4{};
            } else {
                uint16_t e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = (gk < K && gn + j < N) ? p[j] : (uint16_t)0;
                rb[r] = u32x4{e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16,
                              e[4] | (uint32_t)e[5] << 16, e[6] | (uint32_t)e[7] << 16};
            }
        }
    };

    auto store = [&](int buf) {
        uint16_t* as = As + buf * TILE_ELEMS;
        uint16_t* bs = Bs + buf * TILE_ELEMS;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            *reinterpret_cast<u32x4*>(as + (a_row + 32 * i) * PITCH + 8 * a_chunk) = ra[i];
        // 8x8 transpose: column c of the block = n0 + 8*no + c gets k = 8*ko .. +7.
        // Dword j of column c pairs (k = 2j, 2j+1): lo halves for even c, hi for odd.
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t e = rb[2 * j][m];
                const uint32_t o = rb[2 * j + 1][m];
                lo[j] = __builtin_amdgcn_perm(o, e, 0x05040100u);
                hi[j] = __builtin_amdgcn_perm(o, e, 0x07060302u);
            }
            *reinterpret_cast<u32x4*>(bs + (8 * b_no + 2 * m) * PITCH + 8 * b_ko) =
                u32x4{lo[0], lo[1], lo[2], lo[3]};
            *reinterpret_cast<u32x4*>(bs + (8 * b_no + 2 * m + 1) * PITCH + 8 * b_ko) =
                u32x4{hi[0], hi[1], hi[2], hi[3]};
        }
    };

    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};

    const uint32_t li = lane & 31, lh = lane >> 5;

    if (nstages > 0) {
        load(0);
        store(0);
        __syncthreads();
    }
    for (uint32_t s = 0; s < nstages; ++s) {
        const int cur = s & 1;
        if (s + 1 < nstages) load((s + 1) * BK);
        const uint16_t* as = As + cur * TILE_ELEMS + (wm * 128 + li) * PITCH + 8 * lh;
        const uint16_t* bs = Bs + cur * TILE_ELEMS + (wn * 128 + li) * PITCH + 8 * lh;
        // Operands of k-step kk+1 are read from LDS while the 16 MFMAs of kk run.
        bf16x8 a[2][4], b[2][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[0][i] = *reinterpret_cast<const bf16x8*>(as + 32 * i * PITCH);
#pragma unroll
        for (int j = 0; j < 4; ++j) b[0][j] = *reinterpret_cast<const bf16x8*>(bs + 32 * j * PITCH);
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            const int c = kk & 1;
            if (kk + 1 < BK / 16) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    a[c ^ 1][i] = *reinterpret_cast<const bf16x8*>(as + 32 * i * PITCH + 16 * (kk + 1));
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    b[c ^ 1][j] = *reinterpret_cast<const bf16x8*>(bs + 32 * j * PITCH + 16 * (kk + 1));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c][i], b[c][j], acc[i][j],
                                                                         0, 0, 0);
        }
        if (s + 1 < nstages) store(cur ^ 1);
        __syncthreads();
    }

    // Epilogue: lane l, reg r of a 32x32 block -> row 8*(r/4) + 4*(l/32) + r%4, col l%32.
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t gc = n0 + wn * 128 + 32 * j + li;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t gr = m0 + wm * 128 + 32 * i + 8 * (r >> 2) + 4 * lh + (r & 3);
                if (gr < M && gc < N)
                    C[(size_t)gr * N + gc] = f32_to_bf16_rne(acc[i][j][r]);
            }
        }
}

// ---- full-tile kernel (M, N multiples of 256, K of 128, operands < 2 GiB) ----
// Both operands go global -> LDS by DMA (buffer_load ... lds): no staging
// registers and no LDS store instructions, whose VGPR reads stall the MFMA
// issue.  All 160 KB of LDS hold the operand rings:
//  * A in three 64-deep slots (32 KB each: 256 rows of 128 bytes).  Each A
//    DMA instruction fills 8 whole 128-byte lines (8 rows x 8 chunks); chunk c
//    (8 k) of row r sits in slot c ^ ((r / 2) % 8).  The 16x16x32 A operand of
//    row block i is one ds_read_b128: lane l reads row 16 i + l%16, chunk
//    4 h + l/16 (h = which 32-k half of the slot); each 16 lanes hit 16
//    distinct 16-byte bank groups;
//  * B in four 32-deep slots (16 KB each: [32 k][256 n] row-major as in HBM,
//    512-byte k-rows); chunk c (8 n) of k-row r sits in slot c ^ f(r),
//    f(r) = 4 (r % 4) ^ 2 ((r / 8) % 2).  The B operand (8 consecutive k of one
//    column) is two ds_read_b64_tr_b16: in 16-lane group g lane s points at
//    k-row 8 g + 4 q + s/4, columns n0 + 4 (s % 4) .. +3, and receives column
//    n0 + s, those 4 k-rows.  The ^ 2 ((r/8) % 2) term puts k-rows r and r + 8
//    (groups 0 and 1, read in the same LDS cycle) in different banks;
//  * each DMA instruction writes a wave's 64 x 16 B contiguously, so lane l
//    fetches the global chunk that its slot holds.
// The MFMA is v_mfma_f32_16x16x32_bf16, not 32x32x16: on random bf16 data
// the chip is power-limited, and a register-only loop of 16x16x32 sustains
// 1.90-2.12 PF against 1.50-1.85 PF for 32x32x16 at the same power.
//
// Stage s (32 k; B slot s % 4, operands in register set s % 2): wait for this
// wave's DMAs issued three stages earlier and pass one LDS barrier (every
// wave finished reading the slots refilled below, and stage s+1 has landed);
// then the wave's 8 x 8 blocks (64 MFMAs) run with one DMA instruction per
// row of 8 MFMAs (B stage s+4 into slot s % 4 on even rows, a quarter of A
// pair (s+1)/2 + 2 on odd rows) and the 24 reads of stage s+1's operands
// spread under them.  Measured on random operands, power-limited (1400 W),
// same box, 8192^3: 32-deep A and B slots with both DMAs every other row
// 762-772 us; one DMA per row 758-763 us (on zero operands, not
// power-limited, 585 -> 521 us: two DMAs at once stall the MFMA issue); A
// in 128-byte lines as here 735-742 us.  Per 32-k stage the loop takes ~1256
// cycles for 1024 cycles of MFMA work: ~62 at the barrier, ~8 waiting for
// DMAs, the rest issue gaps, ~16 cycles per DMA instruction.  A 64-byte A
// row (the 32-deep A slot) makes each DMA instruction touch 16 half lines
// instead of 8 whole ones; in cycles both run alike, but the whole-line
// version spends less energy per GEMM, so at the power limit it keeps a
// higher clock.
constexpr int KS = 32;                    // k per B slot and per barrier
constexpr int BROWB = BN * 2;             // bytes per B k-row in LDS
constexpr int A_SLOT_BYTES = BM * 128;    // one A slot: 64 k
constexpr int B_SLOT_BYTES = KS * BROWB;  // one B slot: 32 k

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));   // 16 bytes at any element of C: one store instruction all the same
template <int V> struct TailC { static constexpr int v = V; };

// EDGE: M and N of any size (N even), K a multiple of 8: rows past M read row M - 1,
// chunks past K and k-rows past K read zeros, only outputs inside C are stored.
template <bool EDGE>
__global__ __launch_bounds__(256, 1)
void gemm_bf16_full_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                           uint16_t* __restrict__ C, uint32_t M, uint32_t N, uint32_t K,
                           uint32_t tiles_m, uint32_t tiles_n) {
    __shared__ __attribute__((aligned(1024))) uint8_t AL[3 * A_SLOT_BYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t BL[4 * B_SLOT_BYTES];

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: DMA bases
    const uint32_t wm = wave >> 1, wn = wave & 1;
    uint32_t tm, tn;
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, &tm, &tn);
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(tm * BM);
    const uint32_t n0 = __builtin_amdgcn_readfirstlane(tn * BN);
    const uint32_t nstages = EDGE ? (K + 127) / 128 * 4 : K / KS;   // a multiple of 4
    const uint32_t npairs = nstages / 2;

    const i32x4 ars = dma_rsrc(A, M * K * 2), brs = dma_rsrc(B, K * N * 2);
    const uint32_t al = lds_addr(AL), bl = lds_addr(BL);

    // A DMA instruction i (0..7) of wave w for pair q (k 64 q .. 64 q + 63):
    // rows 64 w + 8 i + l/8, slot l%8, which holds chunk
    // (l%8) ^ ((row/2) % 8) = (l%8) ^ ((4 i + l/16) % 8).
    uint32_t a_voff[2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
        a_voff[p] = ((lane >> 3) * K + 8 * ((lane & 7) ^ ((4 * p + (lane >> 4)) & 7))) * 2;
    const uint32_t a_dst = 64 * wave * 128;
    const uint32_t a_src = EDGE ? 0 : (m0 + 64 * wave) * K * 2;
    // B DMA instruction i (0..3) of wave w: k-rows r = 8 w + 2 i + l/32, slot
    // l%32, which holds chunk (l%32) ^ f(r).
    const uint32_t b_r = lane >> 5;
    const uint32_t bx = 2 * (wave & 1);
    const uint32_t b_voff0 = (b_r * N + 8 * ((lane & 31) ^ (4 * b_r) ^ bx)) * 2;
    const uint32_t b_voff1 = (b_r * N + 8 * ((lane & 31) ^ (4 * (2 + b_r)) ^ bx)) * 2;
    const uint32_t b_dst = 8 * wave * BROWB;
    const uint32_t b_src = (8 * wave * N + n0) * 2;
    // DMA instruction i of a stage: lds = the slot's LDS address for this
    // wave, glb = the operand's byte offset for this wave and stage.  What
    // depends on i is a per-lane voffset (one VGPR per instruction) and a
    // loop-invariant LDS offset added into M0, so a DMA costs one scalar
    // instruction besides the load.
    uint32_t a_vo[8], b_vo[4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        a_vo[i] = EDGE ? a_voff[i & 1] + (min(m0 + 64 * wave + 8 * i + (lane >> 3), M - 1) - (lane >> 3)) * K * 2
                       : a_voff[i & 1] + 8 * i * K * 2;
#pragma unroll
    for (int i = 0; i < 4; ++i) b_vo[i] = ((i & 1) ? b_voff1 : b_voff0) + 2 * i * N * 2;
    const uint32_t bl_w = bl + b_dst;
    const uint32_t al_w = al + a_dst;
    auto dma_a = [&](uint32_t lds, uint32_t glb, int i) {
        uint32_t vo = a_vo[i];
        if (EDGE) {   // glb = 128 bytes per pair: this lane's chunk starts at k = glb / 2 + ...
            const uint32_t ch = (lane & 7) ^ ((4 * (i & 1) + (lane >> 4)) & 7);
            vo = glb / 2 + 8 * ch < K ? vo : 0x80000000u;
        }
        dma16_at(ars, lds, 8 * i * 128, vo, glb);
    };
    auto dma_b = [&](int slot, uint32_t glb, int i) {
        dma16_at(brs, bl_w, slot * B_SLOT_BYTES + 2 * i * BROWB, b_vo[i], glb);
    };

    f32x4 acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{};

    // 16x16x32 operands.  A (i): lane l holds row wm*128 + 16 i + l%16,
    // k octet l/16 of the stage's 32-k half h.
    const uint32_t g = lane >> 4, t = lane & 15;
    const uint32_t a_row = (wm * 128 + t) * 128;
    const uint32_t a_half[2] = {16 * ((0 + g) ^ ((t >> 1) & 7)), 16 * ((4 + g) ^ ((t >> 1) & 7))};
    const uint32_t a_rh[2] = {a_row + a_half[0], a_row + a_half[1]};
    // B (j): lane l needs column wn*128 + 16 j + l%16, k = 8 (l/16) .. +7:
    // two ds_read_b64_tr_b16 (k-rows 8g + 4q + t/4, columns 4 (t%4) .. +3 of
    // the 16-column block), each returning 4 k of column t.
    uint32_t b_off[8][2];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t r = 8 * g + 4 * q + (t >> 2);
            const uint32_t c = wn * 128 + 16 * j + 4 * (t & 3);
            const uint32_t f = 4 * (r & 3) ^ 2 * ((r >> 3) & 1);
            b_off[j][q] = r * BROWB + 16 * ((c >> 3) ^ f) + 2 * (c & 7);
        }
    auto b_at = [&](const uint8_t* bs, int j) {
        u32x2 h[2];
#pragma unroll
        for (int q = 0; q < 2; ++q)
            h[q] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_s16x4_t*)(bs + b_off[j][q])));
        return __builtin_bit_cast(bf16x8, u32x4{h[0][0], h[0][1], h[1][0], h[1][1]});
    };
    auto a_at = [&](const uint8_t* as, int i) {
        return *reinterpret_cast<const bf16x8*>(as + 16 * i * 128);
    };
    bf16x8 a[2][8], b[2][8];
    // The MFMAs are inline asm with the accumulators pinned to AccVGPRs
    // ("+a"): with 64 four-register accumulators the register allocator
    // otherwise shuttles them between AccVGPRs and VGPRs every iteration.
    // The wait-count pass sees the asm operands (it waits for the operand
    // reads); the one hazard it cannot see -- reading an accumulator right
    // after the MFMA that writes it -- is padded before the epilogue.
    // Consecutive MFMAs share an operand register (snake order over j).
    // The B fragment goes in the MFMA's first operand and the A fragment in
    // its second, so the MFMA computes the 16x16 block transposed: lane l,
    // register r of acc[i][j] is C row 16 i + l%16, column 16 j + 4 (l/16) + r
    // (four consecutive columns of one row, which the epilogue packs into
    // one 8-byte LDS write).  The products and their k order are the same.
    auto mfma = [&](int c, int i, int jj) {
        const int j = (i & 1) ? 7 - jj : jj;
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[i][j]) : "v"(b[c][j]), "v"(a[c][i]));
    };
    // Stage s at unrolled position u = s % 4.  A pair q occupies slot q % 3
    // and is fetched a quarter per stage over stages 2q - 5 and 2q - 4, i.e.
    // three stages before its first read; its slot held pair q - 3, whose
    // last operands were read during stage 2q - 6.
    // TAIL: 0 = steady state; 1..4 = the last four stages (no DMAs: every
    // operand is already requested), waiting for vmcnt 16 / 8 / 0 and, in the
    // last stage, nothing (its operands were read in stage n-2).
    // Stage s = 4 t + u.  Its scalar operands come from the loop, which
    // carries them from iteration to iteration instead of recomputing them
    // (a pair's slot is pair % 3).  With the divisions, the clamps and the
    // per-DMA address arithmetic the loop issued ~34 scalar and ~3 vector
    // ALU instructions per stage; now ~15 (8 of them the M0 adds) and 1,
    // and the 8192^3 GEMM runs ~4 % faster (715-723 -> 699-700 us,
    // alternated on one box, with the move of the operands ahead of the
    // barrier described below):
    //   rd_slot  slot byte offset of the pair holding stage s+1 (read side);
    //   dma_slot slot byte offset of the pair being fetched;
    //   a_glb, b_glb  this wave's byte offsets of the A pair and B stage being fetched.
    // They are formed before the barrier, under the previous stage's last
    // MFMAs (the empty asm statements keep them there), so that after the
    // barrier the stage's first MFMA follows at once.
    auto stage = [&](int u, uint32_t rd_slot, uint32_t dma_slot, uint32_t a_glb, uint32_t b_glb,
                     auto TL) {
        constexpr int TAIL = decltype(TL)::v;
        const int c = u & 1;
        const int ih = 4 * ((u + 1) & 1);          // its instructions 0-3 (s odd) or 4-7
        uint32_t a_lds = al_w + dma_slot;
        uint32_t nas_off = rd_slot + a_rh[(u + 1) & 1];
        if (TAIL == 0) asm volatile("" : "+s"(a_lds), "+s"(a_glb), "+s"(b_glb));
        if (TAIL != 4) asm volatile("" : "+v"(nas_off));
        __builtin_amdgcn_sched_barrier(0);
        if (TAIL <= 1) __builtin_amdgcn_s_waitcnt(0x4F70);   // vmcnt(16): stages s-1, s-2 may be in flight
        else if (TAIL == 2) __builtin_amdgcn_s_waitcnt(0x0F78);   // vmcnt(8)
        else if (TAIL == 3) __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        if (TAIL != 4) lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t* nas = AL + nas_off;
        const uint8_t* nbs = BL + ((u + 1) & 3) * B_SLOT_BYTES;
        // unit v < 8: B v (two transposing reads); v >= 8: A v-8 (one read),
        // in the order stage s+1 consumes them (its first row needs every B)
        auto rd = [&](int v) {
            if (v < 8) b[c ^ 1][v] = b_at(nbs, v);
            else a[c ^ 1][v - 8] = a_at(nas, v - 8);
        };
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            mfma(c, r, 0);
            if (TAIL == 0) {
                if (r & 1) dma_a(a_lds, a_glb, ih + (r >> 1));
                else dma_b(u, b_glb, r >> 1);
            }
            mfma(c, r, 1);
            if (TAIL != 4) rd(2 * r);
            mfma(c, r, 2);
            mfma(c, r, 3);
            mfma(c, r, 4);
            if (TAIL != 4) rd(2 * r + 1);
            mfma(c, r, 5);
            mfma(c, r, 6);
            mfma(c, r, 7);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // Prologue: A pairs 0-2 and B stages 0-3, in the order A0 B0 B1 A1 B2 B3
    // A2 (40 DMA instructions per wave).  Stage 0's barrier then waits for
    // the first 24 (A0 B0 B1 A1) and stage 0 reloads the second half of A2.
    // The last four stages are peeled: every byte they need is requested
    // by then, so they issue no DMAs and the epilogue waits for none
    // (waiting for clamped reloads there had cost 571 against 550 us on zero
    // operands).
#pragma unroll
    for (int i = 0; i < 8; ++i) dma_a(al_w, a_src, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_b(0, b_src, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_b(1, b_src + KS * N * 2, i);
#pragma unroll
    for (int i = 0; i < 8; ++i) dma_a(al_w + A_SLOT_BYTES, a_src + 128, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_b(2, b_src + 2 * KS * N * 2, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_b(3, b_src + 3 * KS * N * 2, i);
#pragma unroll
    for (int i = 0; i < 8; ++i) dma_a(al_w + 2 * A_SLOT_BYTES, a_src + 2 * 128, i);
    __builtin_amdgcn_s_waitcnt(0x4F7C);   // vmcnt(28): A pair 0 and B stage 0 have landed
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        a[0][i] = a_at(AL + a_row + a_half[0], i);
        b[0][i] = b_at(BL, i);
    }
    // Iteration t (stages 4t .. 4t+3) reads pairs 2t, 2t+1, 2t+1, 2t+2 and
    // fetches pairs 2t+2, 2t+3, 2t+3, 2t+4 and B stages 4t+4 .. 4t+7.  sl0,
    // sl1, sl2 are the slots of pairs 2t, 2t+1, 2t+2 (= 2t+3, 2t+4, ... mod
    // 3); the next iteration's are sl2, sl0, sl1.  Pair 2t+4 is past the last
    // one only in the last iteration (a stage of the tail then reloads pair
    // 2t+3 into its own slot instead: the same bytes, so a concurrent read of
    // it is unaffected).
    uint32_t sl0 = 0, sl1 = A_SLOT_BYTES, sl2 = 2 * A_SLOT_BYTES;
    uint32_t a_t = a_src;                          // A pair 2t
    uint32_t b_t = b_src + 4 * KS * N * 2;         // B stage 4t + 4
    const uint32_t b_u = KS * N * 2;               // one B stage
    uint32_t t2 = 0;                               // 2t
    for (uint32_t s = 0; s + 4 < nstages; s += 4, t2 += 2) {
        const bool last = t2 + 4 > npairs - 1;
        stage(0, sl0, sl2, a_t + 2 * 128, b_t, TailC<0>{});
        stage(1, sl1, sl0, a_t + 3 * 128, b_t + b_u, TailC<0>{});
        stage(2, sl1, sl0, a_t + 3 * 128, b_t + 2 * b_u, TailC<0>{});
        stage(3, sl2, last ? sl0 : sl1, a_t + (last ? 3 : 4) * 128, b_t + 3 * b_u, TailC<0>{});
        const uint32_t s2 = sl2;
        sl2 = sl1;
        sl1 = sl0;
        sl0 = s2;
        a_t += 2 * 128;
        b_t += 4 * b_u;
    }
    stage(0, sl0, 0, 0, 0, TailC<1>{});
    stage(1, sl1, 0, 0, 0, TailC<2>{});
    stage(2, sl1, 0, 0, 0, TailC<3>{});
    stage(3, sl2, 0, 0, 0, TailC<4>{});
    __builtin_amdgcn_s_waitcnt(0);   // no DMA may still target LDS
    // the last MFMAs' results must be written before they are read
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");

    // Epilogue through LDS (32 KB per wave: the three A slots and the first
    // two B slots, 128 rows of 256 B): lane l holds, for block (i, j), row
    // 16 i + l%16, columns 16 j + 4 (l/16) .. +3, written as one packed 8-byte
    // LDS store (the first version wrote 2-byte elements from the
    // untransposed layout: ~2.8 us per tile, LDS-instruction bound; a DPP
    // exchange to 4-byte pairs still took 2.0 us, VALU bound).  The 8-byte
    // chunk c of row r sits at c ^ 4 (r % 8): the 64 lanes of a write (16 rows
    // x 4 chunks) then fill every bank twice, the fewest for 512 bytes, and
    // 16-byte row chunks stay contiguous for the reads below.
    lds_barrier();
    uint8_t* ct = wave < 3 ? AL + wave * A_SLOT_BYTES : BL;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t row = 16 * i + t;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const f32x4 v = acc[i][j];
            const u32x2 w = {
                __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[0], v[1]}, bf16x2)),
                __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2], v[3]}, bf16x2))};
            const uint32_t c8 = (4 * j + g) ^ (4 * (row & 7));
            *reinterpret_cast<u32x2*>(ct + row * 256 + 8 * c8) = w;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    // C is written once and never read here: non-temporal stores keep it out
    // of L2's way (8192^3 random operands at the power limit: 740-748 ->
    // 730-737 us, the same in either run order; output unchanged).
#pragma unroll
    for (int q = 0; q < 32; ++q) {
        const uint32_t row = 4 * q + (lane >> 4), ch = lane & 15;
        const u32x4 v = *reinterpret_cast<const u32x4*>(
            ct + row * 256 + 16 * (ch ^ (2 * (row & 7))));
        const uint32_t gr = m0 + wm * 128 + row, gc = n0 + wn * 128 + 8 * ch;
        uint16_t* at = C + (size_t)gr * N + gc;
        if (!EDGE || ((N & 7) == 0 && ((uintptr_t)C & 15) == 0)) {
            if (!EDGE || (gr < M && gc < N)) __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any*>(at));
        } else if (gr < M) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (gc + e < N) at[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
    }
}


// ---- any shape: tiles of 32 MB x 32 NB ------------------------------------------------
// Four waves in a 2 x 2 grid, each 16 MB x 16 NB outputs (MB x NB
// v_mfma_f32_16x16x32_bf16 per 32-deep stage, operands and products as in the
// full-tile kernel: B first, so a lane holds four consecutive columns of one
// row).  A ring of R LDS slots, one stage each:
//  * A: 32 MB rows of 64 bytes; 16-byte chunk c of row r sits in slot
//    c ^ ((r / 4) % 4) (16 lanes reading 16 rows touch 16 bank groups);
//  * B: 32 k-rows of 64 NB bytes; chunk c of k-row r sits in slot c ^ f(r),
//    so that the eight k-rows that a ds_read_b64_tr_b16 reads per LDS cycle (4
//    r .. 4 r + 3, and 8 further) lie in distinct banks.
// Stage s: wait for this wave's part of stage s+1, pass one barrier (every
// wave has read all of slot s; stage s+1 has landed), fetch stage s+R into slot
// s, then run stage s's MFMAs with the reads of stage s+1's operands among them.
// KG groups of four waves each take a 32-deep part of the stage and are added
// through LDS at the end: with one group a stage is 16 MFMAs (256 cycles) long and
// costs 800 at one workgroup per CU (barrier, LDS latency, instruction issue);
// two groups share those.  What bounds it then is the ring: first use of a line
// by an XCD takes 1.6 us from the memory side, and three to four stages (96-112
// KB per CU) are in flight (512 x 6144 x 4096: 36 us; with the loop's DMAs left
// out 26, with its MFMAs or LDS reads left out 36).
// ODD = false: rows start on 4-byte boundaries (K and N even) and operands go to
// LDS by DMA.  ODD = true: 16-byte chunks are loaded as five dwords, shifted into
// place and stored to LDS two stages ahead.
// Rows past M read row M - 1, what lies past the end of an operand reads as
// zero, and only outputs inside C are stored.  k past K is zero in B; in A's last
// stage it is the next row's values, which are cleared in LDS once they landed.
constexpr uint32_t OOB = 0x80000000u;

template <int NB>
__device__ __forceinline__ uint32_t b_swizzle(uint32_t r) {
    if (NB == 4) return (4 * (r & 3)) ^ (2 * ((r >> 3) & 1));
    if (NB == 2) return (4 * ((r >> 1) & 1)) ^ (2 * ((r >> 3) & 1));
    return 2 * ((r >> 3) & 1);   // NB = 1, 3: four k-rows already lie in distinct banks
}

template <int MB, int NB, int KG, int R, bool ODD>
__global__ __launch_bounds__(256 * KG, 2)
void gemm_bf16_tile_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                           uint16_t* __restrict__ C, uint32_t M, uint32_t N, uint32_t K,
                           uint32_t tiles_m, uint32_t tiles_n, uint32_t band) {
    constexpr int TM = 32 * MB, TN = 32 * NB;
    constexpr uint32_t A_BYTES = TM * 64, SUB = A_BYTES + TN * 64, SLOT = KG * SUB;
    constexpr int KST = 32 * KG;                   // k per stage
    constexpr int BROW = 64 * NB;                  // bytes per B k-row
    constexpr int NI = 2 * MB + 2 * NB;            // 1 KB pieces per k group of a slot
    constexpr int NW = (NI + 3) / 4;               // pieces per wave (the last may be a dummy)
    constexpr int WAVES = 4 * KG;
    extern __shared__ __attribute__((aligned(1024))) uint8_t S[];   // R slots (+ 1 KB for dummies)

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    const uint32_t g = lane >> 4, t = lane & 15;
    uint32_t tm, tn;
    xcd_band_tile(blockIdx.x, gridDim.x, tiles_m, tiles_n, band, &tm, &tn);
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(tm * TM);
    const uint32_t n0 = __builtin_amdgcn_readfirstlane(tn * TN);
    const uint32_t nst = (K + KST - 1) / KST;

    // operands from the 4-byte boundary at or below their start
    const uint32_t a_mis = ODD ? (uint32_t)(uintptr_t)A & 2 : 0, b_mis = ODD ? (uint32_t)(uintptr_t)B & 2 : 0;
    const i32x4 ars = dma_rsrc(reinterpret_cast<const uint8_t*>(A) - a_mis, (M * K * 2 + a_mis + 3) & ~3u);
    const i32x4 brs = dma_rsrc(reinterpret_cast<const uint8_t*>(B) - b_mis, (K * N * 2 + b_mis + 3) & ~3u);

    // this wave's piece q: piece x = wave + WAVES q of the slot, i.e. piece
    // x % NI (A's first) of k group x / NI
    uint32_t vo[NW];         // this lane's byte offset at stage 0
    uint32_t krow[NW];       // B's k-row
    bool is_a[NW], none[NW];
#pragma unroll
    for (int q = 0; q < NW; ++q) {
        const uint32_t x = wave + WAVES * q, sub = x / NI, y = x - sub * NI;
        is_a[q] = y < 2 * MB;
        none[q] = sub >= (uint32_t)KG;
        if (is_a[q]) {
            const uint32_t r = 16 * y + (lane >> 2), ch = (lane & 3) ^ ((r >> 2) & 3);
            vo[q] = a_mis + (min(m0 + r, M - 1) * K + 32 * sub + 8 * ch) * 2;
            krow[q] = 0;
        } else {
            const uint32_t l = 64 * (y - 2 * MB) + lane, r = l / (4 * NB);
            const uint32_t ch = (l - r * (4 * NB)) ^ b_swizzle<NB>(r);
            krow[q] = 32 * sub + r;
            vo[q] = b_mis + (krow[q] * N + n0 + 8 * ch) * 2;
        }
        if (none[q]) vo[q] = OOB;
    }
    const uint32_t l0 = lds_addr(S) + 1024 * wave;
    auto dma = [&](uint32_t slot, uint32_t s) {
        const uint32_t a_so = s * (2 * KST), b_so = s * (2 * KST) * N;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            // (a dummy lands zeros in the KB past the ring)
            const uint32_t at = none[q] ? l0 - 1024 * wave - slot + R * SLOT : l0 + 1024 * WAVES * q;
            if (is_a[q]) dma16_at(ars, slot, at, vo[q], none[q] ? 0 : a_so);
            else dma16_at(brs, slot, at, vo[q], none[q] ? 0 : b_so);
        }
    };
    // ODD: the five dwords that hold each 16-byte chunk, and the chunk
    struct Piece { u32x4 d; uint32_t e; };
    const __amdgpu_buffer_rsrc_t arb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(A) - a_mis), 0,
        __builtin_amdgcn_readfirstlane((M * K * 2 + a_mis + 3) & ~3u), 0x00020000u);
    const __amdgpu_buffer_rsrc_t brb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(B) - b_mis), 0,
        __builtin_amdgcn_readfirstlane((K * N * 2 + b_mis + 3) & ~3u), 0x00020000u);
    auto fetch = [&](Piece (&p)[NW], uint32_t s) {
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            uint32_t off = is_a[q] ? vo[q] + s * (2 * KST) : vo[q] + s * (2 * KST) * N;
            if (none[q] || (!is_a[q] && KST * s + krow[q] >= K)) off = OOB;
            const __amdgpu_buffer_rsrc_t rs = is_a[q] ? arb : brb;
            p[q].d = __builtin_amdgcn_raw_buffer_load_b128(rs, off & ~3u, 0, 0);
            p[q].e = __builtin_amdgcn_raw_buffer_load_b32(rs, (off & ~3u) + 16, 0, 0);
        }
    };
    auto store = [&](const Piece (&p)[NW], uint32_t slot) {
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            if (none[q]) continue;
            const uint32_t sh = 8 * (vo[q] & 2);   // (a stage's rows and columns are even apart)
            const u32x4 d = p[q].d;
            const u32x4 v = {__builtin_amdgcn_alignbit(d[1], d[0], sh), __builtin_amdgcn_alignbit(d[2], d[1], sh),
                             __builtin_amdgcn_alignbit(d[3], d[2], sh), __builtin_amdgcn_alignbit(p[q].e, d[3], sh)};
            *reinterpret_cast<u32x4*>(S + slot + 1024 * (wave + WAVES * q) + 16 * lane) = v;
        }
    };
    // k past K in A's last stage
    const uint32_t kv = K - (nst - 1) * KST;   // k of the last stage
    auto clear_tail = [&](uint32_t slot) {
        for (uint32_t r = tid; r < (uint32_t)(TM * KG); r += 256 * KG) {
            const uint32_t sub = r / TM, row = r - sub * TM;
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) {
                const uint32_t k = 32 * sub + 8 * c;
                uint16_t* at = reinterpret_cast<uint16_t*>(S + slot + sub * SUB + 64 * row +
                                                           16 * (c ^ ((row >> 2) & 3)));
                if (k >= kv) *reinterpret_cast<u32x4*>(at) = u32x4{};
                else for (uint32_t e = kv - k; e < 8; ++e) at[e] = 0;
            }
        }
        __syncthreads();
    };

    const uint32_t a_rd = kg * SUB + (wm * 16 * MB + t) * 64 + 16 * (g ^ ((t >> 2) & 3));
    uint32_t b_rd[NB][2];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t r = 8 * g + 4 * q + (t >> 2), c = wn * 16 * NB + 16 * j + 4 * (t & 3);
            b_rd[j][q] = kg * SUB + A_BYTES + r * BROW + 16 * ((c >> 3) ^ b_swizzle<NB>(r)) + 2 * (c & 7);
        }
    struct Ops { bf16x8 a[MB], b[NB]; };
    auto read = [&](Ops& o, uint32_t slot) {
        const uint8_t* s = S + slot;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            u32x2 h[2];
#pragma unroll
            for (int q = 0; q < 2; ++q)
                h[q] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_s16x4_t*)(s + b_rd[j][q])));
            o.b[j] = __builtin_bit_cast(bf16x8, u32x4{h[0][0], h[0][1], h[1][0], h[1][1]});
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) o.a[i] = *reinterpret_cast<const bf16x8*>(s + a_rd + 1024 * i);
    };
    f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{};
    auto mfma = [&](const Ops& o) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int jj = 0; jj < NB; ++jj) {
                const int j = (i & 1) ? NB - 1 - jj : jj;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.b[j], o.a[i], acc[i][j], 0, 0, 0);
            }
    };
    // at most `younger` stages' DMAs of this wave still in flight
    auto wait = [&](uint32_t younger) {
        if (younger >= R - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 2) * NW) : "memory");
        else if (younger >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NW) : "memory");
        else if (younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    Ops o[2];
    Piece p[2][ODD ? NW : 1];
    auto step = [](uint32_t slot) { return slot + SLOT == R * SLOT ? 0u : slot + SLOT; };
    if constexpr (ODD) {
        auto& pp = reinterpret_cast<Piece (&)[2][NW]>(p);
        fetch(pp[0], 0);
        fetch(pp[1], 1);
        store(pp[0], 0);
        fetch(pp[0], 2);
        store(pp[1], SLOT);
        fetch(pp[1], 3);
    } else {
        for (uint32_t s = 0; s < min(nst, (uint32_t)R); ++s) dma(s * SLOT, s);
        if (nst >= (uint32_t)R) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * NW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    lds_barrier();
    if (kv < (uint32_t)KST && nst == 1) clear_tail(0);
    read(o[0], 0);

    uint32_t here = 0, after = SLOT;   // slots of stages s and s + 1
    // MORE: stages s + 1 .. s + R exist (no tail to look for)
    auto stage = [&](auto c_, auto more_, uint32_t s) {
        constexpr int c = decltype(c_)::value;
        constexpr bool MORE = decltype(more_)::value;
        if constexpr (!ODD) wait(MORE ? R - 2 : nst >= s + 2 ? nst - s - 2 : 0);
        lds_barrier();
        if (!MORE && kv < (uint32_t)KST && s + 2 == nst) clear_tail(after);
        if constexpr (ODD) {
            // stage s + 2 to LDS (its slot's last readers were stage s + 2 - R's), stage s + 4 fetched
            auto& pp = reinterpret_cast<Piece (&)[2][NW]>(p);
            store(pp[c], step(after));
            fetch(pp[c], s + 4);
        } else if (MORE) dma(here, s + R);
        __builtin_amdgcn_sched_barrier(0);
        read(o[c ^ 1], after);
        mfma(o[c]);
#pragma unroll
        for (int x = 0; x < MB * NB; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        here = after;
        after = step(after);
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    uint32_t s = 0;
    for (; s + 1 + R < nst; s += 2) {
        stage(C0{}, std::true_type{}, s);
        stage(C1{}, std::true_type{}, s + 1);
    }
    if (s + R < nst) {   // an odd stage before the last R: keep the operand sets' parity
        stage(C0{}, std::true_type{}, s);
        ++s;
        stage(C1{}, std::false_type{}, s);
        ++s;
    }
    for (; s + 1 < nst; s += 2) {
        stage(C0{}, std::false_type{}, s);
        stage(C1{}, std::false_type{}, s + 1);
    }
    if (s < nst) stage(C0{}, std::false_type{}, s);

    if constexpr (KG == 2) {
        // The two k groups finish every other block of each 16 MB x 16 NB part:
        // each hands the other the blocks it does not store.
        lds_barrier();
        f32x4* mine = reinterpret_cast<f32x4*>(S) + (wave & 3) * (MB * NB * 64);
#pragma unroll
        for (int b = 0; b < MB * NB; ++b)
            if ((b & 1) != (int)kg) mine[b * 64 + lane] = acc[b / NB][b % NB];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < MB * NB; ++b)
            if ((b & 1) == (int)kg) acc[b / NB][b % NB] += mine[b * 64 + lane];
    }

    // lane l holds, for block (i, j), row 16 i + l%16, columns 16 j + 4 (l/16) .. +3
    const bool wide = (N & 3) == 0 && ((uintptr_t)C & 7) == 0;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const uint32_t row = m0 + wm * 16 * MB + 16 * i + t;
        if (row >= M) continue;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (KG == 2 && ((i * NB + j) & 1) != (int)kg) continue;
            const uint32_t col = n0 + wn * 16 * NB + 16 * j + 4 * g;
            const f32x4 v = acc[i][j];
            const u32x2 w = {
                __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[0], v[1]}, bf16x2)),
                __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2], v[3]}, bf16x2))};
            uint16_t* at = C + (size_t)row * N + col;
            if (wide) {
                if (col < N) *reinterpret_cast<u32x2*>(at) = w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < N) at[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
            }
        }
    }
}


// ---- small C: tiles of 16 MB x 16 NC, K dealt to four waves ---------------------------
// Each wave multiplies the whole tile over its units of 32 k (u = wave mod 4, the
// last first), so the waves share nothing and the loop has no barrier; the four
// partial tiles are added through LDS at the end, in wave order.
//  * B goes straight to registers: lane (kq = l / 16, nl = l % 16) loads k-rows 8
//    kq .. 8 kq + 7, columns NC nl .. NC nl + NC - 1 (one row of 16 lanes is
//    contiguous) and transposes the block with v_perm_b32 into the MFMA operands
//    of columns {NC nl + c};
//  * A is loaded as whole row pieces and passes through 1 KB of LDS per 16 rows,
//    the wave's own, to become the MFMA operand (16-byte chunk c of row r in slot
//    c ^ ((r / 4) % 4));
//  * unit j is multiplied while unit j + 1's A passes through LDS, and B of unit j
//    + 2 and A of unit j + 3 are in flight.
// ODD: chunks are loaded from the 4-byte boundary below them, one dword more, and
// shifted into place.  A unit's k past K is zero in B, and cleared in A's operand.
// 256 x 4096 x 4096: 19 us (64 x 64 tiles), 37 with gemm_bf16_tile_kernel's 128 x
// 128; 32 x 6144 x 4096: 14 us (16 x 64 tiles), 3.7 TB/s of B.
constexpr int KW = 4;   // waves

template <int D> struct Dwords { uint32_t v[D]; };
template <int D>
__device__ __forceinline__ Dwords<D> load_dwords(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t soff) {
    Dwords<D> r;
    if constexpr (D == 5) {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, 0);
        r.v[0] = x[0]; r.v[1] = x[1]; r.v[2] = x[2]; r.v[3] = x[3];
        r.v[4] = __builtin_amdgcn_raw_buffer_load_b32(rs, off + 16, soff, 0);
    } else if constexpr (D == 4) {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, 0);
        r.v[0] = x[0]; r.v[1] = x[1]; r.v[2] = x[2]; r.v[3] = x[3];
    } else if constexpr (D == 3) {
        typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
        const u32x3 x = __builtin_amdgcn_raw_buffer_load_b96(rs, off, soff, 0);
        r.v[0] = x[0]; r.v[1] = x[1]; r.v[2] = x[2];
    } else if constexpr (D == 2) {
        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(rs, off, soff, 0);
        r.v[0] = x[0]; r.v[1] = x[1];
    } else {
        r.v[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, soff, 0);
    }
    return r;
}

template <int MB, int NC, bool ODD>
__global__ __launch_bounds__(64 * KW, 1)
void gemm_bf16_kwave_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                            uint16_t* __restrict__ C, uint32_t M, uint32_t N, uint32_t K,
                            uint32_t tiles_m, uint32_t tiles_n, uint32_t band) {
    constexpr int DA = ODD ? 5 : 4, DB = NC / 2 + (ODD ? 1 : 0);   // dwords per loaded chunk
    constexpr int RED = 4 * KW * NC * 1024, RING = KW * MB * 1024;
    __shared__ __attribute__((aligned(1024))) uint8_t S[RED > RING ? RED : RING];

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kq = lane >> 4, nl = lane & 15;
    uint32_t tm, tn;
    xcd_band_tile(blockIdx.x, gridDim.x, tiles_m, tiles_n, band, &tm, &tn);
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(tm * (16 * MB));
    const uint32_t n0 = __builtin_amdgcn_readfirstlane(tn * (16 * NC));
    auto rsrc = [](const uint16_t* p, uint32_t mis, uint32_t elems) {
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(p) - mis), 0,
            __builtin_amdgcn_readfirstlane((elems * 2 + mis + 3) & ~3u), 0x00020000u);
    };
    const uint32_t a_mis = ODD ? (uint32_t)(uintptr_t)A & 2 : 0, b_mis = ODD ? (uint32_t)(uintptr_t)B & 2 : 0;
    const __amdgpu_buffer_rsrc_t ars = rsrc(A, a_mis, M * K), brs = rsrc(B, b_mis, K * N);

    // the wave takes units (32 k) u = wave (mod KW), last first
    const uint32_t units = (K + 31) / 32;
    const uint32_t n = units > wave ? (units - wave + KW - 1) / KW : 0;
    const uint32_t u_top = wave + KW * (n - 1);   // (n > 0)

    // A: chunk lane % 4 of rows 16 i + lane / 4, to LDS; B: k-rows 8 kq + e, columns NC nl ..
    uint32_t a_vo[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
        a_vo[i] = a_mis + (min(m0 + 16 * i + (lane >> 2), M - 1) * K + 8 * (lane & 3)) * 2;
    const uint32_t b_vo = b_mis + (8 * kq * N + n0 + NC * nl) * 2;
    const uint32_t b_odd = ODD ? N & 1 : 0;      // odd k-rows start half a dword further
    uint8_t* sw = S + wave * (MB * 1024);
    const uint32_t a_wr = 64 * (lane >> 2) + 16 * ((lane & 3) ^ (lane >> 4));
    const uint32_t a_rd = 64 * nl + 16 * (kq ^ ((nl >> 2) & 3));

    struct RawA { Dwords<DA> r[MB]; };
    struct RawB { Dwords<DB> r[8]; };
    struct OpsA { bf16x8 a[MB]; };
    // the wave's j-th unit; past its last: out of range, nothing is fetched
    auto load_a = [&](RawA& x, uint32_t j) {
        const uint32_t so = j < n ? (u_top - KW * j) * 64 : OOB;
#pragma unroll
        for (int i = 0; i < MB; ++i) x.r[i] = load_dwords<DA>(ars, ODD ? a_vo[i] & ~3u : a_vo[i], so);
    };
    auto load_b = [&](RawB& x, uint32_t j) {
        const uint32_t k0 = (u_top - KW * j) * 32;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (ODD) {   // k-rows past K would start inside the last dword
                const uint32_t off = b_vo + (k0 + e) * N * 2;
                x.r[e] = load_dwords<DB>(brs, j < n && k0 + 8 * kq + e < K ? off & ~3u : OOB, 0);
            } else {
                x.r[e] = load_dwords<DB>(brs, b_vo, j < n ? (k0 + e) * N * 2 : OOB);
            }
        }
    };
    auto put_a = [&](const RawA& x) {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            u32x4 v;
#pragma unroll
            for (int d = 0; d < 4; ++d)
                v[d] = ODD ? __builtin_amdgcn_alignbit(x.r[i].v[DA == 5 ? d + 1 : d], x.r[i].v[d], 8 * (a_vo[i] & 2))
                           : x.r[i].v[d];
            *reinterpret_cast<u32x4*>(sw + 1024 * i + a_wr) = v;
        }
    };
    auto get_a = [&](OpsA& o) {
#pragma unroll
        for (int i = 0; i < MB; ++i) o.a[i] = *reinterpret_cast<const bf16x8*>(sw + 1024 * i + a_rd);
    };
    f32x4 acc[MB][NC];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[i][c] = f32x4{};
    // column c of every lane: the 8 k of an 8 x NC block, transposed
    auto col = [&](const RawB& x, int c) {
        u32x4 v;
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (ODD) w[e] = __builtin_amdgcn_alignbit(x.r[e].v[c / 2 + (DB > NC / 2 ? 1 : 0)], x.r[e].v[c / 2],
                                                      8 * ((b_vo + e * 2 * b_odd) & 2));
            else w[e] = x.r[e].v[c / 2];
        }
#pragma unroll
        for (int d = 0; d < 4; ++d)
            v[d] = __builtin_amdgcn_perm(w[2 * d + 1], w[2 * d], (c & 1) ? 0x07060302u : 0x05040100u);
        return __builtin_bit_cast(bf16x8, v);
    };

    if (n > 0) {
        RawA ra[2];
        RawB rb[3];
        OpsA oa[2];
        load_a(ra[0], 0);
        __builtin_amdgcn_sched_barrier(0);
        load_b(rb[0], 0);
        __builtin_amdgcn_sched_barrier(0);
        load_a(ra[1], 1);
        __builtin_amdgcn_sched_barrier(0);
        load_b(rb[1], 1);
        __builtin_amdgcn_sched_barrier(0);
        put_a(ra[0]);
        get_a(oa[0]);
        if (32 * u_top + 32 > K) {   // k past K: zero in A (B's are out of range)
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                u32x4 v = __builtin_bit_cast(u32x4, oa[0].a[i]);
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const uint32_t k = 32 * u_top + 8 * kq + 2 * d;
                    v[d] = k + 1 < K ? v[d] : k < K ? v[d] & 0xffffu : 0;
                }
                oa[0].a[i] = __builtin_bit_cast(bf16x8, v);
            }
        }
        load_a(ra[0], 2);
        __builtin_amdgcn_sched_barrier(0);
        // unit j: multiply it while unit j + 1's A goes through LDS; then fetch A of
        // unit j + 3 and B of unit j + 2
        auto unit = [&](auto x_, uint32_t j) {
            constexpr int X = decltype(x_)::value;   // j mod 6
            __builtin_amdgcn_sched_barrier(0);
            load_b(rb[(X + 2) % 3], j + 2);
            put_a(ra[(X + 1) % 2]);
            get_a(oa[(X + 1) % 2]);
            load_a(ra[(X + 1) % 2], j + 3);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const bf16x8 b = col(rb[X % 3], c);
#pragma unroll
                for (int i = 0; i < MB; ++i)
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(oa[X % 2].a[i], b, acc[i][c], 0, 0, 0);
            }
#pragma unroll
            for (int x = 0; x < MB * NC; ++x) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (x < 8) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                else if (x < 8 + MB) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                else if (x < 8 + 2 * MB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                else if (x < 8 + 3 * MB) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        uint32_t j = 0;
        for (; j + 6 <= n; j += 6) {
            unit(std::integral_constant<int, 0>{}, j);
            unit(std::integral_constant<int, 1>{}, j + 1);
            unit(std::integral_constant<int, 2>{}, j + 2);
            unit(std::integral_constant<int, 3>{}, j + 3);
            unit(std::integral_constant<int, 4>{}, j + 4);
            unit(std::integral_constant<int, 5>{}, j + 5);
        }
        if (j < n) {
            unit(std::integral_constant<int, 0>{}, j);
            if (j + 1 < n) {
                unit(std::integral_constant<int, 1>{}, j + 1);
                if (j + 2 < n) {
                    unit(std::integral_constant<int, 2>{}, j + 2);
                    if (j + 3 < n) {
                        unit(std::integral_constant<int, 3>{}, j + 3);
                        if (j + 4 < n) unit(std::integral_constant<int, 4>{}, j + 4);
                    }
                }
            }
        }
    }

    // Four 16-row blocks at a time, wave w finishes block 4 q + w: the others
    // leave their parts in LDS, summed in wave order.  Lane: rows 16 i + 4 kq + r,
    // columns NC nl + c.
    f32x4* red = reinterpret_cast<f32x4*>(S);
    const __amdgpu_buffer_rsrc_t crs = __builtin_amdgcn_make_buffer_rsrc(
        C, 0, __builtin_amdgcn_readfirstlane(M * N * 2), 0x00020000u);
#pragma unroll
    for (int q = 0; q < (MB + 3) / 4; ++q) {
        __syncthreads();
#pragma unroll
        for (int x = 0; x < 4; ++x)
            if (4 * q + x < MB && (uint32_t)x != wave)
#pragma unroll
                for (int c = 0; c < NC; ++c) red[((x * KW + wave) * NC + c) * 64 + lane] = acc[4 * q + x][c];
        __syncthreads();
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            if (4 * q + x >= MB || (uint32_t)x != wave) continue;
            const int i = 4 * q + x;
            f32x4 v[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                v[c] = f32x4{};
#pragma unroll
                for (int w = 0; w < KW; ++w)
                    v[c] += w == x ? acc[i][c] : red[((x * KW + w) * NC + c) * 64 + lane];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = m0 + 16 * i + 4 * kq + r, c0 = n0 + NC * nl;
                uint32_t w[NC / 2];
#pragma unroll
                for (int d = 0; d < NC / 2; ++d)
                    w[d] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2 * d][r], v[2 * d + 1][r]}, bf16x2));
                const uint32_t off = (row * N + c0) * 2;
                if (!ODD && c0 + NC <= N && row < M) {
                    if constexpr (NC == 8) __builtin_amdgcn_raw_buffer_store_b128(u32x4{w[0], w[1], w[2], w[3]}, crs, off, 0, 0);
                    else if constexpr (NC == 4) __builtin_amdgcn_raw_buffer_store_b64(u32x2{w[0], w[1]}, crs, off, 0, 0);
                    else
#pragma unroll
                        for (int d = 0; d < NC / 2; ++d) __builtin_amdgcn_raw_buffer_store_b32(w[d], crs, off + 4 * d, 0, 0);
                } else {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        if (row < M && c0 + c < N)
                            __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(w[c / 2] >> (16 * (c & 1))), crs, off + 2 * c, 0, 0);
                }
            }
        }
    }
}

constexpr size_t SMEM_BYTES = 4 * TILE_ELEMS * sizeof(uint16_t);   // 147456

// The tiles that a shape can run on, and what one costs: rounds of 256 tiles, each
// c0 + c1 us per 32 k.  The launcher takes the cheapest.  Large tiles move the fewest
// bytes per product; small ones fill the chip when C is small, and finish sooner
// when K is short.
//  * `odd`: K or N odd, or A or B off a 4-byte boundary; TILE_REG (gemm_bf16_kernel): no
//    16-byte rows, element-wise loads;
//  * `narrow`: more per tile where rows of C don't start on the boundary of a
//    lane's store (16 bytes in TILE_EDGE, 8 in TILE_GRID), so that each lane stores
//    scattered elements.  With many tiles that bounds a short K: 8192 x 8191 x 9 170 us on
//    128 x 128 tiles, 82 on TILE_REG, whose lanes store 32 neighbours; 8192 x 8190 x 8 119
//    on TILE_EDGE, 84 on 64 x 64 tiles (which store whole dwords), 82 on TILE_REG;
//    7104 x 1466 x 21 34 and 24.
// Fitted to the times of every tile on 489 shapes of 8 to 20000 rows and columns and K
// of 4 to 8000: the choice takes 1.02 times the best tile's time in the mean and at most
// 1.05 times gemm_bf16_kernel's (without `narrow` and TILE_REG 1.09 and 2.1).
enum TileKind { TILE_EDGE, TILE_GRID, TILE_WAVE, TILE_REG };
struct TileChoice {
    TileKind kind;
    uint16_t mb, nb;              // template arguments
    uint16_t tm, tn;              // rows and columns per tile
    float c0, c1, odd_c0, odd_c1; // odd_c1 = 0: not for odd shapes
    float narrow;
};
constexpr TileChoice k_tiles[] = {
    {TILE_EDGE, 0, 0, 256, 256, 6.6f, 0.58f, 0, 0, 18.0f},   // K a multiple of 8
    {TILE_GRID, 8, 4, 256, 128, 2.8f, 0.50f, 0, 0, 10.4f},
    {TILE_GRID, 4, 4, 128, 128, 3.9f, 0.265f, 4.7f, 0.53f, 4.8f},
    {TILE_GRID, 4, 3, 128, 96, 4.4f, 0.25f, 3.9f, 0.59f, 2.8f},
    {TILE_WAVE, 4, 8, 64, 128, 3.8f, 0.155f, 4.5f, 0.37f, 0},
    {TILE_WAVE, 4, 4, 64, 64, 1.27f, 0.125f, 2.5f, 0.245f, 0},
    {TILE_WAVE, 2, 4, 32, 64, 1.28f, 0.10f, 2.3f, 0.165f, 0},
    {TILE_WAVE, 1, 4, 16, 64, 0.96f, 0.088f, 2.0f, 0.165f, 0},
    {TILE_WAVE, 1, 2, 16, 32, 1.0f, 0.055f, 1.3f, 0.12f, 0},
    {TILE_REG, 0, 0, 256, 256, 15.7f, 1.26f, 14.6f, 3.16f, 0},
};

template <int MB, int NB, int KG, int R, bool ODD>
int launch_grid_tile(const uint16_t* a, const uint16_t* b, uint16_t* c, uint32_t m, uint32_t n,
                     uint32_t k, hipStream_t s) {
    const uint32_t tm = cdiv(m, 32 * MB), tn = cdiv(n, 32 * NB);
    constexpr uint32_t ring = R * KG * (32 * MB + 32 * NB) * 64 + 1024, sums = KG == 2 ? 4096 * MB * NB : 0;
    constexpr uint32_t lds = ring > sums ? ring : sums;
    const auto kernel = gemm_bf16_tile_kernel<MB, NB, KG, R, ODD>;
    static std::atomic<bool> ready{false};   // (a failure is not kept: the next call tries again)
    if (!ready.load(std::memory_order_acquire)) {
        MB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        ready.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL(kernel, dim3(tm * tn), dim3(256 * KG), lds, s, a, b, c, m, n, k, tm, tn,
                       std::min(tm, (uint32_t)GM));
    MB_LAUNCH_CHECK("matmul_bf16");
    return MB_OK;
}

template <int MB, int NC>
int launch_wave_tile(const uint16_t* a, const uint16_t* b, uint16_t* c, uint32_t m, uint32_t n,
                     uint32_t k, bool odd, hipStream_t s) {
    const uint32_t tm = cdiv(m, 16 * MB), tn = cdiv(n, 16 * NC), band = std::min(tm, (uint32_t)GM);
    if (odd)
        hipLaunchKernelGGL((gemm_bf16_kwave_kernel<MB, NC, true>), dim3(tm * tn), dim3(64 * KW), 0, s,
                           a, b, c, m, n, k, tm, tn, band);
    else
        hipLaunchKernelGGL((gemm_bf16_kwave_kernel<MB, NC, false>), dim3(tm * tn), dim3(64 * KW), 0, s,
                           a, b, c, m, n, k, tm, tn, band);
    MB_LAUNCH_CHECK("matmul_bf16");
    return MB_OK;
}

// The cheapest tile; `aligned`: 16-byte rows of A and B, c: where C lies.
const TileChoice& choose_tile(uint32_t m, uint32_t n, uint32_t k, bool odd, bool aligned, uintptr_t c) {
    const TileChoice* best = nullptr;
    float least = 0.f;
    for (const TileChoice& t : k_tiles) {
        const bool slow = t.kind == TILE_REG ? !aligned : odd;
        if (slow ? t.odd_c1 == 0.f : t.kind == TILE_EDGE && k % 8) continue;
        const uint64_t tiles = (uint64_t)cdiv(m, t.tm) * cdiv(n, t.tn);
        if (tiles >= 1u << 23) continue;   // 2^32 threads or more (512 to a tile; none of TILE_REG) cannot be launched
        const bool narrow = t.kind == TILE_EDGE ? (n & 7) || (c & 15) : (n & 3) || (c & 7);
        const float cost = (float)((tiles + 255) / 256) *
                           ((slow ? t.odd_c0 + t.odd_c1 * cdiv(k, 32) : t.c0 + t.c1 * cdiv(k, 32)) +
                            (narrow ? t.narrow : 0.f));
        if (!best || cost < least) { best = &t; least = cost; }
    }
    return *best;
}

int launch_tile(const TileChoice& t, const uint16_t* a, const uint16_t* b, uint16_t* c, uint32_t m,
                uint32_t n, uint32_t k, bool odd, hipStream_t s) {
    if (t.kind == TILE_EDGE) {
        const uint32_t tm = cdiv(m, BM), tn = cdiv(n, BN);
        hipLaunchKernelGGL(gemm_bf16_full_kernel<true>, dim3(tm * tn), dim3(256), 0, s, a, b, c, m, n, k,
                           tm, tn);
        MB_LAUNCH_CHECK("matmul_bf16");
        return MB_OK;
    }
    switch (100 * t.kind + 10 * t.mb + t.nb) {
        case 100 * TILE_GRID + 84: return launch_grid_tile<8, 4, 1, 3, false>(a, b, c, m, n, k, s);
        case 100 * TILE_GRID + 44: return odd ? launch_grid_tile<4, 4, 2, 4, true>(a, b, c, m, n, k, s)
                                              : launch_grid_tile<4, 4, 2, 4, false>(a, b, c, m, n, k, s);
        case 100 * TILE_GRID + 43: return odd ? launch_grid_tile<4, 3, 2, 4, true>(a, b, c, m, n, k, s)
                                              : launch_grid_tile<4, 3, 2, 5, false>(a, b, c, m, n, k, s);
        case 100 * TILE_WAVE + 48: return launch_wave_tile<4, 8>(a, b, c, m, n, k, odd, s);
        case 100 * TILE_WAVE + 44: return launch_wave_tile<4, 4>(a, b, c, m, n, k, odd, s);
        case 100 * TILE_WAVE + 24: return launch_wave_tile<2, 4>(a, b, c, m, n, k, odd, s);
        case 100 * TILE_WAVE + 14: return launch_wave_tile<1, 4>(a, b, c, m, n, k, odd, s);
        default: return launch_wave_tile<1, 2>(a, b, c, m, n, k, odd, s);
    }
}

int launch_gemm_bf16(const uint16_t* a, const uint16_t* b, uint16_t* c, uint32_t m, uint32_t n,
                     uint32_t k, hipStream_t s) {
    if (m == 0 || n == 0) return MB_OK;
    if (!a || !b || !c) return fail(MB_E_ARG, "matmul_bf16: null pointer");
    const uint32_t tiles_m = cdiv(m, BM), tiles_n = cdiv(n, BN);
    const uint64_t nblocks = (uint64_t)tiles_m * tiles_n;
    if (nblocks > 0x7fffffffull) return fail(MB_E_ARG, "matmul_bf16: shape too large");
    const bool aligned = (k % 8 == 0) && (n % 8 == 0) &&
                         ((((uintptr_t)a) | ((uintptr_t)b)) & 15) == 0;
    // 32-bit buffer offsets reach every operand, and B's k-rows up to the next multiple
    // of 128 (the deepest stage) without wrapping around to its start
    const bool near = k > 0 && (uint64_t)m * k * 2 < (1ull << 31) && (uint64_t)k * n * 2 < (1ull << 31) &&
                      (uint64_t)m * n * 2 < (1ull << 31) &&
                      (((uint64_t)k + 127) & ~127ull) * n * 2 < (1ull << 32);
    const bool tiles = near && (((uintptr_t)c) & 3) == 0;   // (the k-wave kernel stores dwords)
    // Full 256 x 256 tiles, more than 64 of them (or a C past 2 GB, or off a 4-byte
    // boundary).  Up to 64, one round of tiles a quarter as large or smaller is faster
    // (512 x 6144 x 4096: 66 us on 48 tiles, 36 on 256; 2048^3: 37 and 22); from 65 it
    // takes two rounds (2048 x 4096 x 1024: 23 us and 25).  C may lie anywhere: 4096^3
    // with C 4 or 2 bytes off 94 us (guarded tiles, which store elements, 113;
    // gemm_bf16_kernel 164).
    const bool full = aligned && m % BM == 0 && n % BN == 0 && k % (2 * BK) == 0 && k > 0 &&
                      (uint64_t)m * k * 2 < (1ull << 31) && (uint64_t)k * n * 2 < (1ull << 31);
    if (full && (nblocks > 64 || !tiles)) {
        hipLaunchKernelGGL(gemm_bf16_full_kernel<false>, dim3((uint32_t)nblocks), dim3(256), 0, s, a, b, c,
                           m, n, k, tiles_m, tiles_n);
        MB_LAUNCH_CHECK("matmul_bf16");
        return MB_OK;
    }
    if (tiles) {
        const bool odd = ((k | n) & 1) || ((((uintptr_t)a) | ((uintptr_t)b)) & 3);
        const TileChoice& t = choose_tile(m, n, k, odd, aligned, (uintptr_t)c);
        if (t.kind != TILE_REG) return launch_tile(t, a, b, c, m, n, k, odd, s);
    }
    static bool attr_set[3] = {false, false, false};
    auto go = [&](auto kernel, int mode) -> int {
        if (!attr_set[mode]) {
            MB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)SMEM_BYTES));
            attr_set[mode] = true;
        }
        hipLaunchKernelGGL(kernel, dim3((uint32_t)nblocks), dim3(256), SMEM_BYTES, s, a, b, c, m,
                           n, k, tiles_m, tiles_n);
        MB_LAUNCH_CHECK("matmul_bf16");
        return MB_OK;
    };
    if (aligned) return go(gemm_bf16_kernel<MODE_GUARD>, MODE_GUARD);
    return go(gemm_bf16_kernel<MODE_ELEM>, MODE_ELEM);
}

// Registry launcher: A@0, B@1 (bf16 inputs), C@2 (bf16 output), M@3, N@4, K@5.
int run_gemm_bf16(const Bindings& bs, hipStream_t s, PartMarks*) {
    uint32_t m, n, k;
    int rc;
    if ((rc = bs.u32(3, &m, "M")) || (rc = bs.u32(4, &n, "N")) || (rc = bs.u32(5, &k, "K")))
        return rc;
    void *a, *b, *c;
    if ((rc = bs.buffer(0, MB_DTYPE_BF16, (uint64_t)m * k * 2, false, &a, "A")) ||
        (rc = bs.buffer(1, MB_DTYPE_BF16, (uint64_t)k * n * 2, false, &b, "B")) ||
        (rc = bs.buffer(2, MB_DTYPE_BF16, (uint64_t)m * n * 2, true, &c, "C")))
        return rc;
    return launch_gemm_bf16((const uint16_t*)a, (const uint16_t*)b, (uint16_t*)c, m, n, k, s);
}

}  // namespace

void register_gemm_bf16() {
    register_kernel({"large_matmul_bf16", run_gemm_bf16,
                     reinterpret_cast<const void*>(&gemm_bf16_full_kernel<false>), 1});
}

}  // namespace mb

extern "C" int mb_launch_matmul_bf16(const uint16_t* a, const uint16_t* b, uint16_t* c, uint32_t m,
                                     uint32_t n, uint32_t k, void* stream) {
    mb::clear_error();
    if (!mb::initialized()) return mb::fail(MB_E_STATE, "mb_init() has not been called");
    return mb::launch_gemm_bf16(a, b, c, m, n, k, mb::stream_or_default(stream));
}
