// fp32 transformer sub-ops at the reference's own shapes: row RMSNorm (with an
// optional residual add), RoPE, matrix-vector product, and prefill GQA
// attention, plus the two blocks built from them and the fp32 GEMM family
// (gemm_f32.hip): llama_attention and the prefill llama_decoder_layer.
//
// Specs (reference files; registry bindings in each launcher's comment):
//   rms_norm             mlx/kernels/common/rms_norm.py:7-11 (nn.RMSNorm, unit
//                        gain at init), registry common/registry.py:135-136
//   fused_add_rms_norm   standard/fused_add_rms_norm.py:7-12, registry
//                        standard/registry.py:280-292
//   rope_embedding       standard/rope_embedding.py:15-32, registry
//                        standard/registry.py:103-117
//   matvec               common/matvec.py:9-10, registry common/registry.py:151-162
//   llama_attention      standard/llama_attention.py:18-58, registry
//                        standard/registry.py:398-413
//   llama_decoder_layer  full/llama_decoder_layer.py:17-64, registry
//                        full/registry.py:87-104
//
// gfx950 design.  These shapes are small (the reference runs each in one
// Metal threadgroup), so each op is one or a few short launches:
//  * row ops: one 64-lane wave per row, float4 loads, shuffle reductions;
//  * RoPE angles are formed in fp64 (pos * base^(-2i/D) reaches 127 rad at the
//    reference shape, where an fp32 angle would be off by ~1e-5 rad, i.e. at
//    the registry's atol);
//  * attention: q and k are rotated once, then one workgroup per (head, 16
//    queries) whose waves divide the keys; q.k and p.v are MFMAs, with an
//    online softmax (no mask: the reference attends to every position,
//    standard/llama_attention.py:48-50);
//  * the GEMMs fuse what the blocks put around them: the RMSNorm row scale
//    (from the A operand's own loads), the residual add and SwiGLU.
#include "common.h"

#include <math.h>

#include <algorithm>

namespace mb {
namespace {

constexpr float NEG_BIG = -1.0e30f;   // "no key yet": finite, so max/exp never see inf - inf

// ---- row RMSNorm ---------------------------------------------------------------------------

// y[r] = v * rsqrt(mean(v^2) + eps), v = x[r] (+ res[r]); one wave per row.
template <bool ADD, bool VEC>
__global__ __launch_bounds__(256)
void rms_norm_rows_kernel(const float* __restrict__ x, const float* __restrict__ res,
                          float* __restrict__ y, uint32_t rows, uint32_t cols, float eps) {
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63;
    if (row >= rows) return;   // whole waves only; no barriers in this kernel
    const float* xr = x + (size_t)row * cols;
    const float* rr = ADD ? res + (size_t)row * cols : nullptr;
    float* yr = y + (size_t)row * cols;
    float ss = 0.f;
    if (VEC) {
        for (uint32_t c = 4 * lane; c < cols; c += 256) {
            float4 v = *reinterpret_cast<const float4*>(xr + c);
            if (ADD) {
                const float4 r = *reinterpret_cast<const float4*>(rr + c);
                v.x += r.x; v.y += r.y; v.z += r.z; v.w += r.w;
            }
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
    } else {
        for (uint32_t c = lane; c < cols; c += 64) {
            const float v = xr[c] + (ADD ? rr[c] : 0.f);
            ss += v * v;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float scale = rsqrtf(ss / (float)cols + eps);
    if (VEC) {
        for (uint32_t c = 4 * lane; c < cols; c += 256) {
            float4 v = *reinterpret_cast<const float4*>(xr + c);
            if (ADD) {
                const float4 r = *reinterpret_cast<const float4*>(rr + c);
                v.x += r.x; v.y += r.y; v.z += r.z; v.w += r.w;
            }
            *reinterpret_cast<float4*>(yr + c) =
                make_float4(v.x * scale, v.y * scale, v.z * scale, v.w * scale);
        }
    } else {
        for (uint32_t c = lane; c < cols; c += 64) yr[c] = (xr[c] + (ADD ? rr[c] : 0.f)) * scale;
    }
}

// The same with the row held in registers between the sum and the store: WAVES waves
// per row (the rows of a 256-thread workgroup are 4 / WAVES), NV float4 per lane.  The
// loop above waits for each 256 columns in turn and reads the row twice; here all of a
// row's loads are in flight at once and it is read once.  Up to 1024 columns one wave
// holds the row and adds in the loop's order.
// Bound by latency and, for many wide rows, by memory (4096 x 8192: 4.7 TB/s).  A whole
// residual add and norm, dispatch and wait included, before and after: 8 x 128 14.4 ->
// 14.2 us, 1024 x 1024 15.9 -> 15.4, 4096 x 1024 23.5 -> 20.1, 8 x 4096 18.9 -> 15.0, 4 x
// 8192 23.5 -> 15.1, 4096 x 2048 36.5 -> 27.8, 4096 x 8192 124 -> 85.
template <bool ADD, int WAVES, int NV>
__global__ __launch_bounds__(256)
void rms_norm_held_kernel(const float* __restrict__ x, const float* __restrict__ res,
                          float* __restrict__ y, uint32_t rows, uint32_t cols, float eps) {
    static_assert(WAVES == 1 || WAVES == 4, "a wave or the workgroup per row");
    const uint32_t row = WAVES == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
    const uint32_t t = WAVES == 1 ? threadIdx.x & 63 : threadIdx.x;
    if (row >= rows) return;   // (WAVES = 4: never, one row per workgroup)
    const size_t at = (size_t)row * cols;
    float4 v[NV], r[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const uint32_t c = 4 * (t + 64 * WAVES * i);
        v[i] = r[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (c < cols) {   // cols % 4 == 0: all four columns or none
            v[i] = *reinterpret_cast<const float4*>(x + at + c);
            if (ADD) r[i] = *reinterpret_cast<const float4*>(res + at + c);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if (ADD) { v[i].x += r[i].x; v[i].y += r[i].y; v[i].z += r[i].z; v[i].w += r[i].w; }
        ss += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    if (WAVES == 4) {
        __shared__ float part[4];
        if ((t & 63) == 0) part[t >> 6] = ss;
        __syncthreads();
        ss = part[0] + part[1] + part[2] + part[3];
    }
    const float scale = rsqrtf(ss / (float)cols + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const uint32_t c = 4 * (t + 64 * WAVES * i);
        if (c < cols)
            *reinterpret_cast<float4*>(y + at + c) =
                make_float4(v[i].x * scale, v[i].y * scale, v[i].z * scale, v[i].w * scale);
    }
}

template <bool ADD>
int launch_rms_norm_rows(const float* x, const float* res, float* y, uint32_t rows,
                         uint32_t cols, float eps, hipStream_t s) {
    if (rows == 0 || cols == 0) return MB_OK;
    const bool vec = cols % 4 == 0 &&
                     (((uintptr_t)x | (uintptr_t)res | (uintptr_t)y) & 15) == 0;
    const dim3 grid(cdiv(rows, 4)), block(256);
    auto held = [&](auto kernel, uint32_t groups) {
        hipLaunchKernelGGL(kernel, dim3(groups), block, 0, s, x, res, y, rows, cols, eps);
    };
    // Rows of up to 8 float4 per lane stay in registers: at every width measured, 128 to
    // 8192 columns, faster than the loop (figures at the kernel).  A wave's four float4
    // reach 1024 columns, a workgroup's eight 8192; a workgroup per row only while the
    // launch has fewer than 2^32 threads.
    if (vec && cols <= 256) held(rms_norm_held_kernel<ADD, 1, 1>, grid.x);
    else if (vec && cols <= 512) held(rms_norm_held_kernel<ADD, 1, 2>, grid.x);
    else if (vec && cols <= 1024) held(rms_norm_held_kernel<ADD, 1, 4>, grid.x);
    else if (vec && cols <= 2048 && rows < 1u << 24) held(rms_norm_held_kernel<ADD, 4, 2>, rows);
    else if (vec && cols <= 4096 && rows < 1u << 24) held(rms_norm_held_kernel<ADD, 4, 4>, rows);
    else if (vec && cols <= 8192 && rows < 1u << 24) held(rms_norm_held_kernel<ADD, 4, 8>, rows);
    else if (vec) hipLaunchKernelGGL((rms_norm_rows_kernel<ADD, true>), grid, block, 0, s, x, res, y, rows, cols, eps);
    else hipLaunchKernelGGL((rms_norm_rows_kernel<ADD, false>), grid, block, 0, s, x, res, y, rows, cols, eps);
    MB_LAUNCH_CHECK("rms_norm");
    return MB_OK;
}

// ---- RoPE over rows (position = row index) --------------------------------------------------

// out[p][2i], out[p][2i+1] = rotation of the pair by p * base^(-2i/D).
__global__ __launch_bounds__(256)
void rope_rows_kernel(const float* __restrict__ x, float* __restrict__ y, uint32_t S, uint32_t D,
                      double base) {
    const uint32_t half = D / 2;
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (uint64_t)S * half) return;
    const uint32_t p = (uint32_t)(idx / half), i = (uint32_t)(idx % half);
    const double omega = pow(base, -2.0 * (double)i / (double)D);
    double sn, cs;
    sincos((double)p * omega, &sn, &cs);
    const float2 v = *reinterpret_cast<const float2*>(x + (size_t)p * D + 2 * i);
    *reinterpret_cast<float2*>(y + (size_t)p * D + 2 * i) =
        make_float2((float)(v.x * cs - v.y * sn), (float)(v.x * sn + v.y * cs));
}

// ---- matrix-vector product -------------------------------------------------------------------

// y[m] = sum_k A[m][k] x[k]; one wave per row.
template <bool VEC>
__global__ __launch_bounds__(256)
void matvec_kernel(const float* __restrict__ A, const float* __restrict__ x, float* __restrict__ y,
                   uint32_t M, uint32_t K) {
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63;
    if (row >= M) return;   // whole waves only; no barriers in this kernel
    const float* ar = A + (size_t)row * K;
    float acc = 0.f;
    if (VEC) {
        for (uint32_t c = 4 * lane; c < K; c += 256) {
            const float4 a = *reinterpret_cast<const float4*>(ar + c);
            const float4 v = *reinterpret_cast<const float4*>(x + c);
            acc += a.x * v.x + a.y * v.y + a.z * v.z + a.w * v.w;
        }
    } else {
        for (uint32_t c = lane; c < K; c += 64) acc += ar[c] * x[c];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) y[row] = acc;
}

// ---- prefill GQA attention -------------------------------------------------------------------

// T is the arithmetic of the attention: q, k, v, the rotation, q.k, the online
// softmax and p.v (float, or double for the decoder layer, see
// run_llama_decoder_layer); the output is fp32.
template <typename T>
struct AttnPrefillArgs {
    const T* qkv;       // [S][ldq]: q at column h*Dh, k at D + kvh*Dh, v at D + Hkv*Dh + kvh*Dh;
                        // q and k already rotated by their row (ROT: not yet)
    float* out;         // [S][ldo]: head h at column h*Dh
    uint32_t S, D, H, Hkv, ldq, ldo;
    T scale;            // 1 / sqrt(Dh)
    double base;        // ROT: RoPE base
};

constexpr int QW = 16;   // queries per workgroup

template <typename T> __device__ __forceinline__ T exp_t(T v);
template <> __device__ __forceinline__ float exp_t<float>(float v) { return expf(v); }
template <> __device__ __forceinline__ double exp_t<double>(double v) { return exp(v); }

// 16 x 16 outputs, 4 deep: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and the
// four outputs D[row][l % 16], row = mfma_row(r, l / 16).
template <typename T> struct Mfma;
template <> struct Mfma<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc run(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t row(int r, uint32_t g) { return 4 * g + r; }
};
template <> struct Mfma<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc run(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t row(int r, uint32_t g) { return 4 * r + g; }
};

// Workgroup (head h, 16 queries); its waves divide the keys, 32 at a time each with an
// online softmax, and are merged through LDS.  All products are
// MFMAs in T:
//  * scores: A = 16 keys, B = the 16 queries; lane (t, g) = (l % 16, l / 16) of the d
//    order d = 4 V s + V g + e (V elements in 16 bytes), so operands are whole 16-byte
//    loads.  Lane (t, g) then holds query t's scores of keys row(r, g);
//  * p v: those four registers are the A operand as they are (query t, key row(r, g)),
//    B = v's rows of the same keys, lane t holding d = NV t .. NV t + NV - 1 (whole rows
//    are contiguous).  Lane (t, g) holds query row(r, g), d = NV t + b.
// q and k come rotated.  512 tokens, 16 heads of 64 on 4: 22.6 us, of which fp32 MFMA
// needs 7.  (68 us when the keys were rotated here, with an fp64 sine and cosine per pair
// again for every head and 16 queries, and the products were vector FMAs over LDS.)  What
// remains is the chain load, MFMA, softmax, MFMA of a wave: fetching the values and the
// next keys ahead costs registers (25.2), and a row pitch that spreads the 16 rows of a
// load over the L2 channels changes nothing.
// fp32: eight waves (four: 5 us more on the whole attention at 32 keys a step); fp64: four,
// whose partial outputs for Dh 128 fill 64 KB of LDS.
// ROT (fp32, at most ROT_PAIRS positions x pairs): the workgroup forms the table of all
// sines and cosines first, at most eight per thread, which takes less than the launch that
// rotates longer inputs (16 tokens, 4 heads of 32: 24.5 us in all, 27.8 with that launch; at
// the line the two meet: 64 tokens of 2 heads of 128 33.4, 65 tokens with the launch 34.0).
constexpr uint32_t ROT_PAIRS = 4096;
template <typename T> constexpr int attn_waves() { return sizeof(T) == 4 ? 8 : 4; }
template <int DH, typename T, bool ROT>
__global__ __launch_bounds__(64 * attn_waves<T>())
void attention_prefill_kernel(AttnPrefillArgs<T> a) {
    constexpr int V = 16 / (int)sizeof(T), NS = DH / (4 * V), NV = DH / 16;
    constexpr int KT = 2;            // key tiles of 16 per step (4: 0.5 us more)
    typedef typename Mfma<T>::acc Acc;
    struct alignas(16) Chunk { T v[V]; };
    constexpr uint32_t W = attn_waves<T>();
    __shared__ T po[W][QW][DH];      // per wave: unnormalised output
    __shared__ T pm[W][QW], pl[W][QW];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t t = lane & 15, g = lane >> 4;
    const uint32_t h = blockIdx.x, kvh = h / (a.H / a.Hkv), q0 = blockIdx.y * QW;
    const T* kbase = a.qkv + a.D + kvh * DH;
    const T* vbase = kbase + a.Hkv * DH;

    constexpr uint32_t RP = DH / 2 + 2;   // table pitch (banks; rows stay 16-byte aligned)
    __shared__ alignas(16) float2 rot[ROT ? ROT_PAIRS / (DH / 2) * RP : 1];
    if constexpr (ROT) {
        __shared__ double omega[DH / 2];
        if (tid < DH / 2) omega[tid] = pow(a.base, -2.0 * (double)tid / (double)DH);
        __syncthreads();
        for (uint32_t e = tid; e < a.S * (DH / 2); e += 64 * W) {
            const uint32_t pos = e / (DH / 2), j = e % (DH / 2);
            double sn, cs;
            sincos((double)pos * omega[j], &sn, &cs);
            rot[pos * RP + j] = make_float2((float)cs, (float)sn);
        }
        __syncthreads();
    }
    const auto turn = [&](Chunk& c, uint32_t pos, int s) {   // d = 4 V s + V g ..
        if constexpr (ROT) {
#pragma unroll
            for (int p = 0; p < V / 2; ++p) {
                const float2 f = rot[pos * RP + (4 * V * s + V * g) / 2 + p];
                const T x = c.v[2 * p], y = c.v[2 * p + 1];
                c.v[2 * p] = x * f.x - y * f.y;
                c.v[2 * p + 1] = x * f.y + y * f.x;
            }
        }
    };
    T q[NS][V];
    {
        const uint32_t pos = min(q0 + t, a.S - 1);
        const T* src = a.qkv + (size_t)pos * a.ldq + h * DH + V * g;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            Chunk c = *reinterpret_cast<const Chunk*>(src + 4 * V * s);
            turn(c, pos, s);
#pragma unroll
            for (int e = 0; e < V; ++e) q[s][e] = c.v[e];
        }
    }
    Acc o[NV];
#pragma unroll
    for (int b = 0; b < NV; ++b) o[b] = Acc{};
    T m_run = (T)NEG_BIG, l_run = 0;   // query t (l: this lane's keys)
    const uint32_t per = (a.S + 16 * W - 1) / (16 * W) * 16;                       // keys per wave
    const uint32_t k_begin = min(wave * per, a.S), k_end = min(k_begin + per, a.S);

    for (uint32_t k0 = k_begin; k0 < k_end; k0 += 16 * KT) {
        Acc sc[KT];
#pragma unroll
        for (int x = 0; x < KT; ++x) {
            sc[x] = Acc{};
            if (k0 + 16 * x >= k_end) continue;   // (uniform)
            const uint32_t pos = min(k0 + 16 * x + t, a.S - 1);
            const T* src = kbase + (size_t)pos * a.ldq + V * g;
            Chunk c[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) c[s] = *reinterpret_cast<const Chunk*>(src + 4 * V * s);
#pragma unroll
            for (int s = 0; s < NS; ++s) turn(c[s], pos, s);
            // one chain per element of a chunk, added pairwise: shorter sums (one chain for
            // all of Dh: 62 tokens, 4 heads of 128 4.2e-7 against 64 bits, so 3.1e-7)
            Acc part[V];
#pragma unroll
            for (int e = 0; e < V; ++e) part[e] = Acc{};
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int e = 0; e < V; ++e) part[e] = Mfma<T>::run(c[s].v[e], q[s][e], part[e]);
            sc[x] = V == 4 ? (part[0] + part[1]) + (part[V - 2] + part[V - 1]) : part[0] + part[1];
        }
        T mx = (T)NEG_BIG;
#pragma unroll
        for (int x = 0; x < KT; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool ok = k0 + 16 * x + Mfma<T>::row(r, g) < k_end;
                sc[x][r] = ok ? sc[x][r] * a.scale : (T)NEG_BIG;
                mx = mx > sc[x][r] ? mx : sc[x][r];
            }
#pragma unroll
        for (int o2 = 16; o2 < 64; o2 <<= 1) {
            const T other = __shfl_xor(mx, o2);
            mx = mx > other ? mx : other;
        }
        const T m_new = m_run > mx ? m_run : mx;
        const T alpha = exp_t<T>(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int x = 0; x < KT; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool ok = k0 + 16 * x + Mfma<T>::row(r, g) < k_end;
                sc[x][r] = ok ? exp_t<T>(sc[x][r] - m_new) : (T)0;
                l_run += sc[x][r];
            }
        m_run = m_new;
        T al[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) al[r] = __shfl(alpha, (int)Mfma<T>::row(r, g));
#pragma unroll
        for (int b = 0; b < NV; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[b][r] *= al[r];
#pragma unroll
        for (int x = 0; x < KT; ++x) {
            if (k0 + 16 * x >= k_end) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // rows past the last key: its values, zeroed (an infinity there would make NaN)
                const uint32_t key = k0 + 16 * x + Mfma<T>::row(r, g);
                const T* src = vbase + (size_t)min(key, a.S - 1) * a.ldq + NV * t;
                struct alignas(NV * sizeof(T) < 16 ? NV * sizeof(T) : 16) Row { T v[NV]; };
                const Row v = *reinterpret_cast<const Row*>(src);
#pragma unroll
                for (int b = 0; b < NV; ++b)
                    o[b] = Mfma<T>::run(sc[x][r], key < a.S ? v.v[b] : (T)0, o[b]);
            }
        }
    }
    // the waves' parts, weighted by exp(their maximum - the maximum)
#pragma unroll
    for (int o2 = 16; o2 < 64; o2 <<= 1) l_run += __shfl_xor(l_run, o2);
    if (g == 0) { pm[wave][t] = m_run; pl[wave][t] = l_run; }
#pragma unroll
    for (int b = 0; b < NV; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) po[wave][Mfma<T>::row(r, g)][NV * t + b] = o[b][r];
    __syncthreads();
    for (uint32_t e = tid; e < QW * DH; e += 64 * W) {
        const uint32_t qq = e / DH, d = e % DH;
        if (q0 + qq >= a.S) break;
        T m = pm[0][qq];
#pragma unroll
        for (uint32_t w = 1; w < W; ++w) m = m > pm[w][qq] ? m : pm[w][qq];
        T sum = 0, l = 0;
#pragma unroll
        for (uint32_t w = 0; w < W; ++w) {
            const T f = exp_t<T>(pm[w][qq] - m);
            sum += f * po[w][qq][d];
            l += f * pl[w][qq];
        }
        a.out[(size_t)(q0 + qq) * a.ldo + h * DH + d] = (float)(sum / l);
    }
}

// q and k of qkv [S][ldq] (the first `heads` blocks of Dh columns) rotated in place by
// their row: pairs (2j, 2j + 1) by pos * base^(-2j/Dh), the angle and its sine and
// cosine in fp64 (an fp32 angle is off by ~pos * 6e-8 rad).
__global__ __launch_bounds__(256)
void rope_qk_kernel(float* __restrict__ qkv, uint32_t S, uint32_t heads, uint32_t dh, uint32_t ldq,
                    double base) {
    const uint32_t half = dh / 2, per = heads < 4 ? heads : 4;   // heads per thread
    const uint32_t groups = (heads + per - 1) / per;
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (uint64_t)S * half * groups) return;
    const uint32_t j = (uint32_t)(idx % half), h0 = (uint32_t)(idx / half % groups) * per;
    const uint32_t pos = (uint32_t)(idx / half / groups);
    double sn, cs;
    sincos((double)pos * pow(base, -2.0 * (double)j / (double)dh), &sn, &cs);
    const float c = (float)cs, s = (float)sn;
    float* row = qkv + (size_t)pos * ldq + 2 * j;
    for (uint32_t h = h0; h < min(h0 + per, heads); ++h) {
        float2* at = reinterpret_cast<float2*>(row + h * dh);
        const float2 v = *at;
        *at = make_float2(v.x * c - v.y * s, v.x * s + v.y * c);
    }
}

template <typename T, bool ROT>
int launch_attention_prefill(const AttnPrefillArgs<T>& a, uint32_t dh, hipStream_t s) {
    if (a.S == 0) return MB_OK;
    const dim3 grid(a.H, cdiv(a.S, QW)), block(64 * attn_waves<T>());
    switch (dh) {
        case 32: hipLaunchKernelGGL((attention_prefill_kernel<32, T, ROT>), grid, block, 0, s, a); break;
        case 64: hipLaunchKernelGGL((attention_prefill_kernel<64, T, ROT>), grid, block, 0, s, a); break;
        case 128: hipLaunchKernelGGL((attention_prefill_kernel<128, T, ROT>), grid, block, 0, s, a); break;
        default: return fail(MB_E_ARG, "attention: head dim %u not 32, 64 or 128", dh);
    }
    MB_LAUNCH_CHECK("attention prefill");
    return MB_OK;
}

// ---- fp64 RMSNorm GEMM (the decoder layer's q|k|v projection) -----------------------------

// C[S][N] = rmsnorm(A) B in fp64 from fp32 A [S][K] and B [K][N]: each
// workgroup computes a (16 TR) x (16 TC) tile, thread (ty, tx) the TR x TC
// outputs of rows TR ty .. TR ty + TR - 1 and columns TC tx + j; A and B go
// through LDS 32 k at a time, widened to fp64 on the way in, and the next
// chunk's global loads are in flight while the current one is multiplied.
// The row scale rsqrt(mean(a^2) + eps) is accumulated from the same A chunks.
// (With 64 x 64 tiles and each chunk loaded only after the previous one was
// multiplied, the decoder layer's 64 x 256 x 128 projection ran on 4
// workgroups and took 23.8 us, four load round trips in a row.)
constexpr int GK = 32;

// The first `rot` columns (q and k, heads of dh) are rotated by their row on the way
// out: pairs (2j, 2j + 1) by row * base^(-2j/dh).
template <int TR>   // rows per thread: a (16 TR) x 32 tile
__global__ __launch_bounds__(256)
void rms_gemm_f64_kernel(const float* __restrict__ A, const float* __restrict__ B,
                         double* __restrict__ C, uint32_t S, uint32_t N, uint32_t K,
                         float eps, uint32_t rot, uint32_t dh, double base) {
    constexpr int TC = 2, GR = 16 * TR, GC = 16 * TC;
    constexpr int RT = 256 / GR;      // threads per row for the sums of squares
    __shared__ double as[GR][GK + 1];
    __shared__ double bs[GK][GC + 1];
    __shared__ double rs[GR];
    const uint32_t tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    const uint32_t row0 = blockIdx.y * GR, col0 = blockIdx.x * GC;
    constexpr int LA = GR * GK / 256, LB = GK * GC / 256;   // elements per thread per chunk
    float ra[LA], rb[LB];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const uint32_t e = tid + 256 * i, r = e / GK, c = e % GK;
            const uint32_t gr = row0 + r, gk = k0 + c;
            ra[i] = (gr < S && gk < K) ? A[(size_t)gr * K + gk] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const uint32_t e = tid + 256 * i, kr = e / GC, nc = e % GC;
            rb[i] = (k0 + kr < K && col0 + nc < N) ? B[(size_t)(k0 + kr) * N + col0 + nc] : 0.f;
        }
    };
    double acc[TR][TC] = {};
    double ss = 0;   // sum of squares of row tid / RT, k part (tid % RT) of each chunk
    load(0);
    for (uint32_t k0 = 0; k0 < K; k0 += GK) {
        __syncthreads();   // the previous chunk is no longer read
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const uint32_t e = tid + 256 * i;
            as[e / GK][e % GK] = (double)ra[i];
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const uint32_t e = tid + 256 * i;
            bs[e / GC][e % GC] = (double)rb[i];
        }
        __syncthreads();
        if (k0 + GK < K) load(k0 + GK);
#pragma unroll
        for (int c = 0; c < GK / RT; ++c) {
            const double v = as[tid / RT][(tid % RT) * (GK / RT) + c];
            ss += v * v;
        }
#pragma unroll 4
        for (int kk = 0; kk < GK; ++kk) {
            double av[TR], bv[TC];
#pragma unroll
            for (int i = 0; i < TR; ++i) av[i] = as[TR * ty + i][kk];
#pragma unroll
            for (int j = 0; j < TC; ++j) bv[j] = bs[kk][2 * tx + j];
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] += av[i] * bv[j];
        }
    }
#pragma unroll
    for (int o2 = 1; o2 < RT; o2 <<= 1) ss += __shfl_xor(ss, o2);
    if (tid % RT == 0) rs[tid / RT] = 1.0 / sqrt(ss / (double)K + (double)eps);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TR; ++i) {
        const uint32_t r = row0 + TR * ty + i;
        if (r >= S) continue;
        const uint32_t c = col0 + 2 * tx;
        double v0 = acc[i][0] * rs[TR * ty + i], v1 = acc[i][1] * rs[TR * ty + i];
        if (c < rot) {   // (rot and N are even: a pair is rotated or not, stored or not)
            double sn, cs;
            sincos((double)r * pow(base, -2.0 * (double)(c % dh / 2) / (double)dh), &sn, &cs);
            const double x = v0;
            v0 = x * cs - v1 * sn;
            v1 = x * sn + v1 * cs;
        }
        if (c < N) *reinterpret_cast<double2*>(C + (size_t)r * N + c) = make_double2(v0, v1);
    }
}

int launch_rms_gemm_f64(const float* a, const float* b, double* c, uint32_t S, uint32_t N,
                        uint32_t K, float eps, uint32_t rot, uint32_t dh, double base,
                        hipStream_t s) {
    if (S == 0 || N == 0) return MB_OK;
    if (K == 0) return fail(MB_E_ARG, "rms gemm: K must be positive");
    // 16 x 32 tiles: 32 workgroups at the registry's 64 x 256 (34 us for the
    // layer, against 35-36 us with 32 x 32 or 32 x 64 tiles and 16 x 64)
    hipLaunchKernelGGL((rms_gemm_f64_kernel<1>), dim3(cdiv(N, 32), cdiv(S, 16)), dim3(256), 0,
                       s, a, b, c, S, N, K, eps, rot, dh, base);
    MB_LAUNCH_CHECK("rms_gemm_f64");
    return MB_OK;
}

// Shape checks shared by llama_attention and llama_decoder_layer.
int check_heads(uint32_t S, uint32_t D, uint32_t H, uint32_t HKV, uint32_t* dh) {
    if (S == 0 || D == 0 || H == 0 || HKV == 0 || D % H || H % HKV)
        return fail(MB_E_ARG, "attention: S %u, D %u, H %u, H_kv %u: need D %% H == 0 and "
                    "H %% H_kv == 0", S, D, H, HKV);
    *dh = D / H;
    if (*dh != 32 && *dh != 64 && *dh != 128)
        return fail(MB_E_ARG, "attention: head dim %u not 32, 64 or 128", *dh);
    if (S > 65535u * QW) return fail(MB_E_ARG, "attention: S %u too large", S);
    return MB_OK;
}

// ---- registry launchers ----------------------------------------------------------------------

// rms_norm: x@0 [rows][cols], y@1, cols@2, eps@3 (rows = x's size / cols).
int run_rms_norm(const Bindings& bs, hipStream_t s, PartMarks*) {
    uint32_t cols;
    float eps;
    int rc;
    if ((rc = bs.u32(2, &cols, "cols")) || (rc = bs.f32(3, &eps, "eps"))) return rc;
    if (cols == 0) return fail(MB_E_ARG, "rms_norm: cols must be positive");
    const uint64_t rows = bs.nbytes(0) / ((uint64_t)cols * 4);
    void *x, *y;
    if ((rc = bs.buffer(0, MB_DTYPE_F32, rows * cols * 4, false, &x, "x")) ||
        (rc = bs.buffer(1, MB_DTYPE_F32, rows * cols * 4, true, &y, "y")))
        return rc;
    return launch_rms_norm_rows<false>((const float*)x, nullptr, (float*)y, (uint32_t)rows, cols,
                                       eps, s);
}

// fused_add_rms_norm: x@0, residual@1 [rows][cols], y@2, cols@3, eps@4.
int run_fused_add_rms_norm(const Bindings& bs, hipStream_t s, PartMarks*) {
    uint32_t cols;
    float eps;
    int rc;
    if ((rc = bs.u32(3, &cols, "cols")) || (rc = bs.f32(4, &eps, "eps"))) return rc;
    if (cols == 0) return fail(MB_E_ARG, "fused_add_rms_norm: cols must be positive");
    const uint64_t rows = bs.nbytes(0) / ((uint64_t)cols * 4);
    void *x, *r, *y;
    if ((rc = bs.buffer(0, MB_DTYPE_F32, rows * cols * 4, false, &x, "x")) ||
        (rc = bs.buffer(1, MB_DTYPE_F32, rows * cols * 4, false, &r, "residual")) ||
        (rc = bs.buffer(2, MB_DTYPE_F32, rows * cols * 4, true, &y, "y")))
        return rc;
    return launch_rms_norm_rows<true>((const float*)x, (const float*)r, (float*)y,
                                      (uint32_t)rows, cols, eps, s);
}

// rope_embedding: x@0 [S][D], y@1, S@2, D@3, base@4.
int run_rope(const Bindings& bs, hipStream_t s, PartMarks*) {
    uint32_t S, D;
    float base;
    int rc;
    if ((rc = bs.u32(2, &S, "S")) || (rc = bs.u32(3, &D, "D")) || (rc = bs.f32(4, &base, "base")))
        return rc;
    if (D % 2) return fail(MB_E_ARG, "rope_embedding: D %u must be even", D);
    if (!(base > 0.f)) return fail(MB_E_ARG, "rope_embedding: base must be > 0");
    void *x, *y;
    if ((rc = bs.buffer(0, MB_DTYPE_F32, (uint64_t)S * D * 4, false, &x, "x")) ||
        (rc = bs.buffer(1, MB_DTYPE_F32, (uint64_t)S * D * 4, true, &y, "y")))
        return rc;
    const uint64_t pairs = (uint64_t)S * (D / 2);
    if (pairs == 0) return MB_OK;
    if (pairs > 0xffffffffull) return fail(MB_E_ARG, "rope_embedding: shape too large");
    if (((uintptr_t)x | (uintptr_t)y) & 7) return fail(MB_E_ARG, "rope_embedding: unaligned buffers");
    hipLaunchKernelGGL(rope_rows_kernel, dim3((uint32_t)((pairs + 255) / 256)), dim3(256), 0, s,
                       (const float*)x, (float*)y, S, D, (double)base);
    MB_LAUNCH_CHECK("rope_embedding");
    return MB_OK;
}

// matvec: A@0 [M][K], x@1 [K], y@2 [M], K@3 (M = y's size).
int run_matvec(const Bindings& bs, hipStream_t s, PartMarks*) {
    uint32_t K;
    int rc;
    if ((rc = bs.u32(3, &K, "K"))) return rc;
    const uint64_t M = bs.nbytes(2) / 4;
    void *A, *x, *y;
    if ((rc = bs.buffer(0, MB_DTYPE_F32, M * K * 4, false, &A, "A")) ||
        (rc = bs.buffer(1, MB_DTYPE_F32, (uint64_t)K * 4, false, &x, "x")) ||
        (rc = bs.buffer(2, MB_DTYPE_F32, M * 4, true, &y, "y")))
        return rc;
    if (M == 0) return MB_OK;
    if (M > 0x7ffffffcull) return fail(MB_E_ARG, "matvec: M too large");
    const bool vec = K % 4 == 0 && (((uintptr_t)A | (uintptr_t)x) & 15) == 0;
    const dim3 grid(cdiv((uint32_t)M, 4)), block(256);
    if (vec) hipLaunchKernelGGL(matvec_kernel<true>, grid, block, 0, s, (const float*)A, (const float*)x, (float*)y, (uint32_t)M, K);
    else hipLaunchKernelGGL(matvec_kernel<false>, grid, block, 0, s, (const float*)A, (const float*)x, (float*)y, (uint32_t)M, K);
    MB_LAUNCH_CHECK("matvec");
    return MB_OK;
}

// llama_attention: x@0 [S][D], W_qkv@1 [D][D + 2 Hkv Dh], W_o@2 [D][D], y@3
// [S][D], S@4, D@5, H@6, H_kv@7, base@8.  y = attention(x W_qkv) W_o (no
// norm, no residual: standard/llama_attention.py:30-52).
int run_llama_attention(const Bindings& bs, hipStream_t s, PartMarks*) {
    uint32_t S, D, H, HKV, dh;
    float base;
    int rc;
    if ((rc = bs.u32(4, &S, "S")) || (rc = bs.u32(5, &D, "D")) || (rc = bs.u32(6, &H, "H")) ||
        (rc = bs.u32(7, &HKV, "H_kv")) || (rc = bs.f32(8, &base, "base")))
        return rc;
    if ((rc = check_heads(S, D, H, HKV, &dh))) return rc;
    const uint32_t nqkv = D + 2 * HKV * dh;
    void *x, *wqkv, *wo, *y;
    if ((rc = bs.buffer(0, MB_DTYPE_F32, (uint64_t)S * D * 4, false, &x, "x")) ||
        (rc = bs.buffer(1, MB_DTYPE_F32, (uint64_t)D * nqkv * 4, false, &wqkv, "W_qkv")) ||
        (rc = bs.buffer(2, MB_DTYPE_F32, (uint64_t)D * D * 4, false, &wo, "W_o")) ||
        (rc = bs.buffer(3, MB_DTYPE_F32, (uint64_t)S * D * 4, true, &y, "y")))
        return rc;
    const size_t qkv_bytes = ((size_t)S * nqkv * 4 + 255) & ~(size_t)255;
    uint8_t* ws = static_cast<uint8_t*>(library_workspace(qkv_bytes + (size_t)S * D * 4));
    if (!ws) return MB_E_HIP;
    float* qkv = reinterpret_cast<float*>(ws);
    float* attn = reinterpret_cast<float*>(ws + qkv_bytes);
    if ((rc = launch_gemm_f32_ex(gemm_f32_args((const float*)x, (const float*)wqkv, qkv, S, nqkv, D),
                                 GEMM_F32_PLAIN, 1, s)))
        return rc;
    AttnPrefillArgs<float> a{qkv, attn, S, D, H, HKV, nqkv, D, 1.0f / sqrtf((float)dh), (double)base};
    if ((uint64_t)S * (dh / 2) <= ROT_PAIRS) {
        if ((rc = launch_attention_prefill<float, true>(a, dh, s))) return rc;
    } else {
        const uint32_t heads = H + HKV;
        const uint64_t pairs = (uint64_t)S * (dh / 2) * cdiv(heads, std::min(heads, 4u));
        hipLaunchKernelGGL(rope_qk_kernel, dim3((uint32_t)((pairs + 255) / 256)), dim3(256), 0, s,
                           qkv, S, heads, dh, nqkv, (double)base);
        MB_LAUNCH_CHECK("rope q, k");
        if ((rc = launch_attention_prefill<float, false>(a, dh, s))) return rc;
    }
    return launch_gemm_f32_ex(gemm_f32_args(attn, (const float*)wo, (float*)y, S, D, D),
                              GEMM_F32_PLAIN, 1, s);
}

// llama_decoder_layer (prefill): x@0 [S][D], W_qkv@1, W_o@2, W_gu@3 [D][2 FF]
// ([gate | up]), W_down@4 [FF][D], y@5 [S][D], S@6, D@7, H@8, H_kv@9, FF@10,
// base@11, eps@12.  Five launches:
//   qkv  = rmsnorm(x) W_qkv                    (fp64, RMS row scale in the GEMM)
//   attn = attention(RoPE(q), RoPE(k), v)      (fp64 logits and softmax)
// The attention logits are the ill-conditioned part of this entry: with the
// reference's normal(0, 1) weights q.k / sqrt(Dh) reaches the hundreds, so
// fp32 rounding of q, k and the dot products moves the softmax weights of
// near-tied keys, and the FFN amplifies it; an all-fp32 evaluation of the
// layer lands ~0.15 from float64 on outputs of up to ~6000, one with fp64 q|k|v
// and logits ~0.004.  At S = 64, D = 128 the fp64 work is a few hundred
// thousand multiply-adds.
//   x1   = x + attn W_o                        (residual in the epilogue)
//   act  = silu(rmsnorm(x1) W_gate) * (rmsnorm(x1) W_up)
//   y    = x1 + act W_down
int run_llama_decoder_layer(const Bindings& bs, hipStream_t s, PartMarks* pm) {
    uint32_t S, D, H, HKV, FF, dh;
    float base, eps;
    int rc;
    if ((rc = bs.u32(6, &S, "S")) || (rc = bs.u32(7, &D, "D")) || (rc = bs.u32(8, &H, "H")) ||
        (rc = bs.u32(9, &HKV, "H_kv")) || (rc = bs.u32(10, &FF, "FF")) ||
        (rc = bs.f32(11, &base, "base")) || (rc = bs.f32(12, &eps, "eps")))
        return rc;
    if ((rc = check_heads(S, D, H, HKV, &dh))) return rc;
    if (FF == 0) return fail(MB_E_ARG, "llama_decoder_layer: FF must be positive");
    const uint32_t nqkv = D + 2 * HKV * dh;
    void *x, *wqkv, *wo, *wgu, *wdown, *y;
    if ((rc = bs.buffer(0, MB_DTYPE_F32, (uint64_t)S * D * 4, false, &x, "x")) ||
        (rc = bs.buffer(1, MB_DTYPE_F32, (uint64_t)D * nqkv * 4, false, &wqkv, "W_qkv")) ||
        (rc = bs.buffer(2, MB_DTYPE_F32, (uint64_t)D * D * 4, false, &wo, "W_o")) ||
        (rc = bs.buffer(3, MB_DTYPE_F32, (uint64_t)D * 2 * FF * 4, false, &wgu, "W_gu")) ||
        (rc = bs.buffer(4, MB_DTYPE_F32, (uint64_t)FF * D * 4, false, &wdown, "W_down")) ||
        (rc = bs.buffer(5, MB_DTYPE_F32, (uint64_t)S * D * 4, true, &y, "y")))
        return rc;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t o_qkv = 0, o_attn = al((size_t)S * nqkv * 8),
                 o_x1 = o_attn + al((size_t)S * D * 4), o_act = o_x1 + al((size_t)S * D * 4),
                 total = o_act + al((size_t)S * FF * 4);
    uint8_t* ws = static_cast<uint8_t*>(library_workspace(total));
    if (!ws) return MB_E_HIP;
    double* qkv = reinterpret_cast<double*>(ws + o_qkv);
    float* attn = reinterpret_cast<float*>(ws + o_attn);
    float* x1 = reinterpret_cast<float*>(ws + o_x1);
    float* act = reinterpret_cast<float*>(ws + o_act);
    auto mark = [&](const char* n) { if (pm) pm->mark(s, n); };

    mark("qkv_rmsnorm");
    if ((rc = launch_rms_gemm_f64((const float*)x, (const float*)wqkv, qkv, S, nqkv, D, eps,
                                  D + HKV * dh, dh, (double)base, s)))
        return rc;
    mark("attention");
    AttnPrefillArgs<double> a{qkv, attn, S, D, H, HKV, nqkv, D, 1.0 / sqrt((double)dh), 0.0};
    if ((rc = launch_attention_prefill<double, false>(a, dh, s))) return rc;
    mark("wo_residual");
    GemmF32Args g = gemm_f32_args(attn, (const float*)wo, x1, S, D, D);
    g.r = (const float*)x;
    if ((rc = launch_gemm_f32_ex(g, GEMM_F32_RESID, 1, s))) return rc;
    mark("gate_up_swiglu");
    g = gemm_f32_args(x1, (const float*)wgu, act, S, FF, D);
    g.b2 = (const float*)wgu + FF;
    g.ldb = 2 * FF;
    g.eps = eps;
    if ((rc = launch_gemm_f32_ex(g, GEMM_F32_RMS_SWIGLU, 1, s))) return rc;
    mark("down_residual");
    g = gemm_f32_args(act, (const float*)wdown, (float*)y, S, D, FF);
    g.r = x1;
    return launch_gemm_f32_ex(g, GEMM_F32_RESID, 1, s);
}

}  // namespace

void register_transformer_f32() {
    register_kernel({"rms_norm_f32", run_rms_norm,
                     reinterpret_cast<const void*>(&rms_norm_held_kernel<false, 1, 4>), 1});
    register_kernel({"fused_add_rms_norm_f32", run_fused_add_rms_norm,
                     reinterpret_cast<const void*>(&rms_norm_held_kernel<true, 1, 4>), 1});
    register_kernel({"rope_embedding_f32", run_rope,
                     reinterpret_cast<const void*>(&rope_rows_kernel), 1});
    register_kernel({"matvec_f32", run_matvec,
                     reinterpret_cast<const void*>(&matvec_kernel<true>), 1});
    register_kernel({"llama_attention_f32", run_llama_attention,
                     reinterpret_cast<const void*>(&attention_prefill_kernel<32, float, true>), 1});
    register_kernel({"llama_decoder_layer_f32", run_llama_decoder_layer,
                     reinterpret_cast<const void*>(&attention_prefill_kernel<32, double, false>), 5});
}

}  // namespace mb
