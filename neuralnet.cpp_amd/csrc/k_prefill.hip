// k_prefill.hip — batched prefill of the decoder's attention: T new tokens for each of B
// sequences at positions pos0 .. pos0 + T - 1 in one pass, instead of T decode steps.
//
// Reference: GPTModel::generate fills the KV cache by calling forward_step once per context
// token (include/neuralnet.cpp/compute_layer_gpt.hpp:774-794); each call rotates the new key
// at its position, appends key and value to the caches and attends over positions [0, pos]
// (AttentionBase::forward_step, compute_layer_attention.hpp:1003-1091). The same results for
// all T tokens at once:
//   * k_kv_fill writes the T rotated keys and values of every sequence into cache rows
//     pos0 .. pos0 + T - 1 (RoPE as the decode append: two rounded products and a rounded sum);
//   * k_attn_prefill gives token t the softmax attention over cache rows [0, pos0 + t] (causal),
//     query head h reading KV head h / (H / Hkv).
//
// Layouts (device, f32): q (H*dk, M), k / v (Hkv*dk, M) and out (H*dk, M) feature-major with
// token column m = b*T + t (the BitLinear outputs of the B*T tokens); caches (B, max_len,
// Hkv*dk) as the decode step's; cos / sin (max_len, dk/2).
//
// k_attn_prefill: the fp32 MFMA's rate (157 TFLOP/s) bounded this attention (101 of it at 4 x 2048
// tokens), and the f16 and bf16 MFMAs run 16 times as fast. So its products run on those with every
// f32 operand as a sum of parts, whose products are exact in f32:
//   * S = K . Q^T: two f16 halves, x 2^e = hi + lo to 2^-23 of x, where e brings the largest value of a
//     query or of a tile of K to 2^14..2^15 (f16 caches: K as it is). What is below 2^-40 of that is
//     lost, less than 2^-21 of a score in all where scores cannot reach 2^18. low x low, at most
//     2^-22 of a term, is left out: three MFMAs per product with f32 caches, two with f16 caches.
//   * O = P . V: three bf16 parts, x = b0 + b1 + b2 exactly and without a scale, two for f16 caches' V.
//     The probability of a key and the size of its value have nothing to do with each other, so
//     neither may cost the other bits: no exponent shared by a tile or a sequence holds both (f16
//     halves of V under one scale lost a channel 1e-7 of the others to 1e-4, 1e-10 altogether).
//     Products b_i b_j with i + j > 2, at most 2^-24 of a term, are left out: six and five MFMAs.
// Sums, softmax and output are f32. Against float64, 1024 tokens of 20 heads over 5 KV heads of 128,
// f32 / f16 caches: 2.3e-7 / 2.0e-7 off in norm (f32 products: 3.9e-7 both).
// What the parts cannot hold (infinities, NaN, a query's or K tile's largest value outside 2^+-48,
// outputs below 2^-100, largest values whose scores could reach 2^18) sends the work-group to the f32
// products (attend_f32).
//
// Work-group = 8 waves = (the R = H / Hkv heads of KV head g) x (8 / R blocks of 32 queries) of
// sequence b; all waves share each 32-key tile of K and V, staged in LDS as planes of parts (double
// buffered, one barrier per tile): the next tile is converted from registers while the one after
// it is loaded. A wave computes S^T = K . Q^T (32 keys x 32 queries) and O^T += V^T . P^T, where
// lane l holds query l % 32 throughout: its 16 elements v of S^T are keys 8(v/4) + 4(l/32) + v%4,
// and V^T is staged with its keys in that order, so P^T is an operand as it stands. Row 32d + r of
// V^T is dimension (DK/32) r + d, which lets a staging lane load contiguous dimensions and its
// stores fall on all banks. K rows and V^T rows are padded to odd multiples of 16 bytes.
// Softmax in log2 units with the hardware exp2; a query's reference maximum moves only when it has
// grown by 2^8 (probabilities are at most 2^8), so the sums are rarely rescaled.
// Work-groups are issued heaviest first (the last query blocks attend over the most keys).
// Measured (calls back to back in a graph, us, f32 products / here): f32 caches 4 x 2048 tokens
// 809 / 398, 3 x 1111 at 517 411 / 202, 16 x 2048 3088 / 1498, 1 x 64 22.5 / 17.7; f16 caches 817 / 293,
// 421 / 146, 3153 / 1121, 22.7 / 15.9. Two f16 halves for P and V too (at the cost above) took 295 and
// 198 us at 4 x 2048.
// Caches of f16 elements (compute = F16): the fill rounds the rotated keys and the values to the
// nearest f16 (ties to even), as the decode append does.
#include "common.hpp"

#include <cmath>

namespace nnhip
{
namespace
{

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kPQ = 32;   // queries per wave of the attention, tokens per block of the cache fill
constexpr int kPK = 32;   // keys per tile

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pf_rsrc(const void* base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ float4 ld_f4(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Four cache elements at byte offset off as floats (f32, or f16 widened exactly)
template <typename CT>
__device__ __forceinline__ float4 ld_c4(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    if constexpr (sizeof(CT) == 4) return ld_f4(r, off);
    else
    {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        const h4 h = __builtin_bit_cast(h4, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
        return make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]);
    }
}

// (x0, x1) = (x[j], x[j + dk/2]) -> x*cos + rotate_half(x)*sin: two rounded products and a
// rounded sum per output, as the decode append does.
__device__ __forceinline__ void pf_rope(float x0, float x1, float cs, float sn, float& y0, float& y1)
{
    y0 = __fadd_rn(__fmul_rn(x0, cs), __fmul_rn(-x1, sn));
    y1 = __fadd_rn(__fmul_rn(x1, cs), __fmul_rn(x0, sn));
}

// ------------------------------------------------------------------ cache fill

// Block = (32 tokens, KV head g): the head's dk feature rows of k and v for the 32 tokens are
// read along tokens (coalesced), transposed through LDS and written as cache rows (coalesced
// along features), the keys rotated at their positions. Bound by HBM: each element read and written
// once; every load of a thread (k, v, cos, sin) is in flight at once, since a block lives for one
// round trip, and token positions are stepped, not divided out per element. 5 heads of 128, back to
// back, before / after (us): 8 x 1024 tokens f32 21.5 / 14.4 (5.9 TB/s), 16 x 2048 f32 104 / 73, f16
// 59.7 / 40.0, 3 x 1111 13.1 / 10.2, 1 x 64 6.4 / 3.5.
template <int DK, typename CT>
__global__ __launch_bounds__(256, 4) void k_kv_fill(const float* __restrict__ k, const float* __restrict__ v, int B, int T,
                                                    int Hkv, int pos0, const float* __restrict__ cosT,
                                                    const float* __restrict__ sinT, CT* __restrict__ kc,
                                                    CT* __restrict__ vc, int max_len)
{
    constexpr int HALF = DK / 2;
    constexpr int NR = 256 / kPQ, U = DK / NR;      // feature rows per round of loads, rounds
    constexpr int NT = 256 / HALF, N = kPQ / NT;    // tokens per round of stores, rounds
    __shared__ float sk[DK][kPQ + 1];
    __shared__ float sv[DK][kPQ + 1];
    const int M = B * T;
    const int g = blockIdx.y;
    const int m0 = blockIdx.x * kPQ;
    const int tid = threadIdx.x;
    const int row = Hkv * DK;
    // loads past the last token repeat it (never stored)
    const int c = tid % kPQ, i0 = tid / kPQ;
    const size_t src = (size_t)(g * DK + i0) * (size_t)M + (size_t)min(m0 + c, M - 1);
    float xk[U], xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xk[u] = k[src + (size_t)(NR * u) * (size_t)M];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = v[src + (size_t)(NR * u) * (size_t)M];
    // the tokens this thread stores features j and j + dk / 2 of
    const int j = tid % HALF, c0 = tid / HALF;
    int t = (m0 + c0) % T, b = (m0 + c0) / T, p[N];
    size_t dst[N];
    float cs[N], sn[N];
#pragma unroll
    for (int n = 0; n < N; ++n)
    {
        p[n] = pos0 + t;
        dst[n] = ((size_t)b * (size_t)max_len + (size_t)p[n]) * (size_t)row + (size_t)(g * DK + j);
        t += NT;
        while (t >= T)
        {
            t -= T;
            ++b;
        }
    }
    if (cosT)
    {
#pragma unroll
        for (int n = 0; n < N; ++n)
        {
            cs[n] = cosT[(size_t)p[n] * HALF + j];
            sn[n] = sinT[(size_t)p[n] * HALF + j];
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
    {
        sk[i0 + NR * u][c] = xk[u];
        sv[i0 + NR * u][c] = xv[u];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n)
    {
        const int cn = c0 + NT * n;
        if (m0 + cn >= M) return;
        const float x0 = sk[j][cn], x1 = sk[j + HALF][cn];
        float y0 = x0, y1 = x1;
        if (cosT) pf_rope(x0, x1, cs[n], sn[n], y0, y1);
        kc[dst[n]] = (CT)y0;
        kc[dst[n] + HALF] = (CT)y1;
        vc[dst[n]] = (CT)sv[j][cn];
        vc[dst[n] + HALF] = (CT)sv[j + HALF][cn];
    }
}

// ------------------------------------------------------------------ causal attention

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

constexpr int kPWaves = 8;             // waves of a work-group: R heads x (8 / R) blocks of 32 queries
constexpr int kPThreads = 64 * kPWaves;
constexpr int kPExpMax = 48;           // scalings beyond 2^+-48 take the f32 products
constexpr float kPLazy = 8.0f;         // log2 growth of a query's maximum before its sums are rescaled
// Largest dk max|q| max|k| |scale| log2(e) of a query and a tile: a score's parts below the halves' range
// (2^-40 of the largest value) add up to less than 2^-21, and no score rounds a reference maximum by 2^-5.
constexpr float kPReach = 0x1p18f;
constexpr float kPTiny = 0x1p-100f;    // outputs below this (but for 0) may have lost bits of a bf16 part

struct PrefillArgs
{
    const float* q;
    const void* kc;  // caches of CT elements
    const void* vc;
    const float* cosT;
    const float* sinT;
    float* out;
    int B, T, H, Hkv, R, pos0, max_len, nqb;
    float scale;
    float scale2;  // |scale| * log2(e)
    int f32;       // 1: the f32 products throughout (a scale outside [2^-20, 2^20])
};

template <int DK, typename CT>
struct PrefillTile
{
    static constexpr int kKPlanes = sizeof(CT) == 4 ? 2 : 1;  // K: high and low f16 halves of f32 values
    static constexpr int kVPlanes = sizeof(CT) == 4 ? 3 : 2;  // V: bf16 parts of f32 / f16 values
    // rows are padded by 16 bytes: 16 lanes' reads of consecutive rows fall on all banks, and every
    // chunk is at a constant offset from a lane's first
    static constexpr int kKPitch = DK * 2 + 16, kVPitch = kPK * 2 + 16;
    static constexpr int kKPlane = kPK * kKPitch, kVPlane = DK * kVPitch;
    static constexpr int kV = kKPlanes * kKPlane;            // K planes, then V planes
    static constexpr int kBuf = kV + kVPlanes * kVPlane;
    static constexpr int KROW = DK + 4;                      // f32 products: padded row (floats)
    static constexpr int kF32 = 2 * kPK * KROW * 4;
    static constexpr int kMain = 2 * kBuf > kF32 ? 2 * kBuf : kF32;  // double-buffered
    static constexpr int kBytes = kMain + 64;                // maxima of K in two tiles, the fallback flag
};

// The two halves of two f32 values scaled into f16's range: x = hi + lo up to 2^-23 |x| or 2^-25
__device__ __forceinline__ void split2(float x0, float x1, v2h& hi, v2h& lo)
{
    hi = __builtin_convertvector(v2f{x0, x1}, v2h);
    // x - hi, exact, from the packed half in place (the compiler widens it with an instruction first)
    const uint32_t u = __builtin_bit_cast(uint32_t, hi);
    float l0, l1;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l0) : "v"(u), "v"(x0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(l1) : "v"(u), "v"(x1));
    lo = __builtin_convertvector(v2f{l0, l1}, v2h);
}

// The first N bf16 parts of two values: x = sum of parts, exactly, for f32 values (N = 3) and widened f16
// values (N = 2) from 2^-110 on (each rounding leaves 8 bits less); infinities and NaN give NaN.
template <int N>
__device__ __forceinline__ void split_bf16(float x0, float x1, v2b (&part)[N])
{
#pragma unroll
    for (int n = 0; n < N; ++n)
    {
        part[n] = __builtin_convertvector(v2f{x0, x1}, v2b);
        if (n + 1 == N) break;
        const uint32_t u = __builtin_bit_cast(uint32_t, part[n]);
        x0 -= __builtin_bit_cast(float, u << 16);
        x1 -= __builtin_bit_cast(float, u & 0xFFFF0000u);
    }
}

// 2^e for |e| <= 126
__device__ __forceinline__ float pow2(int e) { return __builtin_bit_cast(float, (uint32_t)(127 + e) << 23); }

// The exponent that brings values whose largest bit pattern is mx (sign cleared) into [2^14, 2^15):
// kPExpMax for all-zero values. Outside +-kPExpMax (infinities and NaN among it) the f32 products run.
__device__ __forceinline__ int f16_exp(uint32_t mx) { return mx == 0 ? kPExpMax : 14 + 127 - (int)(mx >> 23); }

// The wave's largest value
__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    for (int off = 32; off >= 1; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off, kWave));
    return v;
}

// Where a wave works: query head, first query, the lane's query
struct PrefillWave
{
    int b, g, head, t0, qt, qpos;
    bool live;  // the wave has queries
};

// The lane's rotated query value pairs, f(c, e, value, value of the dimension DK/2 further) for its
// dimensions 2Gc + Gh + e below DK/2. The cos / sin rows of 32 queries are 32 lines apart, so they
// are read four at a time. Lanes past the last token repeat it (they are never stored).
template <int DK, int G, typename F>
__device__ __forceinline__ void load_query(const PrefillArgs& a, const PrefillWave& w, int h, F&& f)
{
    constexpr int HALF = DK / 2, NG = HALF / (2 * G);
    const int M = a.B * a.T;
    const __amdgpu_buffer_rsrc_t rq = pf_rsrc(a.q, (uint32_t)((size_t)a.H * DK * (size_t)M * 4u));
    const uint32_t rope_bytes = a.cosT ? (uint32_t)((size_t)a.max_len * HALF * 4u) : 0u;
    const __amdgpu_buffer_rsrc_t rc = pf_rsrc(a.cosT ? a.cosT : a.q, rope_bytes);
    const __amdgpu_buffer_rsrc_t rs = pf_rsrc(a.cosT ? a.sinT : a.q, rope_bytes);
    const int qt = min(w.qt, a.T - 1);
    const uint32_t q_at = (uint32_t)(((size_t)(w.head * DK + G * h) * (size_t)M + (size_t)(w.b * a.T + qt)) * 4u);
    const uint32_t r_at = (uint32_t)(((size_t)(a.pos0 + qt) * HALF + (size_t)(G * h)) * 4u);
#pragma unroll
    for (int c = 0; c < NG; ++c)
    {
        float x[2][G];
        float4 cs[G / 4], sn[G / 4];
#pragma unroll
        for (int e = 0; e < G; ++e)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                x[q][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rq, q_at, (2 * G * c + e + HALF * q) * M * 4, 0));
#pragma unroll
        for (int e = 0; e < G / 4; ++e)
        {
            cs[e] = ld_f4(rc, r_at + (uint32_t)(2 * G * c + 4 * e) * 4u);
            sn[e] = ld_f4(rs, r_at + (uint32_t)(2 * G * c + 4 * e) * 4u);
        }
#pragma unroll
        for (int e = 0; e < G; ++e)
        {
            const float cv = e % 4 == 0 ? cs[e / 4].x : e % 4 == 1 ? cs[e / 4].y : e % 4 == 2 ? cs[e / 4].z : cs[e / 4].w;
            const float sv = e % 4 == 0 ? sn[e / 4].x : e % 4 == 1 ? sn[e / 4].y : e % 4 == 2 ? sn[e / 4].z : sn[e / 4].w;
            float y0 = x[0][e], y1 = x[1][e];
            if (a.cosT) pf_rope(x[0][e], x[1][e], cv, sv, y0, y1);
            f(c, e, y0, y1);
        }
    }
}

// out[head*DK + i][m] = y(d, v) for the lane's query: element v of block d belongs to row
// r = 8(v/4) + 4h + v%4 of the block; dim(d, r) is its dimension
template <int DK, typename D, typename Y>
__device__ __forceinline__ void store_out(const PrefillArgs& a, const PrefillWave& w, int h, D&& dim, Y&& y)
{
    if (w.qt >= a.T) return;
    const int M = a.B * a.T, m = w.b * a.T + w.qt;
#pragma unroll
    for (int d = 0; d < DK / 32; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v)
            a.out[(size_t)(w.head * DK + dim(d, 8 * (v >> 2) + 4 * h + (v & 3))) * (size_t)M + (size_t)m] = y(d, v);
}

// The work-group's attention on the fp32 MFMA (v_mfma_f32_32x32x2_f32), for inputs that the f16
// and bf16 parts cannot hold (see the top of the file). Per 32-key
// tile S^T (not S) is in the accumulators, so lane l holds query l % 32 and keys
// 8(v/4) + 4(l/32) + v%4 of its 16 elements v: the B operand of the P . V products when the keys of
// product s are taken in that order. The sum over the head dimension takes product s = 4c + e over
// dimensions 8c + e and 8c + 4 + e (the two lane halves).
template <int DK, typename CT>
__device__ void attend_f32(const PrefillArgs& a, const PrefillWave& w, int last_key, __amdgpu_buffer_rsrc_t rk,
                           __amdgpu_buffer_rsrc_t rv, float* ks)
{
    constexpr int NC = DK / 8, ND = DK / 32, KROW = PrefillTile<DK, CT>::KROW;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
    const int row = a.Hkv * DK;
    float* vs = ks + kPK * KROW;
    float qv[DK / 2];  // qv[4c + e] = rotated query value of dimension 8c + 4h + e
    load_query<DK, 4>(a, w, h, [&](int c, int e, float y0, float y1) {
        qv[4 * c + e] = y0;
        qv[4 * (c + NC / 2) + e] = y1;
    });
    v16f o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = v16f{};
    float m_run = -__builtin_inff(), l_run = 0.0f;
    for (int kb = 0; kb <= last_key / kPK; ++kb)
    {
        __syncthreads();  // every wave is done with the previous tile
        for (int u = tid; u < kPK * DK / 4; u += kPThreads)
        {
            const int key = u / (DK / 4), c4 = u % (DK / 4);
            const uint32_t off = (uint32_t)(((size_t)(kb * kPK + key) * (size_t)row + (size_t)w.g * DK + 4 * c4) * sizeof(CT));
            *reinterpret_cast<float4*>(ks + key * KROW + 4 * c4) = ld_c4<CT>(rk, off);
            *reinterpret_cast<float4*>(vs + key * KROW + 4 * c4) = ld_c4<CT>(rv, off);
        }
        __syncthreads();
        if (!w.live || kb * kPK > a.pos0 + w.t0 + kPQ - 1) continue;
        v16f s = v16f{};
#pragma unroll
        for (int c = 0; c < NC; ++c)
        {
            const float4 kk = *reinterpret_cast<const float4*>(ks + l32 * KROW + 8 * c + 4 * h);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.x, qv[4 * c + 0], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.y, qv[4 * c + 1], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.z, qv[4 * c + 2], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.w, qv[4 * c + 3], s, 0, 0, 0);
        }
        float sc[16];
        float mx = -__builtin_inff();
#pragma unroll
        for (int v = 0; v < 16; ++v)
        {
            const int key = kb * kPK + 8 * (v >> 2) + 4 * h + (v & 3);
            const float x = s[v] * a.scale;
            sc[v] = key <= w.qpos ? x : -__builtin_inff();
            mx = fmaxf(mx, sc[v]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const bool any = m_new != -__builtin_inff();
        const float corr = any ? expf(m_run - m_new) : 1.0f;
        float ls = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v)
        {
            sc[v] = any ? expf(sc[v] - m_new) : 0.0f;
            ls += sc[v];
        }
        ls += __shfl_xor(ls, 32);
        l_run = l_run * corr + ls;
        m_run = m_new;
        // corr is exactly 1 where the running maximum did not move
        if (__builtin_amdgcn_ballot_w64(corr != 1.0f) != 0)
        {
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[d][v] *= corr;
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int sp = 0; sp < 16; ++sp)
            {
                const int key = 8 * (sp >> 2) + 4 * h + (sp & 3);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vs[key * KROW + 32 * d + l32], sc[sp], o[d], 0, 0, 0);
            }
    }
    if (w.live)
        store_out<DK>(a, w, h, [](int d, int r) { return 32 * d + r; }, [&](int d, int v) { return o[d][v] / l_run; });
}

template <int DK, typename CT>
__global__ __launch_bounds__(kPThreads) void k_attn_prefill(PrefillArgs a)
{
    using Tile = PrefillTile<DK, CT>;
    constexpr bool F32C = sizeof(CT) == 4;
    constexpr int NC = DK / 16;  // MFMA steps over the head dimension
    constexpr int ND = DK / 32;  // 32-row blocks of O^T, and dimensions per lane when staging V
    constexpr int CH = DK / 8;   // 16-byte chunks of a K row
    constexpr int KU = CH * kPK / 256;  // chunks a thread stages
    extern __shared__ __align__(16) uint8_t smem[];
    uint32_t* smax = reinterpret_cast<uint32_t*>(smem + Tile::kMain);  // [2][4]: per tile parity and K wave; f16 caches: [8] per wave
    // set to send the work-group to the f32 products: written in iteration kb (or before the loop) into
    // [(kb + 1) & 1] and read after the barrier of iteration kb + 1, so all waves read the same value
    int* sflag = reinterpret_cast<int*>(smem + Tile::kMain + 32);

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // heaviest items first: the last queries attend over the most keys
    const int per_qb = a.B * a.Hkv;
    const int qb = a.nqb - 1 - (int)blockIdx.x / per_qb;
    const int bg = (int)blockIdx.x % per_qb;
    PrefillWave w;
    w.b = bg / a.Hkv;
    w.g = bg % a.Hkv;
    w.head = w.g * a.R + wave % a.R;
    const int qn = kPQ * (kPWaves / a.R);  // queries of the work-group
    w.t0 = qb * qn + wave / a.R * kPQ;
    w.qt = w.t0 + l32;
    w.qpos = a.pos0 + w.qt;
    w.live = w.t0 < a.T;
    const int row = a.Hkv * DK;
    const int valid = a.pos0 + a.T;  // cache rows [0, valid) hold keys / values
    const int last_key = a.pos0 + min(qb * qn + qn, a.T) - 1;
    const int nkb = last_key / kPK + 1;
    const size_t seq_off = (size_t)w.b * (size_t)a.max_len * (size_t)row;
    // rows at or past `valid` read as zeros: their scores are masked and their zero values keep
    // 0 * v finite
    const uint32_t seq_bytes = (uint32_t)((size_t)min(valid, a.max_len) * (size_t)row * sizeof(CT));
    const __amdgpu_buffer_rsrc_t rk = pf_rsrc(static_cast<const CT*>(a.kc) + seq_off, seq_bytes);
    const __amdgpu_buffer_rsrc_t rv = pf_rsrc(static_cast<const CT*>(a.vc) + seq_off, seq_bytes);

    if (tid < 2) sflag[tid] = tid == 0 ? a.f32 : 0;
    __syncthreads();

    // ---- staging, 16 elements per thread: waves 0-3 take V (thread = 4 keys x ND dimensions), waves
    // 4-7 take K (thread = KU chunks of 8 dimensions of a key). raw holds them as loaded.
    constexpr int RW = F32C ? 16 : 8;  // words
    uint32_t raw[RW];
    const bool is_v = wave < 4;
    const int u = tid & 255;
    const int vq = u >> 5, vg = u & 31;  // V: key quad, dimension group
    // the thread's offsets within a tile; the tile's rows are reached through the buffer's base
    constexpr int NL = F32C ? 4 : (4 > KU ? 4 : KU);
    uint32_t at[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i)
    {
        const int ct = u + 256 * i;
        at[i] = is_v ? (uint32_t)(((4 * vq + i) * row + w.g * DK + ND * vg) * (int)sizeof(CT))
                     : (uint32_t)((ct / CH * row + w.g * DK + 8 * (ct % CH)) * (int)sizeof(CT));
    }
    const uint32_t tile_bytes = (uint32_t)(kPK * row) * (uint32_t)sizeof(CT);
    const CT* const kvb = (is_v ? static_cast<const CT*>(a.vc) : static_cast<const CT*>(a.kc)) + seq_off;
    auto load_raw = [&](int kb) {
        const uint64_t before = (uint64_t)kb * tile_bytes;
        const __amdgpu_buffer_rsrc_t rt = pf_rsrc(reinterpret_cast<const uint8_t*>(kvb) + before,
                                                  before < seq_bytes ? seq_bytes - (uint32_t)before : 0u);
        if (is_v)
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                constexpr int W = ND * (int)sizeof(CT) / 4;  // words per key
                if constexpr (W == 4)
                {
                    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rt, at[i], 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[4 * i + e] = x[e];
                }
                else if constexpr (W == 2)
                {
                    const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(rt, at[i], 0, 0);
                    raw[2 * i] = x[0];
                    raw[2 * i + 1] = x[1];
                }
                else raw[i] = __builtin_amdgcn_raw_buffer_load_b32(rt, at[i], 0, 0);
            }
        }
        else
        {
#pragma unroll
            for (int j = 0; j < KU; ++j)
#pragma unroll
                for (int q = 0; q < (F32C ? 2 : 1); ++q)
                {
                    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rt, at[j] + 16 * q, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[(F32C ? 8 : 4) * j + 4 * q + e] = x[e];
                }
        }
    };
    // words of raw in use
    constexpr int VW = 4 * ND * (int)sizeof(CT) / 4, KW = KU * 8 * (int)sizeof(CT) / 4;
    static_assert(VW == KW && VW <= RW, "V and K threads stage the same amount");
    // f32 caches: the wave's largest magnitude in K, for the tile's scaling
    auto post_max = [&](int kb) {
        if (!F32C || is_v) return;
        uint32_t mx = 0;
#pragma unroll
        for (int e = 0; e < KW; ++e) mx = max(mx, raw[e] & 0x7FFFFFFFu);
        mx = wave_max(mx);
        if (lane == 0) smax[(kb & 1) * 4 + wave - 4] = mx;
    };
    int ek = 0;        // exponent of the staged tile's K
    float eqf = 0.0f;  // the lane's query: 2^-eq |scale| log2(e)
    float klim = 0.0f; // f16 caches: the largest key element within kPReach of every query of the work-group
    // K's exponent, then raw as f16 halves (K) and bf16 parts (V) into buffer kb & 1
    auto convert = [&](int kb, int* flag) {
        uint8_t* buf = smem + (kb & 1) * Tile::kBuf;
        if constexpr (F32C)
        {
            const uint32_t* sm = smax + (kb & 1) * 4;
            ek = __builtin_amdgcn_readfirstlane(f16_exp(max(max(sm[0], sm[1]), max(sm[2], sm[3]))));
            if (abs(ek) > kPExpMax)
            {
                if (tid == 0) *flag = 1;
                ek = 0;
            }
            // |q| 2^eq and |k| 2^ek are at most 2^15
            else if (__builtin_amdgcn_ballot_w64(eqf * pow2(-ek) > kPReach / (DK * 0x1p30f)) != 0 && lane == 0) *flag = 1;
        }
        else if (!is_v)
        {
            u16x2 m = {0, 0};
#pragma unroll
            for (int e = 0; e < KW; ++e) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, raw[e] & 0x7FFF7FFFu));
            const uint16_t top = max(m[0], m[1]);
            if (__builtin_amdgcn_ballot_w64(!((float)__builtin_bit_cast(_Float16, top) <= klim)) != 0 && lane == 0) *flag = 1;
        }
        const float sk = F32C ? pow2(ek) : 1.0f;
        if (is_v)
        {
            // row 32e + vg = dimension ND vg + e; its 4 chunks are (16-key half s, lane half) and hold
            // keys 16s + 8a + 4h + i in the order (a, i): the accumulators' order of S^T
            const int s = vq >> 2, ah = (vq >> 1) & 1, hh = vq & 1;
#pragma unroll
            for (int e = 0; e < ND; ++e)
            {
                const int r = 32 * e + vg;
                uint8_t* dst = buf + Tile::kV + r * Tile::kVPitch + 32 * s + 16 * hh + 8 * ah;
                float x[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    if constexpr (F32C) x[i] = __builtin_bit_cast(float, raw[ND * i + e]);
                    else x[i] = (float)__builtin_bit_cast(v2h, raw[ND / 2 * i + e / 2])[e & 1];
                }
                v2b p0[Tile::kVPlanes], p1[Tile::kVPlanes];
                split_bf16(x[0], x[1], p0);
                split_bf16(x[2], x[3], p1);
#pragma unroll
                for (int q = 0; q < Tile::kVPlanes; ++q)
                    *reinterpret_cast<u32x2*>(dst + q * Tile::kVPlane) =
                        u32x2{__builtin_bit_cast(uint32_t, p0[q]), __builtin_bit_cast(uint32_t, p1[q])};
            }
        }
        else
        {
#pragma unroll
            for (int j = 0; j < KU; ++j)
            {
                const int ct = u + 256 * j, key = ct / CH, c = ct % CH;
                uint8_t* dst = buf + key * Tile::kKPitch + 16 * c;
                if constexpr (F32C)
                {
                    v8h hi, lo;
#pragma unroll
                    for (int e = 0; e < 8; e += 2)
                    {
                        v2h x, y;
                        split2(__builtin_bit_cast(float, raw[8 * j + e]) * sk, __builtin_bit_cast(float, raw[8 * j + e + 1]) * sk, x, y);
                        hi[e] = x[0], hi[e + 1] = x[1];
                        lo[e] = y[0], lo[e + 1] = y[1];
                    }
                    *reinterpret_cast<v8h*>(dst) = hi;
                    *reinterpret_cast<v8h*>(dst + Tile::kKPlane) = lo;
                }
                else
                    *reinterpret_cast<u32x4*>(dst) = u32x4{raw[4 * j], raw[4 * j + 1], raw[4 * j + 2], raw[4 * j + 3]};
            }
        }
    };

    // Fragments from LDS, up to four 16-byte reads at a time, a group ahead of the products that use them:
    // group g of K holds steps GK g .., group g of V^T (block, half) pairs GV g .., each with its planes.
    constexpr int PK = Tile::kKPlanes, PV = Tile::kVPlanes, GK = 4 / PK, GV = 4 / PV;
    constexpr int GKN = NC / GK, GVN = 2 * ND / GV;  // groups
    static_assert(NC % GK == 0 && (2 * ND) % GV == 0, "whole groups");
    const uint32_t k_at = (uint32_t)(l32 * Tile::kKPitch + 16 * h), v_at = (uint32_t)(Tile::kV + l32 * Tile::kVPitch + 16 * h);
    auto read_k = [&](u32x4(&f)[4], uint32_t par, int g) {
        const uint8_t* p = smem + (par + k_at);
#pragma unroll
        for (int e = 0; e < GK; ++e)
#pragma unroll
            for (int q = 0; q < PK; ++q)
                f[PK * e + q] = *reinterpret_cast<const u32x4*>(p + 32 * (GK * g + e) + q * Tile::kKPlane);
    };
    auto read_v = [&](u32x4(&f)[4], uint32_t par, int g) {
        const uint8_t* p = smem + (par + v_at);
#pragma unroll
        for (int e = 0; e < GV; ++e)
        {
            const int d = (GV * g + e) >> 1, t = (GV * g + e) & 1;
#pragma unroll
            for (int q = 0; q < PV; ++q)
                f[PV * e + q] = *reinterpret_cast<const u32x4*>(p + 32 * d * Tile::kVPitch + 32 * t + q * Tile::kVPlane);
        }
    };

    load_raw(0);

    // ---- the lane's rotated query in halves: step c holds dimensions 16c + 8h + 0..7, scaled by 2^eq
    v8h qh[NC], ql[NC];
    if (w.live)
    {
        float qv[DK / 2];
        uint32_t mx = 0;
        const float sign = a.scale < 0.0f ? -1.0f : 1.0f;
        load_query<DK, 8>(a, w, h, [&](int c, int e, float y0, float y1) {
            qv[8 * c + e] = y0;
            qv[8 * (c + NC / 2) + e] = y1;
            mx = max(mx, max(__builtin_bit_cast(uint32_t, y0) & 0x7FFFFFFFu, __builtin_bit_cast(uint32_t, y1) & 0x7FFFFFFFu));
        });
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, 32, kWave));
        int eq = f16_exp(mx);
        const bool far = abs(eq) > kPExpMax;
        if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) sflag[0] = 1;
        if (far) eq = 0;
        const float sq = sign * pow2(eq);
        eqf = a.scale2 * pow2(-eq);
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 8; e += 2)
            {
                v2h x, y;
                split2(qv[8 * c + e] * sq, qv[8 * c + e + 1] * sq, x, y);
                qh[c][e] = x[0], qh[c][e + 1] = x[1];
                ql[c][e] = y[0], ql[c][e + 1] = y[1];
            }
    }
    v16f o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = v16f{};
    float m_ref = -__builtin_inff(), l_run = 0.0f;  // log2 units; l_run: this lane half's keys

    post_max(0);
    if constexpr (!F32C)
    {
        const uint32_t mx = wave_max(__builtin_bit_cast(uint32_t, eqf));  // not negative
        if (lane == 0) smax[wave] = mx;
    }
    __syncthreads();
    if constexpr (!F32C)
    {
        uint32_t mx = 0;
#pragma unroll
        for (int i = 0; i < kPWaves; ++i) mx = max(mx, smax[i]);
        klim = kPReach / (DK * 0x1p15f) / __builtin_bit_cast(float, mx);  // |q| 2^eq is at most 2^15
    }
    convert(0, sflag);
    if (nkb > 1)
    {
        load_raw(1);
        post_max(1);
    }
    bool fallback = false;
    for (int kb = 0; kb < nkb; ++kb)
    {
        __syncthreads();  // tile kb is in LDS, the maxima of tile kb + 1 too; buffer (kb + 1) & 1 is free
        if (sflag[kb & 1])
        {
            fallback = true;
            break;
        }
        const int ek_now = ek;
        // this tile's first K fragments, in flight during the conversion of the next tile
        const uint32_t par = (uint32_t)(kb & 1) * Tile::kBuf;
        u32x4 fr[2][4];
        read_k(fr[0], par, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (kb + 1 < nkb)
        {
            convert(kb + 1, sflag + ((kb + 1) & 1));
            if (kb + 2 < nkb) load_raw(kb + 2);  // in flight during this tile's products
        }
        if (w.live && kb * kPK <= a.pos0 + w.t0 + kPQ - 1)
        {
            // S^T = K . Q^T: the products of the halves but low x low (at most 2^-22 of a term)
            v16f s = v16f{};
#pragma unroll
            for (int g = 0; g < GKN; ++g)
            {
                if (g + 1 < GKN) read_k(fr[(g + 1) & 1], par, g + 1);
                else read_v(fr[(g + 1) & 1], par, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < GK; ++e)
                {
                    const int c = GK * g + e;
                    const v8h kh = __builtin_bit_cast(v8h, fr[g & 1][PK * e]);
                    if constexpr (F32C)
                        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, fr[g & 1][PK * e + 1]), qh[c], s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[c], s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[c], s, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // scores in log2 units are s * f; the causal mask only where the tile reaches past the
            // wave's first query
            const float f = F32C ? eqf * pow2(-ek_now) : eqf;
            if (kb * kPK + kPK - 1 > a.pos0 + w.t0)
            {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (kb * kPK + 8 * (v >> 2) + 4 * h + (v & 3) > w.qpos) s[v] = -__builtin_inff();
            }
            float mx = s[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
            mx = fmaxf(mx, __shfl_xor(mx, 32)) * f;
            // the reference of a query moves only when its maximum has grown by 2^8 (or is new)
            const bool grown = mx > m_ref + kPLazy;
            if (__builtin_amdgcn_ballot_w64(grown) != 0)
            {
                const float m_new = grown ? mx : m_ref;
                const float corr = __builtin_amdgcn_exp2f(m_ref - m_new);  // 0 on the first tile
                l_run *= corr;
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[d][v] *= corr;
                m_ref = m_new;
            }
            v8b p[3][2];
#pragma unroll
            for (int v = 0; v < 16; v += 2)
            {
                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], f, -m_ref));
                const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v + 1], f, -m_ref));
                l_run += p0;
                l_run += p1;
                v2b x[3];
                split_bf16(p0, p1, x);
#pragma unroll
                for (int q = 0; q < 3; ++q) p[q][v >> 3][v & 7] = x[q][0], p[q][v >> 3][(v & 7) + 1] = x[q][1];
            }
            __builtin_amdgcn_sched_barrier(0);
            // O^T += V^T . P^T: the products of parts i and j with i + j <= 2, smallest first; the rest is
            // at most 2^-24 of a term. A tile is summed from zero and added once: that rounds the running
            // sum once in 32 keys. The add of a block runs beside the products of the next.
            v16f sum[2];
#pragma unroll
            for (int g = 0; g < GVN; ++g)
            {
                const u32x4(&f4)[4] = fr[(GKN + g) & 1];
                if (g + 1 < GVN) read_v(fr[(GKN + g + 1) & 1], par, g + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < GV; ++e)
                {
                    const int d = (GV * g + e) >> 1, t = (GV * g + e) & 1;
                    if (t == 0) sum[d & 1] = v16f{};
                    if (t == 1 - (GV & 1) && d > 0) o[d - 1] += sum[(d - 1) & 1];
#pragma unroll
                    for (int n = 2; n >= 0; --n)
#pragma unroll
                        for (int i = PV - 1 < n ? PV - 1 : n; i >= 0; --i)
                            sum[d & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, f4[PV * e + i]), p[n - i][t], sum[d & 1], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            o[ND - 1] += sum[(ND - 1) & 1];
        }
        if (kb + 2 < nkb) post_max(kb + 2);
    }
    // V is not looked through for infinities and NaN: any that matters is in the sums. Nor for values whose smallest part would lie below bf16's range: their output is tiny then.
    l_run += __shfl_xor(l_run, 32);
    bool bad = !(l_run < __builtin_inff());
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v)
        {
            const float y = fabsf(o[d][v]);
            bad |= !(y < __builtin_inff()) || (y < l_run * kPTiny && y != 0.0f);
        }
    if (__syncthreads_or(!fallback && w.live && bad) || fallback)
    {
        attend_f32<DK, CT>(a, w, last_key, rk, rv, reinterpret_cast<float*>(smem));
        return;
    }
    if (!w.live) return;
    // o / l, correctly rounded but for the last step's double rounding: the residual is exact
    const float r = 1.0f / l_run;
    store_out<DK>(a, w, h, [](int d, int i) { return ND * i + d; }, [&](int d, int v) {
        const float q = o[d][v] * r;
        return __builtin_fmaf(__builtin_fmaf(-q, l_run, o[d][v]), r, q);
    });
}

template <int DK, typename CT>
hipError_t launch_prefill_dk(hipStream_t st, const PrefillArgs& a)
{
    constexpr int lds = PrefillTile<DK, CT>::kBytes;
    static bool attr_set = false;
    if (!attr_set)
    {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_prefill<DK, CT>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const unsigned blocks = (unsigned)(a.nqb * a.B * a.Hkv);
    hipLaunchKernelGGL((k_attn_prefill<DK, CT>), dim3(blocks), dim3(kPThreads), lds, st, a);
    return hipGetLastError();
}

}  // namespace

bool prefill_dk_supported(size_t dk) { return dk == 64 || dk == 128; }

template <typename CT>
hipError_t launch_kv_fill_ct(hipStream_t st, const float* k, const float* v, size_t B, size_t T, size_t Hkv, size_t dk,
                             size_t pos0, const float* cosT, const float* sinT, CT* kc, CT* vc, size_t max_len)
{
    const dim3 grid((unsigned)ceil_div(B * T, kPQ), (unsigned)Hkv);
    if (dk == 64)
        hipLaunchKernelGGL((k_kv_fill<64, CT>), grid, dim3(256), 0, st, k, v, (int)B, (int)T, (int)Hkv, (int)pos0, cosT,
                           sinT, kc, vc, (int)max_len);
    else if (dk == 128)
        hipLaunchKernelGGL((k_kv_fill<128, CT>), grid, dim3(256), 0, st, k, v, (int)B, (int)T, (int)Hkv, (int)pos0, cosT,
                           sinT, kc, vc, (int)max_len);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_kv_fill(hipStream_t st, const float* k, const float* v, size_t B, size_t T, size_t Hkv, size_t dk,
                          size_t pos0, const float* cosT, const float* sinT, void* kc, void* vc, bool cache_f16,
                          size_t max_len)
{
    if (B * T == 0) return hipSuccess;
    if (cache_f16)
        return launch_kv_fill_ct(st, k, v, B, T, Hkv, dk, pos0, cosT, sinT, static_cast<_Float16*>(kc),
                                 static_cast<_Float16*>(vc), max_len);
    return launch_kv_fill_ct(st, k, v, B, T, Hkv, dk, pos0, cosT, sinT, static_cast<float*>(kc),
                             static_cast<float*>(vc), max_len);
}

hipError_t launch_attn_prefill(hipStream_t st, const float* q, const void* kc, const void* vc, bool cache_f16,
                               size_t B, size_t T, size_t H, size_t Hkv, size_t dk, size_t pos0, const float* cosT,
                               const float* sinT, size_t max_len, float scale, float* out)
{
    if (B * T == 0) return hipSuccess;
    const size_t R = H / Hkv;
    const float mag = std::fabs(scale);
    const bool f32 = !(mag >= 0x1p-20f && mag <= 0x1p20f);
    PrefillArgs a{q, kc, vc, cosT, sinT, out, (int)B, (int)T, (int)H, (int)Hkv, (int)R, (int)pos0,
                  (int)max_len, (int)ceil_div(T, kPQ * (kPWaves / R)), scale, (float)(mag * 1.4426950408889634), f32 ? 1 : 0};
    if (cache_f16)
    {
        if (dk == 64) return launch_prefill_dk<64, _Float16>(st, a);
        if (dk == 128) return launch_prefill_dk<128, _Float16>(st, a);
        return hipErrorInvalidValue;
    }
    if (dk == 64) return launch_prefill_dk<64, float>(st, a);
    if (dk == 128) return launch_prefill_dk<128, float>(st, a);
    return hipErrorInvalidValue;
}

}  // namespace nnhip
