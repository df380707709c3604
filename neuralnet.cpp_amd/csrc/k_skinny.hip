// k_skinny.hip — ternary x int8 products of 17 to a few hundred tokens on gfx950 int8 MFMA, between
// the decode GEMV (k_gemv.hip, M <= 16) and the prefill GEMM (k_gemm.hip), and of fewer tokens on the
// shapes that the decode GEMV is not built for.
//
// There the GEMM's 64 x 64 blocks are few (40 for 2560 rows and up to 64 tokens, of 256 CUs) and each
// walks the whole reduction stage by stage, so its time is a chain of K / 256 memory latencies: 8 us
// at K=2560, 16.8 us at K=6912, whatever M and N are. Here a block takes 16 to 64 rows and 16 or 32
// tokens and splits the reduction over its waves (a wave takes k tiles w, w + waves, ...), so every
// wave has one or two tiles to load and all loads are in flight at once. No two waves of a block
// share an operand, so both come straight from memory in MFMA layout, without LDS; the waves' partial
// sums (integers, exact in any order) meet in LDS once, and the epilogue is one step over the block.
// Activations are the MFMA's A operand and codes its B (gemv_tile.hpp): lane 16g + r holds tokens
// 4g + i of row r, four consecutive floats of a feature-major output, or the four digits of one
// float token (k_digits.hip).
// What bounds it as M and N grow is the lines its loads touch (an activation load takes 64 bytes of
// 16 lines); skinny_plan picks the block shape by that count and draws the line against the GEMM.
// Kernel times (us, GEMM / here): 2560 -> 2560 17 tokens 8.0 / 3.7, 64 8.0 / 4.4, 192 8.2 / 6.2;
// 6912 -> 2560 40 tokens 16.8 / 6.2, 128 16.6 / 10.7; 2560 -> 6912 40 tokens 8.2 / 5.9; 4096 -> 11008
// 32 tokens 11.2 / 7.5. Float products (k_digits.hip and this): 2560 -> 6912 5 tokens 13.6 / 10.3,
// 6912 -> 2560 16 tokens 27.7 / 17.9.
#include "common.hpp"
#include "gemv_tile.hpp"

namespace nnhip
{
namespace
{

constexpr int kSkPlain = 0, kSkGlu = 1, kSkDigits = 2;
constexpr int kSkMaxWaves = 16;
constexpr double kSkGemmRound = 660.0;   // skinny_plan's cost of a 256 x 128 GEMM round per k tile

// G groups of 16 tokens and RT row tiles per block; at least RT * G waves (one output item of four
// tokens per thread)
template <int G, int RT, int MODE>
__global__ __launch_bounds__(64 * kSkMaxWaves) void k_skinny(GemvProblem p, DigitOut dg)
{
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NW = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int KT = p.KT, RTs = (p.N + 15) >> 4;
    const uint32_t Kp = (uint32_t)KT * kTileK;
    const int rt0 = blockIdx.x * RT, m0 = blockIdx.y * 16 * G;
    const __amdgpu_buffer_rsrc_t rw = rsrc(p.rp, (uint32_t)RTs * (uint32_t)KT * 1024u);  // past N: code 0
    const __amdgpu_buffer_rsrc_t rx = rsrc(p.xi, (uint32_t)p.M * Kp);                    // past M: 0
    uint32_t xo[G];
#pragma unroll
    for (int q = 0; q < G; ++q)
    {
        const int m = m0 + 16 * q + r;
        xo[q] = m < p.M ? (uint32_t)m * Kp + 16u * (uint32_t)g : kOOB;
    }

    // ---- this thread's output item: tokens mt .. mt + 3 of row tile it_rt's row ir (and its operands)
    const bool has = tid < RT * G * 64;
    const int ir = tid & 15, ig = (tid >> 4) & 3, iq = (tid >> 6) % G, it_rt = (tid >> 6) / G;
    const int n = (rt0 + it_rt) * 16 + ir, mt = m0 + 16 * iq + 4 * ig;
    const bool out = has && n < p.N && mt < p.M;
    float tau = 1.0f, bias = 0.0f, tau_u = 1.0f, bias_u = 0.0f, sv[4], res[4];
    int rs[4], ex = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const int m = min(mt + i, p.M - 1);
        rs[i] = out ? 2 * p.rowsum[m] : 0;
        sv[i] = out && MODE != kSkDigits ? p.s[m] : 0.0f;
        res[i] = MODE == kSkPlain && out && p.res ? p.res[(size_t)n * p.M + m] : 0.0f;
    }
    if (out && p.tau) tau = p.tau[n];
    if (MODE != kSkDigits && out && p.bias) bias = p.bias[n];
    if (MODE == kSkGlu && out && ir < 8)  // up row of the feature, 8 rows below its gate row
    {
        tau_u = p.tau[n + 8];
        if (p.bias) bias_u = p.bias[n + 8];
    }
    if (MODE == kSkDigits && out) ex = dg.ex[mt >> 2];

    // ---- the wave's k tiles
    v4i acc[RT][G];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < G; ++q) acc[t][q] = v4i{0, 0, 0, 0};
    for (int kt = wave; kt < KT; kt += NW)
    {
        u32x4 w[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t)
            w[t] = __builtin_bit_cast(u32x4, ld16<0>(rw, ((uint32_t)(rt0 + t) * (uint32_t)KT + (uint32_t)kt) * 1024u + 16u * (uint32_t)lane, 0));
        v4i x[G][4];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) x[q][j] = ld16<0>(rx, xo[q] + 64u * j, (uint32_t)kt * kTileK);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < RT; ++t)
            {
                const v4i c = __builtin_bit_cast(v4i, (w[t] >> (2 * j)) & kM3);
#pragma unroll
                for (int q = 0; q < G; ++q) acc[t][q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[q][j], c, acc[t][q], 0, 0, 0);
            }
    }

    // ---- partial sums of the waves
    v4i* part = reinterpret_cast<v4i*>(lds);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < G; ++q) part[((wave * RT + t) * G + q) * 64 + lane] = acc[t][q];
    __syncthreads();
    if (!out || (MODE == kSkGlu && ir >= 8)) return;
    v4i a = v4i{0, 0, 0, 0}, au = v4i{0, 0, 0, 0};
    for (int i = 0; i < NW; ++i)
    {
        a += part[i * RT * G * 64 + tid];
        if (MODE == kSkGlu) au += part[i * RT * G * 64 + tid + 8];
    }

    if constexpr (MODE == kSkDigits)
    {
        if (ex == kDigitSpecial) return;  // its rows are written by the digit kernels
        const long long T = (long long)(a[0] - rs[0]) + ((long long)(a[1] - rs[1]) << 8) +
                            ((long long)(a[2] - rs[2]) << 16) + ((long long)(a[3] - rs[3]) << 24);
        const float y = tau * ldexpf((float)T, ex - 30);
        const size_t at = (size_t)n * (size_t)(p.M >> 2) + (size_t)(mt >> 2);
        if (dg.y16) static_cast<_Float16*>(dg.y)[at] = (_Float16)y;
        else static_cast<float*>(dg.y)[at] = y;
    }
    else
    {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            float v = (tau * sv[i]) * (float)(a[i] - rs[i]);
            if (p.bias) v = v + bias;
            if (MODE == kSkGlu)
            {
                float u = (tau_u * sv[i]) * (float)(au[i] - rs[i]);
                if (p.bias) u = u + bias_u;
                v = glu_one(v, u, p.glu - 1);
            }
            else if (p.res) v = v + res[i];
            y[i] = v;
        }
        const int row = MODE == kSkGlu ? 8 * (rt0 + it_rt) + ir : n;
        if (MODE == kSkGlu && row >= p.glu_F) return;
        typedef float vf __attribute__((ext_vector_type(4), aligned(4)));  // M may be odd
        float* dst = p.y + (size_t)row * (size_t)p.M + (size_t)mt;
        if (mt + 3 < p.M) *reinterpret_cast<vf*>(dst) = vf{y[0], y[1], y[2], y[3]};
        else
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (mt + i < p.M) dst[i] = y[i];
    }
}

template <int G, int RT, int MODE>
hipError_t launch_skinny_g(hipStream_t st, const GemvProblem& p, const DigitOut& dg, int waves, int mb)
{
    constexpr int kLds = kSkMaxWaves * RT * G * 1024;
    static bool set = false;
    if (!set && kLds > 65536)
    {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_skinny<G, RT, MODE>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess) return e;
        set = true;
    }
    const unsigned nb = (unsigned)ceil_div(ceil_div((size_t)p.N, 16), (size_t)RT);
    hipLaunchKernelGGL((k_skinny<G, RT, MODE>), dim3(nb, (unsigned)mb), dim3(64 * waves), waves * RT * G * 1024, st, p, dg);
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_skinny_mode(hipStream_t st, const GemvProblem& p, const DigitOut& dg, const SkinnyPlan& s)
{
    if (s.groups == 2) return launch_skinny_g<2, 4, MODE>(st, p, dg, s.waves, s.mblocks);
    if (s.row_tiles == 4) return launch_skinny_g<1, 4, MODE>(st, p, dg, s.waves, s.mblocks);
    if (s.row_tiles == 2) return launch_skinny_g<1, 2, MODE>(st, p, dg, s.waves, s.mblocks);
    return launch_skinny_g<1, 1, MODE>(st, p, dg, s.waves, s.mblocks);
}

}  // namespace

// Cost of a plan = rounds of blocks over the CUs x k tiles x lines a block reads per k tile: 8 per
// row tile (1 KiB as stored), 64 per 16 tokens (4 loads of 16 lines). The line rate is what bounds it:
// 3.7 cycles each, time = 2.8 us + 1.74 ns x cost fits 2560 -> 6912, 64 tokens (4 row tiles x 2 groups,
// 216 blocks: 5.6 estimated, 6.1 us measured), 6912 -> 2560, 128 tokens (4 x 1, 320 blocks: 11.8, 11.3)
// and 4096 -> 11008, 48 tokens (4 x 1, 516 blocks: 10.8, 11.4). A 256 x 128 round of the GEMM costs
// kSkGemmRound per k tile on that scale (its single-round 64 x 64 blocks: 0.45 of it, 8.0 us at
// K=2560, 16.8 at K=6912), and keeps what is within 5 % of it: 2560 -> 6912, 96 tokens 8.5 against 9.0.
SkinnyPlan skinny_plan(const GemvProblem& p, int num_cus, double gemm_rounds)
{
    SkinnyPlan best{};
    const int cus = num_cus > 0 ? num_cus : 256;
    const int RTs = (p.N + 15) / 16, groups = (p.M + 15) / 16;
    double cost = 0.95 * kSkGemmRound * gemm_rounds;
    // the shapes that come out cheapest over N, M up to 32768, 4096 (two groups on fewer row tiles do not)
    constexpr int kShapes[4][2] = {{1, 1}, {2, 1}, {4, 1}, {4, 2}};
    for (const auto& shape : kShapes)
    {
        const int rt = shape[0], g = shape[1];
        if (g > groups) continue;
        const int mb = (groups + g - 1) / g, blocks = (RTs + rt - 1) / rt * mb, rounds = (blocks + cus - 1) / cus;
        const double c = rounds * (8.0 * rt + 4.0 * p.M / mb);
        if (c >= cost) continue;
        cost = c;
        best.row_tiles = rt;
        best.groups = g;
        best.mblocks = mb;
        // 16 waves per CU while there is a block per CU, 8 beyond, and as even as the k tiles go
        int want = rounds == 1 ? kSkMaxWaves : (8 * cus + blocks - 1) / blocks;
        want = want < rt * g ? rt * g : want;
        want = want > p.KT ? p.KT : want;
        const int steps = (p.KT + want - 1) / want;
        best.waves = (p.KT + steps - 1) / steps;
        if (best.waves < rt * g) best.waves = rt * g;
    }
    return best;
}

hipError_t launch_skinny(hipStream_t st, const GemvProblem& p, const DigitOut* dg, const SkinnyPlan& s)
{
    const DigitOut none{};
    if (dg) return launch_skinny_mode<kSkDigits>(st, p, *dg, s);
    if (p.glu) return launch_skinny_mode<kSkGlu>(st, p, none, s);
    return launch_skinny_mode<kSkPlain>(st, p, none, s);
}

// M <= 16: the shapes the deep GEMV is not built for, but for the ones the streaming GEMV has waves
// and LDS for (more than 4 row tiles per CU, activations within its budget: 2560 -> 60000 at 16 tokens
// 9.0 against 10.6 us). Elsewhere that kernel walks the k tiles in turn: 5120 -> 3000 at 1 / 16 tokens
// 7.1 / 24.7 -> 3.4 / 4.8 us, 11008 -> 4096 13.4 / 44.3 -> 4.4 / 8.0, 12000 -> 16000 16.7 / 49.2 ->
// 9.6 / 11.1. The deep GEMV's own shapes stay with it: in a decode step, whose weights come from HBM,
// 552 against 560 us with this kernel in its place.
bool gemv_split_ok(const GemvProblem& p, int num_cus)
{
    if (p.M < 1 || p.M > kGemvMaxM || p.ytm || gemv_deep_ok(p, num_cus)) return false;
    const bool streams = (uint32_t)p.M * (uint32_t)p.KT * kTileK <= kGemvLdsBudget &&
                         (p.N + 15) / 16 > kGemvDeepMaxTilesPerCu * (num_cus > 0 ? num_cus : 256);
    return !streams;
}

hipError_t launch_gemv_split(hipStream_t st, const GemvProblem& p, int num_cus)
{
    return launch_skinny(st, p, nullptr, skinny_plan(p, num_cus, 1e300));
}

}  // namespace nnhip
