// Projection of a prefill chunk over a Q8_0 weight matrix for gfx950: y[t][row] = sum_k W[row][k] x[t][k] with f16
// operands (the output projection W_o, and W_q, W_k, W_v in front of the attention).
//
// v_mfma_f32_32x32x16_f16 with A = x (f32 -> f16, round to nearest), B = W dequantized to f16 (d*q, one rounding: the
// precision class of the reference's f16-operand prefill kernels and of this library's chunk attention), fp32
// accumulation in the order of k whatever the tile: a token's row has the same bits in every chunk it travels in.
//
// gemm_q8_f16_kernel: a workgroup computes a tile of TT tokens x TM weight rows with two kinds of waves.  CT x CM
// consumer waves hold 32 AT x 32 BT pieces of it in registers and do nothing but LDS operand reads and MFMAs; NW
// producer waves fetch the next steps' activations and weights, dequantize or convert them, and write the f16 operand
// tiles.  A step is KU pairs of blocks (64 KU values of k); the tiles are double buffered, with one barrier per step.
//
// What bounds it (timing-only builds at 12288 x 5120 over 672 tokens, 192 x 192 tiles, us): the consumers alone 76
// (1,110 TFLOP/s; a large library f16 GEMM reaches 1,200 on the same card), the producers' staging alone 42, their
// loads alone 90 (f32 activations) or 67 (f16).  Hence:
//  * large tiles.  128 x 128 tiles read 128 bytes of LDS per cycle for 100 % MFMA, all that LDS serves, and move 80
//    bytes of f32 activations and weights per cycle through the CU's 64-byte vector memory path; 192 x 192 need 83 and
//    53, 256 x 192 need 73 and 50.
//  * half of the producer waves ask for the next record before they stage, the other half behind it.  Asked for by all
//    of them at once the loads queue up (one request per ~25 cycles and CU) while no wave stages, and a step costs the
//    sum of both: 2,150 cycles against 1,500 (192 x 192: 146 -> 117 us; 256 x 192 over 1,024 tokens: 166 -> 144 us).
//  * small tiles with longer steps (KU 2 and 4) and eight producer waves where there are too few outputs for large
//    ones: a step's cost is then latency, not work (1024 x 5120 over 117 tokens: 32 x 32 tiles 15 us, 128 x 128 48 us).
// Before (128 x 128 tiles for every shape) and now, us: 12288 x 5120 over 117 / 672 / 1,024 / 2,048 tokens 78 / 173 /
// 217 / 432 -> 34 / 117 / 144 / 284; 1024 x 5120 over the same 54 / 56 / 58 / 60 -> 15 / 25 / 32 / 49; 5120 x 6144
// (f16 activations) 50 / 58 / 111 / 172 -> 24 / 58 / 81 / 137.
//
// Weight fetch: the four lanes of a quad take the quarters of a pair of blocks of one row, 12 bytes of the even block
// (2 bytes in; the scales ride along in lanes 0 and 3) and 8 of the odd one, dword aligned.
// A tile row in LDS is an odd number of 16-byte groups: 128-bit reads and writes of 16 consecutive rows touch every
// bank once.

#include "q8_weights.h"

#include <type_traits>

namespace hipml {

constexpr int gemm_pitch(int ku) { return 128 * ku + 16; } // bytes of a tile row
constexpr int gemm_lds(int tt, int tm, int ku) { return 2 * (tt + tm) * gemm_pitch(ku); } // double buffered

template <int WN, int XN>
struct GemmFetch {
    uint3a4 e[WN]; // even-block quarter (+ scales in quad lanes 0 and 3)
    uint2a4 o[WN]; // odd-block quarter
    float4v x[XN]; // f32: 4 activations; f16: 8
};

__device__ __forceinline__ half8 dequant8(uint32_t w0, uint32_t w1, _Float16 d)
{
    const half8 q = int8x8_to_f16(w0, w1);
    const half8 dv = {d, d, d, d, d, d, d, d};
    return q * dv;
}


template <bool X16, int CT, int CM, int AT, int BT, int KU, int NW, int R>
__global__ void __launch_bounds__(64 * (NW + CT * CM)) gemm_q8_f16_kernel(const uint8_t *__restrict__ w,
                                                                              const void *__restrict__ xv,
                                                                              float *__restrict__ y, int m, int k,
                                                                              int tokens)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int NT = 64 * NW; // producer threads
    constexpr int NC = CT * CM;
    constexpr int TT = 32 * AT * CT, TM = 32 * BT * CM;
    constexpr int kGemmK = 64 * KU;           // values of k per step: KU 68-byte pairs of blocks per weight row
    constexpr int kGemmPitch = gemm_pitch(KU);
    constexpr int kXTile = TT * kGemmPitch, kBuf = (TT + TM) * kGemmPitch;
    const bool producer = threadIdx.x >= 64 * NC;
    const int tid = producer ? threadIdx.x - 64 * NC : threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63; // within the role
    const int m0 = blockIdx.x * TM, t0 = blockIdx.y * TT;
    const int nsteps = k / kGemmK;

    if (producer) {
        const uint32_t row_bytes = (uint32_t)(k >> 5) * kQ8Block;
        constexpr int WP = TM * 4 * KU / NT; // weight (unit, row, quarter) triples per producer thread
        static_assert(WP * NT == TM * 4 * KU, "");
        constexpr int XELT = X16 ? 2 : 4;  // bytes per activation
        constexpr int XV = 16 / XELT;      // activations per 16-byte piece
        constexpr int XPR = kGemmK / XV;   // pieces per tile row
        constexpr int XN = TT * XPR / NT;  // pieces per producer thread
        static_assert(XN * NT == TT * XPR, "");
        constexpr int XROWS = NT / XPR;    // rows covered by one piece of the workgroup
        const uint8_t *wb = w + (size_t)m0 * row_bytes;
        uint32_t woff[WP], wlds[WP];
#pragma unroll
        for (int h = 0; h < WP; h++) {
            const int rest = (h * NT + tid) >> 2, fg = tid & 3;
            const int r = rest % TM, unit = rest / TM; // (four lanes share a row: its k quarters)
            const int row = m0 + r < m ? r : m - 1 - m0;
            woff[h] = (uint32_t)row * row_bytes + unit * (2 * kQ8Block) + fg * 8;
            wlds[h] = kXTile + r * kGemmPitch + unit * 128 + fg * 16;
        }
        const int xr = tid / XPR, xc = tid % XPR;
        const uint8_t *xb = static_cast<const uint8_t *>(xv) + (size_t)t0 * k * XELT;
        uint32_t xoff[XN];
#pragma unroll
        for (int i = 0; i < XN; i++) {
            const int t = t0 + xr + XROWS * i < tokens ? xr + XROWS * i : tokens - 1 - t0;
            xoff[i] = (uint32_t)t * (uint32_t)(k * XELT) + xc * 16;
        }
        typedef GemmFetch<WP, XN> Fetch;
        // piece h of a record: WP of them, each one weight pair and its share of the activations
        auto fetch_piece = [&](Fetch &f, int s, int h) {
            const int sc = s < nsteps ? s : nsteps - 1;
            const uint8_t *ws = wb + (size_t)sc * (2 * KU * kQ8Block);
            const uint8_t *xs = xb + (size_t)sc * (kGemmK * XELT);
            const uint8_t *unit = ws + woff[h];
            f.e[h] = *reinterpret_cast<const uint3a4 *>(unit);
            f.o[h] = *reinterpret_cast<const uint2a4 *>(unit + 36);
#pragma unroll
            for (int i = h * XN / WP; i < (h + 1) * XN / WP; i++)
                f.x[i] = *reinterpret_cast<const float4v *>(xs + xoff[i]);
        };
        auto fetch = [&](Fetch &f, int s) {
#pragma unroll
            for (int h = 0; h < WP; h++)
                fetch_piece(f, s, h);
        };
        uint8_t *xdst = lds + xr * kGemmPitch + xc * (X16 ? 16 : 8);
        auto stage_piece = [&](const Fetch &f, int b, int h) {
            const uint3a4 e = f.e[h];
            const uint32_t s0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e[0], 0x00, 0xf, 0xf, true);
            const uint32_t s1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e[2], 0xFF, 0xf, 0xf, true);
            const _Float16 d0 = __builtin_bit_cast(_Float16, (uint16_t)(s0 & 0xffffu));
            const _Float16 d1 = __builtin_bit_cast(_Float16, (uint16_t)(s1 >> 16));
            const half8 v0 = dequant8(__builtin_amdgcn_alignbit(e[1], e[0], 16),
                                      __builtin_amdgcn_alignbit(e[2], e[1], 16), d0);
            const half8 v1 = dequant8(f.o[h][0], f.o[h][1], d1);
            uint8_t *dw = lds + b * kBuf + wlds[h];
            *reinterpret_cast<half8 *>(dw) = v0;      // k = fg*8 .. of the even block
            *reinterpret_cast<half8 *>(dw + 64) = v1; // k = 32 + fg*8 .. (the odd block)
#pragma unroll
            for (int i = h * XN / WP; i < (h + 1) * XN / WP; i++) {
                uint8_t *d = xdst + b * kBuf + XROWS * i * kGemmPitch;
                if (X16)
                    *reinterpret_cast<float4v *>(d) = f.x[i];
                else // round to nearest even: truncation would bias every product the same way
                    *reinterpret_cast<half4v *>(d) = __builtin_convertvector(f.x[i], half4v);
            }
        };
        auto stage = [&](const Fetch &f, int b) {
#pragma unroll
            for (int h = 0; h < WP; h++)
                stage_piece(f, b, h);
        };
        Fetch rec[R];
        constexpr int U = R & 1 ? 2 * R : R;
        auto produce = [&](auto first) {
            constexpr bool kLoadFirst = decltype(first)::value;
            // records: step s + 1 .. s + R are on the way (load first: s + 1 .. s + R - 1, the newest is asked for at
            // the head of the turn)
#pragma unroll
            for (int r = 0; r < R; r++)
                fetch(rec[r], r);
            stage(rec[0], 0);
            if (!kLoadFirst)
                fetch(rec[0], R);
            __syncthreads();
            auto step = [&](int u, int s) {
                if (kLoadFirst) {
                    fetch(rec[u % R], s + R);
                    __builtin_amdgcn_sched_barrier(0);
                    stage(rec[(u + 1) % R], (u + 1) & 1);
                } else {
                    stage(rec[(u + 1) % R], (u + 1) & 1);
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(rec[(u + 1) % R], s + 1 + R);
                }
            };
            int s = 0;
#pragma unroll 1
            for (; s + U < nsteps; s += U) {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    step(u, s + u);
                    __syncthreads();
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (s + u + 1 < nsteps)
                    step(u, s + u);
                if (s + u < nsteps)
                    __syncthreads();
            }
        };
        if (wave & 1)
            produce(std::integral_constant<bool, true>{});
        else
            produce(std::integral_constant<bool, false>{});
        return;
    }
    // consumer wave (wt, wm): tokens wt * 32 AT .., weight rows wm * 32 BT ..
    const int wt_ = wave / CM, wm_ = wave % CM;
    const int ln = lane & 31, lh = lane >> 5;
    float16v acc[AT][BT];
#pragma unroll
    for (int a = 0; a < AT; a++)
#pragma unroll
        for (int b = 0; b < BT; b++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                acc[a][b][i] = 0.0f;
    auto multiply = [&](const uint8_t *buf) {
        const uint8_t *xa = buf + (wt_ * 32 * AT + ln) * kGemmPitch + lh * 16;
        const uint8_t *wb = buf + kXTile + (wm_ * 32 * BT + ln) * kGemmPitch + lh * 16;
        constexpr int per = AT + BT, mf = AT * BT, rr = (per + mf - 1) / mf;
        constexpr int pairs = per < mf ? per : mf;
        // operands of 16 values of k are read while those of the 16 before them are multiplied: one MFMA and one
        // read in turn
        half8 A[2][AT], B[2][BT];
        auto read = [&](int kk) {
#pragma unroll
            for (int a = 0; a < AT; a++)
                A[kk & 1][a] = *reinterpret_cast<const half8 *>(xa + a * 32 * kGemmPitch + kk * 32);
#pragma unroll
            for (int b = 0; b < BT; b++)
                B[kk & 1][b] = *reinterpret_cast<const half8 *>(wb + b * 32 * kGemmPitch + kk * 32);
        };
        read(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 4 * KU; kk++) {
            if (kk + 1 < 4 * KU)
                read(kk + 1);
#pragma unroll
            for (int a = 0; a < AT; a++)
#pragma unroll
                for (int b = 0; b < BT; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[kk & 1][a], B[kk & 1][b], acc[a][b], 0, 0, 0);
            if (kk + 1 < 4 * KU) {
#pragma unroll
                for (int i = 0; i < pairs; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, rr, 0);
                }
                if (mf > pairs)
                    __builtin_amdgcn_sched_group_barrier(0x008, mf - pairs, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __syncthreads();
#pragma unroll 1
    for (int s = 0; s < nsteps; s++) {
        multiply(lds + (s & 1) * kBuf);
        __syncthreads();
    }

    // C tile: lane holds column ln (weight row), rows (i/4)*8 + lh*4 + i%4 (tokens)
#pragma unroll
    for (int a = 0; a < AT; a++)
#pragma unroll
        for (int b = 0; b < BT; b++) {
            const int row = m0 + (wm_ * BT + b) * 32 + ln;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int t = t0 + (wt_ * AT + a) * 32 + (i >> 2) * 8 + lh * 4 + (i & 3);
                if (t < tokens && row < m)
                    y[(size_t)t * m + row] = acc[a][b][i];
            }
        }
}

// x16[i] = f16(x[i] * sigmoid(gate[i])) (gate may be null: plain conversion), 8 values per thread.
// The gate is the expression every gating kernel of this library uses, the rounding the one the
// f32-activation GEMM applies when it stages x: the two routes give the same bits.
__global__ void __launch_bounds__(256) gate_f16_kernel(const float4v *__restrict__ x,
                                                      const float4v *__restrict__ gate,
                                                      half8 *__restrict__ x16, size_t n8)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8)
        return;
    float4v a = x[2 * i], b = x[2 * i + 1];
    if (gate != nullptr) {
        const float4v ga = gate[2 * i], gb = gate[2 * i + 1];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            a[j] = gated(a[j], ga[j]);
            b[j] = gated(b[j], gb[j]);
        }
    }
    const half4v ha = __builtin_convertvector(a, half4v), hb = __builtin_convertvector(b, half4v);
    half8 h;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        h[j] = ha[j];
        h[4 + j] = hb[j];
    }
    x16[i] = h;
}

// ---- which tile ----------------------------------------------------------------------------------------------
//
// (token rows and weight rows of the tile, 64-value units per step, microseconds per unit and round of the chip's 256
// CUs as measured with one round of workgroups at k = 5120)
struct GemmTile {
    int tt, tm, ku;
    float cost;
};
constexpr GemmTile kGemmTiles[] = {
    {32, 32, 4, 0.14f},    {32, 64, 4, 0.17f},    {64, 64, 2, 0.23f},    {64, 128, 2, 0.35f},
    {128, 128, 1, 0.53f},  {192, 128, 1, 0.70f},  {128, 192, 1, 0.76f},  {192, 192, 1, 0.92f}, {256, 192, 1, 1.12f},
    {64, 64, 1, 0.33f}, // (the smallest for an odd number of units)
};
constexpr int kGemmNTiles = sizeof(kGemmTiles) / sizeof(kGemmTiles[0]);

// The tile for a shape: the cheapest by rounds x cost, where a round of 256 workgroups slows down as it fills (they
// share L2, HBM and the power budget: 1.5 times the cost of a lone workgroup when all CUs have one).  The estimate is
// within 10 % of the measured time at 40 shapes, and picks the measured best or one within 5 % of it.
static int gemm_tile(int m, int k, int tokens)
{
    int best = -1;
    float best_cost = 0.0f;
    for (int i = 0; i < kGemmNTiles; i++) {
        const GemmTile &g = kGemmTiles[i];
        // (a tile's rows are addressed with 32-bit offsets)
        if (k % (64 * g.ku) != 0 || (uint64_t)(g.tt > g.tm ? g.tt : g.tm) * (uint64_t)k * 4 >= (1ull << 32))
            continue;
        const long long wg = (long long)((m + g.tm - 1) / g.tm) * ((tokens + g.tt - 1) / g.tt);
        const long long rounds = (wg + 255) / 256;
        const float fill = (float)wg / (256.0f * (float)rounds);
        const float cost = (float)rounds * g.cost * (1.0f + 0.5f * fill * fill);
        if (best < 0 || cost < best_cost) {
            best = i;
            best_cost = cost;
        }
    }
    return best;
}

// Calls f with the kernel of tile i and its launch figures: (kernel, threads, tile tokens, tile rows, LDS bytes).
template <bool X16, typename F>
static bool with_gemm_kernel(int i, F &&f)
{
#define HIPML_GEMM(idx, CT, CM, AT, BT, KU, NW, R)                                                                     \
    case idx: {                                                                                                       \
        constexpr int tt = 32 * AT * CT, tm = 32 * BT * CM;                                                           \
        static_assert(kGemmTiles[idx].tt == tt && kGemmTiles[idx].tm == tm && kGemmTiles[idx].ku == KU, "the table"); \
        return f(&gemm_q8_f16_kernel<X16, CT, CM, AT, BT, KU, NW, R>, 64 * (NW + CT * CM), tt, tm,                    \
                 gemm_lds(tt, tm, KU));                                                                               \
    }
    switch (i) {
        HIPML_GEMM(0, 1, 1, 1, 1, 4, 8, 2)
        HIPML_GEMM(1, 1, 2, 1, 1, 4, 8, 2)
        HIPML_GEMM(2, 2, 2, 1, 1, 2, 8, 2)
        HIPML_GEMM(3, 2, 2, 1, 2, 2, 8, 2)
        HIPML_GEMM(4, 2, 2, 2, 2, 1, 8, 4)
        HIPML_GEMM(5, 2, 2, 3, 2, 1, 4, 2)
        HIPML_GEMM(6, 2, 2, 2, 3, 1, 4, 2)
        HIPML_GEMM(7, 2, 2, 3, 3, 1, 4, 2)
        HIPML_GEMM(8, 2, 2, 4, 3, 1, 4, 2)
        HIPML_GEMM(9, 2, 2, 1, 1, 1, 4, 4)
    default:
        return false;
    }
#undef HIPML_GEMM
}

int gemm_init()
{
    hipError_t e = hipSuccess;
    auto raise = [&](auto kernel, int, int, int, int lds) {
        if (e == hipSuccess)
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        return true;
    };
    for (int i = 0; i < kGemmNTiles; i++) {
        with_gemm_kernel<false>(i, raise);
        with_gemm_kernel<true>(i, raise);
    }
    if (e != hipSuccess)
        return fail((int)e, "hipFuncSetAttribute(chunk projection LDS) failed: %d (%s)", (int)e, hipGetErrorString(e));
    return 0;
}

// x16 != nullptr: gate (optional) and convert into x16 first, then the GEMM over f16 activations;
// x == nullptr: x16 already holds them.
int launch_gemm_q8_f16(hipStream_t st, const uint8_t *w, const float *x, const float *gate, float *y, int m,
                       int k, int tokens, void *x16)
{
    if (x16 != nullptr && x != nullptr) {
        const size_t n8 = (size_t)tokens * k / 8;
        HIPML_LAUNCH(gate_f16_kernel, dim3((unsigned)((n8 + 255) / 256), 1, 1), dim3(256, 1, 1), 0, st,
                           reinterpret_cast<const float4v *>(x), reinterpret_cast<const float4v *>(gate),
                           static_cast<half8 *>(x16), n8);
        int rc = launched("gate_f16");
        if (rc)
            return rc;
    }
    const void *act = x16 != nullptr ? x16 : x;
    auto go = [&](auto kernel, int threads, int tt, int tm, int lds) {
        HIPML_LAUNCH(kernel, dim3((unsigned)((m + tm - 1) / tm), (unsigned)((tokens + tt - 1) / tt), 1),
                     dim3(threads, 1, 1), lds, st, w, act, y, m, k, tokens);
        return true;
    };
    const int tile = gemm_tile(m, k, tokens);
    if (tile < 0)
        return fail(HIPML_ATTN_E_RANGE, "k %d: 32 rows of activations exceed 4 GB", k);
    if (x16 != nullptr)
        with_gemm_kernel<true>(tile, go);
    else
        with_gemm_kernel<false>(tile, go);
    return launched("gemm_q8_0_f16");
}

} // namespace hipml
