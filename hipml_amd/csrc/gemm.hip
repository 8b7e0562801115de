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
//    Not so for 128 x 128 tiles over f16 activations, whose step has the fewest loads for its eight producer waves: there
//    all of them stage first and four records cover the loads (5120 x 6144 over 512 / 672 tokens 50.8 -> 47.5 / 62.6 ->
//    58.6 us).
//  * small tiles with longer steps (KU 2 and 4) and eight producer waves where there are too few outputs for large
//    ones: a step's cost is then latency, not work (1024 x 5120 over 117 tokens: 64 x 64 tiles 23 us, 128 x 128 44 us; the
//    smallest tiles are gemm_q8_few_kernel's).
//  * weights by whole 64-byte sectors, one aligned request of a quad of lanes each, where their rows allow it.  A row's
//    pair of blocks is 68 bytes: asked for as it lies (12 and 8 bytes a lane) it takes three requests, most of them
//    across a sector boundary, and the weights of a step cost the vector memory path as much as the activations
//    (192 x 192 over 672 tokens 121 -> 108 us, 64 x 128 over 117 48 -> 42, 64 x 64 31 -> 27).  Tried on it: two sectors
//    of a line asked for together (no gain), activations non-temporal (10 % slower), deeper records (no gain).
// The kernel before this one (128 x 128 tiles for every shape) and this one, us: 12288 x 5120 over 117 / 672 / 1,024 /
// 2,048 tokens 76 / 178 / 202 / 397 -> 40 / 114 / 144 / 282; 1024 x 5120 over the same 52 / 55 / 58 / 63 -> 11 / 24 / 28 /
// 51; 5120 x 6144 (f16 activations) 44 / 58 / 102 / 166 -> 23 / 58 / 80 / 131.
//
// A tile row in LDS is an odd number of 16-byte groups: 128-bit reads and writes of 16 consecutive rows touch every
// bank once.

#include "q8_weights.h"

#include <type_traits>

namespace hipml {

constexpr int gemm_pitch(int ku) { return 128 * ku + 16; } // bytes of a tile row
constexpr int gemm_lds(int tt, int tm, int ku) { return 2 * (tt + tm) * gemm_pitch(ku); } // double buffered

__device__ __forceinline__ half8 dequant8(uint32_t w0, uint32_t w1, _Float16 d)
{
    const half8 q = int8x8_to_f16(w0, w1);
    const half8 dv = {d, d, d, d, d, d, d, d};
    return q * dv;
}


// The lane at quad position i gets the value of position i + 1, the last one that of position 0.
__device__ __forceinline__ uint32_t quad_next(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x39, 0xf, 0xf, true);
}

// ... position i - 1, the first one that of position 3.
__device__ __forceinline__ uint32_t quad_prev(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x93, 0xf, 0xf, true);
}

// The weights of one producer thread's rows, for rows of whole 64-byte sectors (k a multiple of 1,024, W at a 64-byte
// boundary): the four lanes of a quad share a row and load a sector in one request, lane i its 16 bytes i.  A set is
// the five sectors that hold four units: unit u (17 dwords) starts u % 16 dwords into sector u + u / 16.
template <int WS, int SETS>
struct WideWeights {
    uint4v p[SETS][WS][5];
};
// The same for any k of whole units and W at a 4-byte boundary: a lane takes a quarter of a pair of blocks, 12 bytes
// of the even block (2 bytes in; the scales ride along in lanes 0 and 3) and 8 of the odd one.
template <int WP, int SETS>
struct QuarterWeights {
    uint3a4 e[SETS][WP];
    uint2a4 o[SETS][WP];
};

// Unit j of a set from the sectors it starts in and behind, into a row of the LDS tile.  In set c it starts j dwords into
// the 16 bytes of lane q = c % 4 of sector j.  The lanes from q on, then those before it with the next sector, are the
// unit's logical lanes 0 .. 3 (this one is lane (qi - q) % 4, and dst its place): a logical lane's 16 values are its own
// dwords j .. 3 and the first of the lane behind it (for the last, of the next sector of lane q).  Logical lanes 0 and 1
// hold the even block, whose values start 2 bytes in, 2 and 3 the odd one, a dword further; the scales lie at the head of
// lane 0 and in the upper half of lane 2's first dword.
__device__ __forceinline__ void stage_unit(const uint4v p0, const uint4v p1, const int j, int qi, int q, uint8_t *dst)
{
    const int li = (qi - q) & 3;
    const bool here = qi >= q, past = qi > q, odd = li >= 2;
    const uint32_t pick = odd ? 0x07060504u : 0x05040302u, shift = odd ? 16u : 0u;
    uint32_t d[5];
#pragma unroll
    for (int n = 0; n < 5; n++) {
        const int e = (j + n) & 3;
        d[n] = j + n < 4 ? (here ? p0[e] : p1[e]) : quad_next(past ? p0[e] : p1[e]);
    }
    const uint32_t prev = quad_prev(d[0]); // (outside the choice: every lane takes part)
    const uint32_t sc = ((li & 1) ? prev : d[0]) >> shift;
    const _Float16 scale = __builtin_bit_cast(_Float16, (uint16_t)sc);
    uint32_t v[4];
#pragma unroll
    for (int n = 0; n < 4; n++)
        v[n] = __builtin_amdgcn_perm(d[n + 1], d[n], pick);
    *reinterpret_cast<half8 *>(dst) = dequant8(v[0], v[1], scale);
    *reinterpret_cast<half8 *>(dst + 16) = dequant8(v[2], v[3], scale);
}

// TURNS: half of the producer waves ask for the next record before they stage (above); else all of them stage first,
// activations ahead of weights, and R records cover the loads.
template <bool X16, bool WIDE, int CT, int CM, int AT, int BT, int KU, int NW, int R, bool TURNS = true>
__global__ void __launch_bounds__(64 * (NW + CT * CM)) gemm_q8_f16_kernel(const uint8_t *__restrict__ w,
                                                                          const void *__restrict__ xv,
                                                                          float *__restrict__ y, int m, int k, int tokens)
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
        // ---- activations: XN pieces of 16 bytes per thread and step, R steps on the way
        constexpr int XELT = X16 ? 2 : 4; // bytes per activation
        constexpr int XV = 16 / XELT;     // activations per piece
        constexpr int XPR = kGemmK / XV;  // pieces per tile row
        constexpr int XN = TT * XPR / NT;
        static_assert(XN * NT == TT * XPR, "");
        constexpr int XROWS = NT / XPR; // rows covered by one piece of the workgroup
        const int xr = tid / XPR, xc = tid % XPR;
        const uint8_t *xb = static_cast<const uint8_t *>(xv) + (size_t)t0 * k * XELT;
        uint32_t xoff[XN];
#pragma unroll
        for (int i = 0; i < XN; i++) {
            const int t = t0 + xr + XROWS * i < tokens ? xr + XROWS * i : tokens - 1 - t0;
            xoff[i] = (uint32_t)t * (uint32_t)(k * XELT) + xc * 16;
        }
        float4v xrec[R][XN]; // f32: 4 activations; f16: 8
        auto fetch_x = [&](int r, int s) {
            const uint8_t *xs = xb + (size_t)(s < nsteps ? s : nsteps - 1) * (kGemmK * XELT);
#pragma unroll
            for (int i = 0; i < XN; i++)
                xrec[r][i] = *reinterpret_cast<const float4v *>(xs + xoff[i]);
        };
        uint8_t *xdst = lds + xr * kGemmPitch + xc * (X16 ? 16 : 8);
        auto stage_x = [&](int r, int b) {
#pragma unroll
            for (int i = 0; i < XN; i++) {
                uint8_t *d = xdst + b * kBuf + XROWS * i * kGemmPitch;
                if (X16)
                    *reinterpret_cast<float4v *>(d) = xrec[r][i];
                else // round to nearest even: truncation would bias every product the same way
                    *reinterpret_cast<half4v *>(d) = __builtin_convertvector(xrec[r][i], half4v);
            }
        };

        // ---- weights
        const uint32_t row_bytes = (uint32_t)(k >> 5) * kQ8Block;
        const uint8_t *wb = w + (size_t)m0 * row_bytes;
        constexpr int CS = WIDE ? 4 / KU : 1;                     // steps per set
        constexpr int SETS = WIDE ? (KU == 1 ? 1 : 2) : R;
        constexpr int WWAVES = WIDE && TM < 16 * NW ? TM / 16 : NW; // waves that carry weights
        constexpr int WS = WIDE ? TM / (16 * WWAVES) : TM * 4 * KU / NT; // rows, or (unit, row, quarter) triples, per thread
        static_assert(WIDE ? WS * 16 * WWAVES == TM : WS * NT == TM * 4 * KU, "");
        typename std::conditional<WIDE, WideWeights<WS, SETS>, QuarterWeights<WS, SETS>>::type wrec;
        uint32_t woff[WS], wlds[WS];
        const int qi = tid & 3; // four lanes share a row
#pragma unroll
        for (int h = 0; h < WS; h++) {
            const int rest = WIDE ? (h * 64 * WWAVES + tid) >> 2 : (h * NT + tid) >> 2;
            const int r = rest % TM, unit = rest / TM;
            const int row = m0 + r < m ? r : m - 1 - m0;
            woff[h] = (uint32_t)row * row_bytes + (WIDE ? qi * 16 : unit * (2 * kQ8Block) + qi * 8);
            wlds[h] = kXTile + r * kGemmPitch + (WIDE ? 0 : unit * 128 + qi * 16);
        }
        const int nsets = nsteps / CS;
        // what staging position v (a step within the SETS sets) leaves free of set v / CS is asked for anew, SETS sets on
        auto fetch_w = [&](int v, int s) {
            const int set = v / CS % SETS, sub = v % CS;
            if constexpr (WIDE) {
                int c = (s + CS * SETS) / CS;
                c = c < nsets ? c : nsets - 1;
                const uint8_t *ws = wb + (size_t)(4 * c + (c >> 2)) * 64;
#pragma unroll
                for (int h = 0; h < WS; h++) {
#pragma unroll
                    for (int j = sub * KU; j < (sub + 1) * KU; j++)
                        wrec.p[set][h][j] = *reinterpret_cast<const uint4v *>(ws + woff[h] + j * 64);
                    if (sub == CS - 1)
                        wrec.p[set][h][4] = *reinterpret_cast<const uint4v *>(ws + woff[h] + 256);
                }
            } else {
                const int c = s + SETS < nsteps ? s + SETS : nsteps - 1;
                const uint8_t *ws = wb + (size_t)c * (2 * KU * kQ8Block);
#pragma unroll
                for (int h = 0; h < WS; h++) {
                    wrec.e[set][h] = *reinterpret_cast<const uint3a4 *>(ws + woff[h]);
                    wrec.o[set][h] = *reinterpret_cast<const uint2a4 *>(ws + woff[h] + 36);
                }
            }
        };
        auto stage_w = [&](int v, int s, int b) {
            const int set = v / CS % SETS, sub = v % CS;
            if constexpr (WIDE) {
                const int q = (s / CS) & 3;
                uint8_t *const dst0 = lds + b * kBuf + ((qi - q) & 3) * 32;
#pragma unroll
                for (int h = 0; h < WS; h++)
#pragma unroll
                    for (int u = 0; u < KU; u++) {
                        const int j = sub * KU + u;
                        stage_unit(wrec.p[set][h][j], wrec.p[set][h][j + 1], j, qi, q, dst0 + wlds[h] + u * 128);
                    }
            } else {
#pragma unroll
                for (int h = 0; h < WS; h++) {
                    const uint3a4 e = wrec.e[set][h];
                    const uint32_t s0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e[0], 0x00, 0xf, 0xf, true);
                    const uint32_t s1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e[2], 0xFF, 0xf, 0xf, true);
                    const _Float16 d0 = __builtin_bit_cast(_Float16, (uint16_t)(s0 & 0xffffu));
                    const _Float16 d1 = __builtin_bit_cast(_Float16, (uint16_t)(s1 >> 16));
                    uint8_t *dst = lds + b * kBuf + wlds[h];
                    *reinterpret_cast<half8 *>(dst) = dequant8(__builtin_amdgcn_alignbit(e[1], e[0], 16),
                                                               __builtin_amdgcn_alignbit(e[2], e[1], 16), d0);
                    *reinterpret_cast<half8 *>(dst + 64) = dequant8(wrec.o[set][h][0], wrec.o[set][h][1], d1);
                }
            }
        };

        constexpr int CYCLE = CS * SETS;
        constexpr int U0 = R % 2 ? 2 * R : R, U = CYCLE > U0 ? CYCLE : U0;
        static_assert(U % U0 == 0 && U % CYCLE == 0, "the records of a turn of the loop are named at compile time");
        auto produce = [&](auto load_first, auto weights) {
            constexpr bool kLoadFirst = decltype(load_first)::value, kWeights = decltype(weights)::value;
            auto fetch = [&](int v, int s) { // what staging step s (position v) has left free
                if (kWeights)
                    fetch_w(v % CYCLE, s);
                fetch_x(v % R, s + R);
            };
            auto stage = [&](int v, int s) {
                if (!TURNS)
                    stage_x(v % R, v & 1);
                if (kWeights)
                    stage_w(v % CYCLE, s, v & 1);
                if (TURNS)
                    stage_x(v % R, v & 1);
            };
            if (kWeights) {
#pragma unroll
                for (int v = 0; v < CYCLE; v++)
                    fetch_w(v, v - CYCLE);
            }
#pragma unroll
            for (int r = 0; r < R; r++)
                fetch_x(r, r);
            stage(0, 0);
            if (!kLoadFirst)
                fetch(0, 0);
            __syncthreads();
            auto step = [&](int u, int s) { // stage step s + 1 while step s is multiplied
                if (kLoadFirst) {
                    fetch(u, s);
                    __builtin_amdgcn_sched_barrier(0);
                    stage(u + 1, s + 1);
                } else {
                    stage(u + 1, s + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(u + 1, s + 1);
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
        const std::true_type yes;
        const std::false_type no;
        if (WWAVES < NW && wave >= WWAVES) {
            if (TURNS && (wave & 1))
                produce(yes, no);
            else
                produce(no, no);
        } else if (TURNS && (wave & 1)) {
            produce(yes, yes);
        } else {
            produce(no, yes);
        }
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
    // operands of 16 values of k are read while those of the 16 before them are multiplied: one MFMA and one read in turn.
    // A step's barrier stands where its last operands have been read, in front of the last MFMAs, behind which the next
    // step's first operands are read: the barrier and the first reads behind it cost little MFMA time (with the barrier at
    // the end of the step the large tiles take 1 to 3 % more: 12288 x 5120 over 1,024 tokens 146.5 us, here 143.5).
    const uint8_t *xa = lds + (wt_ * 32 * AT + ln) * kGemmPitch + lh * 16;
    const uint8_t *wb = lds + kXTile + (wm_ * 32 * BT + ln) * kGemmPitch + lh * 16;
    half8 A[2][AT], B[2][BT];
    auto read = [&](int kk) {
#pragma unroll
        for (int a = 0; a < AT; a++)
            A[kk & 1][a] = *reinterpret_cast<const half8 *>(xa + a * 32 * kGemmPitch + kk * 32);
#pragma unroll
        for (int b = 0; b < BT; b++)
            B[kk & 1][b] = *reinterpret_cast<const half8 *>(wb + b * 32 * kGemmPitch + kk * 32);
    };
    auto multiply = [&](int kk) {
        constexpr int per = AT + BT, mf = AT * BT, rr = (per + mf - 1) / mf;
        constexpr int pairs = per < mf ? per : mf;
#pragma unroll
        for (int a = 0; a < AT; a++)
#pragma unroll
            for (int b = 0; b < BT; b++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[kk & 1][a], B[kk & 1][b], acc[a][b], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < pairs; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, rr, 0);
        }
        if (mf > pairs)
            __builtin_amdgcn_sched_group_barrier(0x008, mf - pairs, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int kSlices = 4 * KU; // of 16 values of k in a step: an even number
    __syncthreads();
    read(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int s = 0; s < nsteps; s++) {
#pragma unroll
        for (int kk = 0; kk + 1 < kSlices; kk++) {
            read(kk + 1);
            multiply(kk);
        }
        __syncthreads();
        const int other = s & 1 ? -kBuf : kBuf;
        xa += other;
        wb += other;
        read(0); // (behind the last step: whatever the other buffer holds, not used)
        multiply(kSlices - 1);
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

// A producer wave's turns in the two kernels below: R steps on the way, step s + 1 staged while step s is multiplied.
// fetch(record, step), past the last step too; stage(record, step, buffer).
template <int R, typename F, typename S>
__device__ __forceinline__ void produce_steps(int nsteps, F &&fetch, S &&stage)
{
    constexpr int U = R % 2 ? 2 * R : R;
#pragma unroll
    for (int r = 0; r < R; r++)
        fetch(r, r);
    stage(0, 0, 0);
    fetch(0, R);
    __syncthreads();
    int s = 0;
#pragma unroll 1
    for (; s + U < nsteps; s += U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            stage((u + 1) % R, s + u + 1, (u + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
            fetch((u + 1) % R, s + u + 1 + R);
            __syncthreads();
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (s + u + 1 < nsteps) {
            stage((u + 1) % R, s + u + 1, (u + 1) & 1);
            if (u + 1 + R < U)
                fetch((u + 1) % R, s + u + 1 + R);
        }
        if (s + u < nsteps)
            __syncthreads();
    }
}

// ---- gemm_q8_few_kernel: 16 AT tokens x 32 weight rows ------------------------------------------------------------
//
// The same product for calls with few outputs, where a step of the kernel above is latency: 1024 x 5120 over 16 tokens
// took as long as over 200 (15.6 and 16.6 us for some 5 us of loads).  Here a workgroup's waves each have one short thing
// to do per step of 256 values of k: four weight waves stage 16 rows x 128 values each (three sectors asked for, two units
// dequantized; a wave of the kernel above had 16 rows x 256 values, its longest chain), four the activations, and two
// consumer waves multiply with v_mfma_f32_16x16x32_f16, whose chain takes as long for 32 values of k as that of
// v_mfma_f32_32x32x16_f16 for 16 (and gives its bits).  16 tokens a tile also make twice the workgroups of 32 x 32.
// R steps are on the way in registers: three with AT = 1, two with 2 (three need more registers than ten waves have).
// Weights as WIDE above (whole sectors, k a multiple of 1,024).
// Tile 0 of the kernel above before, us over f32 / f16 activations: 1024 x 5120 over 16 / 117 / 200 tokens 15.7 / 16.2 / 16.9
// and 15.5 / 15.9 / 16.4, here 9.7 / 10.9 / 14.0 and 9.4 / 10.3 / 12.2; 5120 x 6144 over 16 tokens 19.3 and 18.8, here 15.6
// and 12.5.  Tried on it: 16 x 64, 32 x 64, 64 x 32 and 64 x 64 tiles (behind the kernel above wherever they beat 32 x 32);
// weights by quarters of a pair of blocks instead of whole sectors (10 % slower); 16 x 32 with two steps on the way (6 to
// 30 % slower).
template <bool X16, int AT, int R>
__global__ void __launch_bounds__(640) gemm_q8_few_kernel(const uint8_t *__restrict__ w, const void *__restrict__ xv,
                                                          float *__restrict__ y, int m, int k, int tokens)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int KU = 4, NC = 2, NA = 4, TT = 16 * AT, TM = 32;
    constexpr int kPitch = gemm_pitch(KU), kXTile = TT * kPitch, kBuf = (TT + TM) * kPitch;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m0 = blockIdx.x * TM, t0 = blockIdx.y * TT;
    const int nsteps = k / (64 * KU);

    if (wave >= NC) {
        if (wave < NC + NA) {
            // ---- weights: units 2 H and 2 H + 1 of a step's four of 16 rows, as WideWeights above
            const uint32_t row_bytes = (uint32_t)(k >> 5) * kQ8Block;
            const int qi = lane & 3, r = (wave - NC) / 2 * 16 + (lane >> 2);
            const int row = m0 + r < m ? r : m - 1 - m0;
            auto weights = [&](auto half_) {
                constexpr int H = decltype(half_)::value;
                const uint8_t *const wb = w + (size_t)m0 * row_bytes;
                const uint32_t woff = (uint32_t)row * row_bytes + (uint32_t)(qi * 16 + H * 128);
                uint8_t *const wdst = lds + kXTile + r * kPitch + H * 256;
                uint4v rec[R][3];
                auto fetch = [&](int v, int s) {
                    const int c = s < nsteps ? s : nsteps - 1;
                    const uint8_t *const ws = wb + (size_t)(4 * c + (c >> 2)) * 64;
#pragma unroll
                    for (int j = 0; j < 3; j++)
                        rec[v][j] = *reinterpret_cast<const uint4v *>(ws + woff + j * 64);
                };
                auto stage = [&](int v, int s, int b) {
                    const int q = s & 3, li = (qi - q) & 3;
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        stage_unit(rec[v][u], rec[v][u + 1], 2 * H + u, qi, q, wdst + b * kBuf + li * 32 + u * 128);
                };
                produce_steps<R>(nsteps, fetch, stage);
            };
            if (wave & 1)
                weights(std::integral_constant<int, 1>{});
            else
                weights(std::integral_constant<int, 0>{});
        } else {
            // ---- activations: XN pieces of 16 bytes per thread
            constexpr int XELT = X16 ? 2 : 4, XPR = 64 * KU * XELT / 16, XROWS = 256 / XPR, XN = TT / XROWS;
            const int xt = threadIdx.x - 64 * (NC + NA), xr = xt / XPR, xc = xt % XPR;
            const uint8_t *const xb = static_cast<const uint8_t *>(xv) + (size_t)t0 * k * XELT;
            uint32_t xoff[XN];
#pragma unroll
            for (int i = 0; i < XN; i++) {
                const int t = t0 + xr + XROWS * i < tokens ? xr + XROWS * i : tokens - 1 - t0;
                xoff[i] = (uint32_t)t * (uint32_t)(k * XELT) + xc * 16;
            }
            uint8_t *const xdst = lds + xr * kPitch + xc * (X16 ? 16 : 8);
            float4v rec[R][XN];
            auto fetch = [&](int v, int s) {
                const uint8_t *const xs = xb + (size_t)(s < nsteps ? s : nsteps - 1) * (64 * KU * XELT);
#pragma unroll
                for (int i = 0; i < XN; i++)
                    rec[v][i] = *reinterpret_cast<const float4v *>(xs + xoff[i]);
            };
            auto stage = [&](int v, int, int b) {
#pragma unroll
                for (int i = 0; i < XN; i++) {
                    uint8_t *const d = xdst + b * kBuf + XROWS * i * kPitch;
                    if (X16)
                        *reinterpret_cast<float4v *>(d) = rec[v][i];
                    else // (rounded as the kernel above rounds)
                        *reinterpret_cast<half4v *>(d) = __builtin_convertvector(rec[v][i], half4v);
                }
            };
            produce_steps<R>(nsteps, fetch, stage);
        }
        return;
    }
    // consumer wave: 16 weight rows
    const int lm = lane & 15, lg = lane >> 4;
    float4v acc[AT];
#pragma unroll
    for (int a = 0; a < AT; a++)
        acc[a] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
    const uint8_t *xa = lds + lm * kPitch + lg * 16;
    const uint8_t *wb = lds + kXTile + (wave * 16 + lm) * kPitch + lg * 16;
    half8 A[2][AT], B[2];
    auto read = [&](int kk) {
#pragma unroll
        for (int a = 0; a < AT; a++)
            A[kk & 1][a] = *reinterpret_cast<const half8 *>(xa + a * 16 * kPitch + kk * 64);
        B[kk & 1] = *reinterpret_cast<const half8 *>(wb + kk * 64);
    };
    auto multiply = [&](int kk) {
#pragma unroll
        for (int a = 0; a < AT; a++)
            acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[kk & 1][a], B[kk & 1], acc[a], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int kSlices = 2 * KU; // of 32 values of k in a step: an even number
    __syncthreads();
    read(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int s = 0; s < nsteps; s++) {
#pragma unroll
        for (int kk = 0; kk + 1 < kSlices; kk++) {
            read(kk + 1);
            multiply(kk);
        }
        __syncthreads();
        const int other = s & 1 ? -kBuf : kBuf;
        xa += other;
        wb += other;
        read(0); // (behind the last step: whatever the other buffer holds, not used)
        multiply(kSlices - 1);
    }
    // C tile: lane holds column lm (weight row), rows 4 lg + j (tokens)
    const int row = m0 + wave * 16 + lm;
#pragma unroll
    for (int a = 0; a < AT; a++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int t = t0 + a * 16 + lg * 4 + j;
            if (t < tokens && row < m)
                y[(size_t)t * m + row] = acc[a][j];
        }
}

// ---- gemm_q8_direct_kernel: activations from L2 straight into operand registers -----------------------------------
//
// In the kernel above every activation passes through LDS once as it is staged and is read back by CM consumer waves: at
// 12288 x 5120 that, and the producers' loads behind it, cost as much as the MFMAs.  Here pack_f16_kernel has rounded the
// activations to f16 (after the gate, if any) and laid them out as the MFMA's operand: for each 32 values of k and 16
// tokens the 64 lanes' 16 bytes in a row.  A consumer wave loads its 16 AT tokens' operands from L2 with one request a
// KB, P slices of 32 k ahead, and no other wave of the workgroup reads them; only the weights, which every consumer wave
// needs, go through LDS, KU = 4 units a step, staged by NP producer waves (each half of a step's units of BT / (NP / 2) groups
// of 16 rows, SETS steps ahead).  Consumers: 16 AT tokens x 16 BT weight rows each, NC of them side by side in tokens.
// WB: slices of weight operands in registers, two, or one where the tile leaves no room for more (512 x 96).
// Loaded from the row-major rows instead it is slower than the kernel above: 16 rows 10,240 bytes apart lie in two of
// L2's channels.
// What bounds it (12288 x 5120 over 672 tokens, 384 x 96 tiles, timing-only builds): MFMAs and LDS reads alone 72 us, all
// of it 86, packing 5.  The kernel above with f32 rows before, this one with packing, us: 12288 x 5120 over 117 / 200 / 382 /
// 672 / 1,024 / 2,048 tokens 38.5 / 56.2 / 81.7 / 112 / 143 / 278 -> 32.8 / 44.6 / 58.2 / 94.0 / 121 / 233 (over 1,024 and
// 2,048 without the 512 x 96 tile 137 and 252); after a gate 5120 x 6144 over 200 / 382 / 672 / 1,024 / 1,500 41.4 / 47.5 /
// 66.8 / 91.9 / 123 -> 33.0 / 42.0 / 60.5 / 81.5 / 110; over f16 rows 5120 x 6144 over 200 / 382 / 512 / 1,024 / 1,500 37.2 /
// 41.8 / 59.0 / 81.3 / 109 -> 32.7 / 38.4 / 50.1 / 77.0 / 99.9.  Tried on it: weights by LDS DMA and dequantized by the
// consumers (behind the kernel above), weights loaded non-temporally (20 % slower), three or four steps of weights on the
// way (no gain), one slice of weight operands in the smaller tiles too (1 % slower), 384 x 128 (60 % slower).
// Layout of the packed activations: slice s (k from 32 s) starts at s * tokens * 64 bytes, its tokens from 16 t at t * 1024;
// there value k = 32 s + 8 g + e of token 16 t + i at (g * n + i) * 16 + 2 e, with n = 16, or what is left of the tokens.
// That is tokens * k * 2 bytes in all.

// One wave: 16 tokens x 128 values of k, each lane 8 values of 4 slices.
__global__ void __launch_bounds__(256) pack_f16_kernel(const float *__restrict__ x, const float *__restrict__ gate,
                                                       uint8_t *__restrict__ x16, int k, int tokens)
{
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * 16, n = tokens - t0 < 16 ? tokens - t0 : 16;
    const int s0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 4;
    if (i >= n)
        return;
    const size_t from = (size_t)(t0 + i) * k + g * 8;
    float4v a[4][2], ga[4][2];
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (s0 + u < k / 32)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                a[u][h] = *reinterpret_cast<const float4v *>(x + from + (s0 + u) * 32 + h * 4);
                if (gate != nullptr)
                    ga[u][h] = *reinterpret_cast<const float4v *>(gate + from + (s0 + u) * 32 + h * 4);
            }
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (s0 + u < k / 32) {
            half8 v;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float4v f = a[u][h];
                if (gate != nullptr)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        f[j] = gated(f[j], ga[u][h][j]);
                const half4v r = __builtin_convertvector(f, half4v); // (rounded as gate_f16_kernel rounds)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    v[4 * h + j] = r[j];
            }
            *reinterpret_cast<half8 *>(x16 + (size_t)(s0 + u) * tokens * 64 + (size_t)t0 * 64 + (g * n + i) * 16) = v;
        }
}

// The same of rows that are f16 already.
__global__ void __launch_bounds__(256) pack_rows_f16_kernel(const uint8_t *__restrict__ rows, uint8_t *__restrict__ x16, int k,
                                                            int tokens)
{
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * 16, n = tokens - t0 < 16 ? tokens - t0 : 16;
    const int s0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 4;
    if (i >= n)
        return;
    const uint8_t *const from = rows + (size_t)(t0 + i) * k * 2 + g * 16;
    half8 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (s0 + u < k / 32)
            v[u] = *reinterpret_cast<const half8 *>(from + (s0 + u) * 64);
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (s0 + u < k / 32)
            *reinterpret_cast<half8 *>(x16 + (size_t)(s0 + u) * tokens * 64 + (size_t)t0 * 64 + (g * n + i) * 16) = v[u];
}

template <int NC, int AT, int BT, int NP, int P, int SETS, int WB>
__global__ void __launch_bounds__(64 * (NP + NC)) gemm_q8_direct_kernel(const uint8_t *__restrict__ w,
                                                                        const void *__restrict__ xv,
                                                                        float *__restrict__ y, int m, int k, int tokens)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int KU = 4, TM = 16 * BT, TT = 16 * AT * NC;
    constexpr int kPitch = gemm_pitch(KU), kBuf = TM * kPitch;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m0 = blockIdx.x * TM, t0 = blockIdx.y * TT;
    const int nsteps = k / (64 * KU);

    if (wave >= NC) {
        const int pw = wave - NC;
        constexpr int G = BT / (NP / 2); // groups of 16 weight rows of a wave
        static_assert(G * (NP / 2) == BT && NP % 2 == 0, "");
        const uint32_t row_bytes = (uint32_t)(k >> 5) * kQ8Block;
        const uint8_t *const wb = w + (size_t)m0 * row_bytes;
        const int qi = lane & 3;
        auto produce = [&](auto half_) {
            constexpr int H = decltype(half_)::value; // units 2 H and 2 H + 1 of a step's four
            uint32_t woff[G], wlds[G];
#pragma unroll
            for (int g = 0; g < G; g++) {
                const int r = ((pw >> 1) * G + g) * 16 + (lane >> 2);
                const int row = m0 + r < m ? r : m - 1 - m0;
                woff[g] = (uint32_t)row * row_bytes + (uint32_t)(qi * 16 + H * 128);
                wlds[g] = (uint32_t)(r * kPitch + H * 256);
            }
            uint4v rec[SETS][G][3];
            auto fetch = [&](int v, int s) {
                const int c = s < nsteps ? s : nsteps - 1;
                const uint8_t *const ws = wb + (size_t)(4 * c + (c >> 2)) * 64;
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int j = 0; j < 3; j++)
                        rec[v][g][j] = *reinterpret_cast<const uint4v *>(ws + woff[g] + j * 64);
            };
            auto stage = [&](int v, int s, int b) {
                const int q = s & 3;
                uint8_t *const dst0 = lds + b * kBuf + ((qi - q) & 3) * 32;
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        stage_unit(rec[v][g][u], rec[v][g][u + 1], 2 * H + u, qi, q, dst0 + wlds[g] + u * 128);
            };
            produce_steps<SETS>(nsteps, fetch, stage);
        };
        if (pw & 1)
            produce(std::integral_constant<int, 1>{});
        else
            produce(std::integral_constant<int, 0>{});
        return;
    }
    const int lm = lane & 15, lg = lane >> 4;
    const int tw = t0 / 16 + wave * AT; // the wave's first 16 tokens
    float4v acc[AT][BT];
#pragma unroll
    for (int a = 0; a < AT; a++)
#pragma unroll
        for (int b = 0; b < BT; b++)
            acc[a][b] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t xoff[AT]; // (tokens past the last: the last one's)
#pragma unroll
    for (int a = 0; a < AT; a++) {
        const int last = (tokens - 1) >> 4, t = tw + a < last ? tw + a : last;
        const int n = tokens - 16 * t < 16 ? tokens - 16 * t : 16;
        xoff[a] = (uint32_t)(t * 64 + lg * n + (lm < n ? lm : n - 1)) * 16u;
    }
    const uint8_t *const xb = static_cast<const uint8_t *>(xv);
    const size_t xstep = (size_t)tokens * 64;
    const int nslice = k / 32;
    half8 X[P][AT], W[WB][BT];
    auto load = [&](int v, int s) {
        const uint8_t *const xs = xb + (size_t)(s < nslice ? s : nslice - 1) * xstep;
#pragma unroll
        for (int a = 0; a < AT; a++)
            X[v][a] = *reinterpret_cast<const half8 *>(xs + xoff[a]);
    };
    const uint8_t *wl = lds + lm * kPitch + lg * 16;
    auto read = [&](int kk) {
#pragma unroll
        for (int b = 0; b < BT; b++)
            W[kk % WB][b] = *reinterpret_cast<const half8 *>(wl + b * 16 * kPitch + kk * 64);
    };
    auto multiply = [&](int kk) { // (weights as the first operand: a lane's four sums are one token's)
#pragma unroll
        for (int b = 0; b < BT; b++)
#pragma unroll
            for (int a = 0; a < AT; a++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(W[kk % WB][b], X[kk % P][a], acc[a][b], 0, 0, 0);
    };
    constexpr int kSlices = 2 * KU;
    static_assert(kSlices % P == 0, "the records of a step are named at compile time");
#pragma unroll
    for (int v = 0; v < P; v++)
        load(v, v);
    __syncthreads();
    if constexpr (WB == 2) {
        read(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
        for (int s = 0; s < nsteps; s++) {
#pragma unroll
            for (int kk = 0; kk + 1 < kSlices; kk++) {
                read(kk + 1);
                multiply(kk);
                load(kk % P, s * kSlices + kk + P);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads(); // (behind the step's last reads, in front of its last products)
            wl += s & 1 ? -kBuf : kBuf;
            read(0); // (behind the last step: whatever the other buffer holds, not used)
            multiply(kSlices - 1);
            load((kSlices - 1) % P, s * kSlices + kSlices - 1 + P);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll 1
        for (int s = 0; s < nsteps; s++) {
#pragma unroll
            for (int kk = 0; kk < kSlices; kk++) {
                read(kk);
                multiply(kk);
                load(kk % P, s * kSlices + kk + P);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
            wl += s & 1 ? -kBuf : kBuf;
        }
    }
    // C tile: lane holds column lm (token), rows 4 lg + j (weight rows)
    const bool wide = (m & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
#pragma unroll
    for (int a = 0; a < AT; a++) {
        const int t = (tw + a) * 16 + lm;
        if (t < tokens) {
            float *const yt = y + (size_t)t * m;
#pragma unroll
            for (int b = 0; b < BT; b++) {
                const int row = m0 + 16 * b + 4 * lg;
                if (wide) {
                    if (row < m)
                        *reinterpret_cast<float4v *>(yt + row) = acc[a][b];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (row + j < m)
                            yt[row + j] = acc[a][b][j];
                }
            }
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
// (token rows and weight rows of the tile, 64-value units per step, sectors or quarters for the weights; microseconds
// per unit and round of the chip's 256 CUs where weight rows are whole sectors, over f32 and over f16 activations, and
// where they are not; 0: not for these.  Less 4 us per launch, with the slow-down of a full chip below taken out)
struct GemmTile {
    int tt, tm, ku;
    bool wide;
    float sectors, sectors16, other, other16;
};
constexpr GemmTile kGemmTiles[] = {
    {32, 32, 4, true, 0.101f, 0.086f, 0.0f, 0.0f},   {32, 64, 4, true, 0.145f, 0.119f, 0.0f, 0.0f},
    {64, 64, 2, true, 0.216f, 0.0f, 0.0f, 0.0f},     {64, 128, 2, true, 0.341f, 0.311f, 0.0f, 0.0f},
    {128, 128, 1, true, 0.504f, 0.0f, 0.0f, 0.0f},   {192, 128, 1, true, 0.729f, 0.585f, 0.0f, 0.0f},
    {128, 192, 1, true, 0.725f, 0.642f, 0.0f, 0.0f}, {192, 192, 1, true, 0.931f, 0.814f, 0.0f, 0.0f},
    {256, 192, 1, true, 0.0f, 0.972f, 0.0f, 0.0f},
    // quarters: the largest tile over f32 activations, whose registers do not hold sectors too; 128 x 128 over f16
    // activations, which they serve better; rows of weights that are not whole sectors
    {256, 192, 1, false, 1.171f, 0.0f, 1.35f, 1.152f}, {192, 192, 1, false, 0.0f, 0.0f, 1.054f, 0.902f},
    {128, 128, 1, false, 0.0f, 0.417f, 0.616f, 0.465f}, {64, 64, 2, false, 0.0f, 0.0f, 0.208f, 0.174f},
    {64, 64, 1, false, 0.0f, 0.0f, 0.229f, 0.184f},
    // cuts that fit 256 workgroups where those above do not (12,288 weight rows: 128 tiles of 96); over f16 activations
    // the 64 x 64 tile of longer steps stands for that of shorter ones
    {64, 96, 2, true, 0.291f, 0.0f, 0.0f, 0.0f},     {64, 64, 4, true, 0.0f, 0.18f, 0.0f, 0.0f},
    // gemm_q8_few_kernel, as tile 0: the costs of both and of tile 1 are fitted to these three and their neighbours at 468
    // shapes of 8 to 382 tokens (0.7 % behind the best of them on average; 16 shapes more than 5 %)
    {16, 32, 4, true, 0.074f, 0.06f, 0.0f, 0.0f},
};
constexpr int kGemmNTiles = sizeof(kGemmTiles) / sizeof(kGemmTiles[0]);

// Rounds of a tile over the chip's 256 CUs, a full one weighing 1 + slope.
static float tile_rounds(int m, int tokens, int tt, int tm, float slope)
{
    const long long wg = (long long)((m + tm - 1) / tm) * ((tokens + tt - 1) / tt);
    const long long rounds = (wg + 255) / 256;
    const float fill = (float)wg / (256.0f * (float)rounds);
    return (float)rounds * (1.0f + slope * fill * fill);
}

// The tile for a shape: the cheapest by rounds x cost, where a round of 256 workgroups slows down as it fills (they
// share L2, HBM and the power budget: 1.5 times the cost of a lone workgroup when all CUs have one).  The costs are fitted
// to every tile's time at 173 shapes (1,024 to 12,288 weight rows, k of 576 to 6,144, 24 to 2,048 tokens), 346 with the
// types of activations: the tile picked is the measured best or within 5 % of it at 340 of them, 14 % behind it at most
// (1024 x 5120 over 1,400 tokens: 42.4 us, best 37.1), 0.2 % on average.
static int gemm_tile(int m, int k, int tokens, bool sectors, bool x16, float *cost_of_unit)
{
    int best = -1;
    float best_cost = 0.0f;
    for (int i = 0; i < kGemmNTiles; i++) {
        const GemmTile &g = kGemmTiles[i];
        const float tile_cost = sectors ? (x16 ? g.sectors16 : g.sectors) : (x16 ? g.other16 : g.other);
        // (a tile's rows are addressed with 32-bit offsets)
        if (k % (64 * g.ku) != 0 || tile_cost == 0.0f ||
            (uint64_t)(g.tt > g.tm ? g.tt : g.tm) * (uint64_t)k * 4 >= (1ull << 32))
            continue;
        const float cost = tile_cost * tile_rounds(m, tokens, g.tt, g.tm, 0.5f);
        if (best < 0 || cost < best_cost) {
            best = i;
            best_cost = cost;
        }
    }
    if (cost_of_unit != nullptr)
        *cost_of_unit = best_cost;
    return best;
}

// For tests and the benchmark: the tile (its place in the table) that a call takes.
extern "C" int hipml_dbg_gemm_tile(int m, int k, int tokens, int sectors, int x16)
{
    return gemm_tile(m, k, tokens, sectors != 0, x16 != 0, nullptr);
}

// Calls f with the kernel of tile i and its launch figures: (kernel, threads, tile tokens, tile rows, LDS bytes).
template <bool X16, typename F>
static bool with_gemm_kernel(int i, F &&f)
{
#define HIPML_GEMM(idx, WIDE, CT, CM, AT, BT, KU, NW, R, ...)                                                          \
    case idx: {                                                                                                       \
        constexpr int tt = 32 * AT * CT, tm = 32 * BT * CM;                                                           \
        static_assert(kGemmTiles[idx].tt == tt && kGemmTiles[idx].tm == tm && kGemmTiles[idx].ku == KU &&             \
                          kGemmTiles[idx].wide == WIDE,                                                               \
                      "the table");                                                                                   \
        return f(&gemm_q8_f16_kernel<X16, WIDE, CT, CM, AT, BT, KU, NW, R __VA_OPT__(, ) __VA_ARGS__>,               \
                 64 * (NW + CT * CM), tt, tm,                                                                         \
                 gemm_lds(tt, tm, KU));                                                                               \
    }
#define HIPML_GEMM_FEW(idx, AT, R)                                                                                     \
    case idx:                                                                                                         \
        static_assert(kGemmTiles[idx].tt == 16 * AT && kGemmTiles[idx].tm == 32 && kGemmTiles[idx].ku == 4 &&         \
                          kGemmTiles[idx].wide,                                                                       \
                      "the table");                                                                                   \
        return f(&gemm_q8_few_kernel<X16, AT, R>, 640, 16 * AT, 32, gemm_lds(16 * AT, 32, 4));
    switch (i) {
        HIPML_GEMM_FEW(0, 2, 2)
        HIPML_GEMM_FEW(16, 1, 3)
        HIPML_GEMM(1, true, 1, 2, 1, 1, 4, 8, 2)
        HIPML_GEMM(3, true, 2, 2, 1, 2, 2, 8, 2)
        HIPML_GEMM(5, true, 2, 2, 3, 2, 1, 4, 2)
        HIPML_GEMM(6, true, 2, 2, 2, 3, 1, 4, 2)
        HIPML_GEMM(7, true, 2, 2, 3, 3, 1, 4, 2)
    case 8: // (f16 activations only)
    case 15:
        if constexpr (X16) {
            switch (i) {
                HIPML_GEMM(8, true, 2, 2, 4, 3, 1, 4, 2)
                HIPML_GEMM(15, true, 2, 2, 1, 1, 4, 8, 2)
            }
        }
        return false;
    case 2: // (f32 activations only)
    case 4:
    case 14:
        if constexpr (!X16) {
            switch (i) {
                HIPML_GEMM(2, true, 2, 2, 1, 1, 2, 8, 2)
                HIPML_GEMM(4, true, 2, 2, 2, 2, 1, 8, 2)
                HIPML_GEMM(14, true, 2, 1, 1, 3, 2, 8, 2)
            }
        }
        return false;
        HIPML_GEMM(9, false, 2, 2, 4, 3, 1, 4, 2)
        HIPML_GEMM(10, false, 2, 2, 3, 3, 1, 4, 2)
        HIPML_GEMM(11, false, 2, 2, 2, 2, 1, 8, 4, !X16)
        HIPML_GEMM(12, false, 2, 2, 1, 1, 2, 8, 2)
        HIPML_GEMM(13, false, 2, 2, 1, 1, 1, 4, 4)
    default:
        return false;
    }
#undef HIPML_GEMM
#undef HIPML_GEMM_FEW
}

// The packed route's tiles (tokens and weight rows; microseconds as in the table above, with a full chip's slow-down of 1.1
// instead of 1.5) and its kernels.
struct DirectTile {
    int tt, tm;
    float cost;
};
constexpr DirectTile kDirectTiles[] = {
    {128, 32, 0.21f}, {128, 48, 0.248f}, {128, 64, 0.281f},  {128, 96, 0.366f},  {192, 48, 0.298f}, {192, 96, 0.522f},
    {192, 128, 0.691f}, {256, 64, 0.476f}, {256, 96, 0.668f}, {256, 128, 0.807f}, {384, 96, 0.825f},
    {512, 96, 1.2f},
};
constexpr int kDirectNTiles = sizeof(kDirectTiles) / sizeof(kDirectTiles[0]);

template <typename F>
static bool with_direct_kernel(int i, F &&f)
{
#define HIPML_DIRECT(idx, NC, AT, BT, NP, P, WB)                                                                       \
    case idx: {                                                                                                       \
        constexpr int tt = 16 * AT * NC, tm = 16 * BT;                                                                \
        static_assert(kDirectTiles[idx].tt == tt && kDirectTiles[idx].tm == tm, "the table");                         \
        return f(&gemm_q8_direct_kernel<NC, AT, BT, NP, P, 2, WB>, 64 * (NP + NC), tt, tm, 2 * tm * gemm_pitch(4));       \
    }
    switch (i) {
        HIPML_DIRECT(0, 4, 2, 2, 4, 8, 2)
        HIPML_DIRECT(1, 4, 2, 3, 6, 8, 2)
        HIPML_DIRECT(2, 4, 2, 4, 4, 4, 2)
        HIPML_DIRECT(3, 4, 2, 6, 4, 4, 2)
        HIPML_DIRECT(4, 4, 3, 3, 6, 4, 2)
        HIPML_DIRECT(5, 4, 3, 6, 4, 4, 2)
        HIPML_DIRECT(6, 4, 3, 8, 4, 4, 2)
        HIPML_DIRECT(7, 4, 4, 4, 4, 4, 2)
        HIPML_DIRECT(8, 4, 4, 6, 4, 4, 2)
        HIPML_DIRECT(9, 4, 4, 8, 4, 2, 2)
        HIPML_DIRECT(10, 8, 3, 6, 4, 4, 2)
        HIPML_DIRECT(11, 8, 4, 6, 4, 2, 1)
    default:
        return false;
    }
#undef HIPML_DIRECT
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
    for (int i = 0; i < kDirectNTiles; i++)
        with_direct_kernel(i, raise);
    if (e != hipSuccess)
        return fail((int)e, "hipFuncSetAttribute(chunk projection LDS) failed: %d (%s)", (int)e, hipGetErrorString(e));
    return 0;
}

// How f32 rows are multiplied where the caller gives scratch for them as f16: as they lie (only without a gate), rounded
// into the scratch row by row, or packed into it for the direct kernel (weights in whole sectors only).  The cheapest by
// the tiles' costs and that of the pass that fills the scratch: 3 us (a launch 2, scratch from an allocator 1) and the
// rows read and written (3.4 M / 10.5 M values: 5.0 / 9.8 us in all, alone).  As they lie, too, below a k of 2,048, where
// the pass is not paid back (6000 x 1024 over 1,024 / 2,048 tokens: 24.3 / 39.3 us, with scratch 25.6 / 41.4).  The costs
// are fitted like the table above at 253 shapes (1,024 to 16,384 weight rows, 32 to 2,048 tokens): 1 % behind the best of
// all routes and tiles on average, 11 % at most; 12 % ahead of the tiles over the rows as they lie, at 3 shapes more than
// 2 % behind them.  (The 512 x 96 tile came later and has its cost from six shapes: at 68 others the rule is 0.6 % behind the
// best packed tile on average; it takes this tile at eight, where it is the best, and leaves it at two where it would be 4
// and 11 % faster.)
// Rows that are f16 already are multiplied as they lie or packed, by a pass of half the bytes.
enum class GemmRoute { kNone, kRows, kRowsF16, kPacked };
enum class GemmRows { kF32, kGated, kF16 };
struct GemmChoice {
    GemmRoute route;
    int tile;
};
static GemmChoice gemm_choice(int m, int k, int tokens, bool sectors, GemmRows rows)
{
    GemmChoice best = {GemmRoute::kNone, -1};
    float best_cost = 0.0f;
    auto offer = [&](GemmRoute route, int tile, float cost) {
        if (tile >= 0 && (best.tile < 0 || cost < best_cost)) {
            best = {route, tile};
            best_cost = cost;
        }
    };
    const float units = (float)(k / 64), values = (float)tokens * (float)k;
    const float pass = 3.0f + (rows == GemmRows::kF16 ? 0.4e-6f : 0.75e-6f) * values;
    float cost = 0.0f;
    if (rows == GemmRows::kF32) {
        const int tile = gemm_tile(m, k, tokens, sectors, false, &cost);
        offer(GemmRoute::kRows, tile, units * cost);
    }
    if (rows != GemmRows::kGated && k < 2048 && best.tile >= 0)
        return best;
    const int tile = gemm_tile(m, k, tokens, sectors, true, &cost);
    offer(GemmRoute::kRowsF16, tile, units * cost + (rows == GemmRows::kF16 ? 0.0f : pass));
    if (rows == GemmRows::kF16 && k < 2048)
        return best;
    // (32-bit offsets in a tile's weights and in a slice of the activations, and the passes' grids)
    if (sectors && tile >= 0 && k <= 1 << 23 && tokens <= 1 << 22)
        for (int i = 0; i < kDirectNTiles; i++) {
            const DirectTile &g = kDirectTiles[i];
            offer(GemmRoute::kPacked, i, units * g.cost * tile_rounds(m, tokens, g.tt, g.tm, 0.1f) + pass);
        }
    return best;
}

// For tests and the benchmark: 100 x route (1 as they lie, 2 f16 row by row, 3 packed) + tile of a call with scratch, over
// rows in f32 (0), in f32 with a gate (1), in f16 (2).
extern "C" int hipml_dbg_gemm_choice(int m, int k, int tokens, int sectors, int rows)
{
    const GemmChoice c = gemm_choice(m, k, tokens, sectors != 0, (GemmRows)rows);
    return c.tile < 0 ? -1 : 100 * (int)c.route + c.tile;
}

// Whether scratch makes the product over rows without a gate faster (W at a 64-byte boundary): over f32 rows scratch for
// them as f16, over f16 rows scratch to pack them into.
bool gemm_wants_scratch(int m, int k, int tokens, bool f16_rows)
{
    const GemmChoice c = gemm_choice(m, k, tokens, k % 1024 == 0, f16_rows ? GemmRows::kF16 : GemmRows::kF32);
    return c.tile >= 0 && c.route != (f16_rows ? GemmRoute::kRowsF16 : GemmRoute::kRows);
}

// f32 rows x (with a gate or without): x16 != nullptr is scratch for them as f16.  x == nullptr: x16 holds the rows as
// f16, row by row, and packed != nullptr is scratch to pack them into.
int launch_gemm_q8_f16(hipStream_t st, const uint8_t *w, const float *x, const float *gate, float *y, int m,
                       int k, int tokens, void *x16, void *packed)
{
    // (rows of weights in whole 64-byte sectors)
    const bool sectors = k % 1024 == 0 && (reinterpret_cast<uintptr_t>(w) & 63) == 0;
    const bool f16_rows = x == nullptr;
    GemmChoice c;
    if (f16_rows ? packed != nullptr : x16 != nullptr)
        c = gemm_choice(m, k, tokens, sectors, f16_rows ? GemmRows::kF16 : gate != nullptr ? GemmRows::kGated : GemmRows::kF32);
    else
        c = {f16_rows ? GemmRoute::kRowsF16 : GemmRoute::kRows, gemm_tile(m, k, tokens, sectors, f16_rows, nullptr)};
    if (c.tile < 0)
        return fail(HIPML_ATTN_E_RANGE, "k %d: 32 rows of activations exceed 4 GB", k);
    const void *act = c.route == GemmRoute::kRows ? static_cast<const void *>(x) : x16;
    int rc = 0;
    if (c.route == GemmRoute::kPacked) {
        const dim3 grid((unsigned)((tokens + 15) / 16), (unsigned)((k / 32 + 15) / 16), 1);
        if (f16_rows) {
            act = packed;
            HIPML_LAUNCH(pack_rows_f16_kernel, grid, dim3(256, 1, 1), 0, st, static_cast<const uint8_t *>(x16),
                         static_cast<uint8_t *>(packed), k, tokens);
        } else {
            HIPML_LAUNCH(pack_f16_kernel, grid, dim3(256, 1, 1), 0, st, x, gate, static_cast<uint8_t *>(x16), k, tokens);
        }
        rc = launched("pack_f16");
    } else if (c.route == GemmRoute::kRowsF16 && !f16_rows) {
        const size_t n8 = (size_t)tokens * k / 8;
        HIPML_LAUNCH(gate_f16_kernel, dim3((unsigned)((n8 + 255) / 256), 1, 1), dim3(256, 1, 1), 0, st,
                           reinterpret_cast<const float4v *>(x), reinterpret_cast<const float4v *>(gate),
                           static_cast<half8 *>(x16), n8);
        rc = launched("gate_f16");
    }
    if (rc)
        return rc;
    auto go = [&](auto kernel, int threads, int tt, int tm, int lds) {
        HIPML_LAUNCH(kernel, dim3((unsigned)((m + tm - 1) / tm), (unsigned)((tokens + tt - 1) / tt), 1),
                     dim3(threads, 1, 1), lds, st, w, act, y, m, k, tokens);
        return true;
    };
    if (c.route == GemmRoute::kPacked)
        with_direct_kernel(c.tile, go);
    else if (c.route == GemmRoute::kRowsF16)
        with_gemm_kernel<true>(c.tile, go);
    else
        with_gemm_kernel<false>(c.tile, go);
    return launched("gemm_q8_0_f16");
}

} // namespace hipml
