// Projections over Q8_0 weight matrices for gfx950 (wave64, MFMA): the step after the attention
// core (the output projection W_o) and, with other shapes, the one before it (W_q, W_k, W_v).
//
// W is [m][k/32] blocks of 34 bytes (f16 scale d, 32 int8), row-major; y[r][row] = sum_k W[row][k] x[r][k]
// (crates/hipml-core/src/quant.rs:653-675, crates/hipml-core/src/ops.rs:102-104,136-176).
//
// gemv_q8_rows_kernel: one or two activation rows over shapes gemv_q8_digits_kernel does not take, bound by streaming W
// once from HBM.
//   All MFMAs are v_mfma_f32_16x16x32_f16 with A = x (activation rows), B = W (16 weight rows),
//   one q8 block = one contraction, so the f16 block scale multiplies an exact integer dot product
//   in fp32: acc += d * (x . q), as the CPU definition's d*q products summed in fp32.
//   Fetch: a step is a pair of blocks of one weight row, 68 bytes at a dword boundary.  Lane 4*r + g
//   requests, with dword-aligned loads only, the 12 bytes that hold quarter g of the even block
//   (2 bytes in, realigned with alignbit) and the 8 of the odd block's quarter; the scales ride
//   along in lanes g = 0 and g = 3.  The four lanes of a quad read contiguous bytes.  (The MFMA's own
//   lane order, row = lane % 16, with 2-byte aligned 64-bit loads made every lane several requests
//   of its own: 9.5 M cache accesses per call and 1.0 TB/s.)  One ds_bpermute per register then
//   moves the data to the MFMA lane (row lm, quarter lg).  The C
//   tile puts weight row lm back in lane lm (rows of C are activation rows), where its scale is.
//   int8 -> f16 exactly: byte b^0x80 = b+128 under a high byte 0x64 is the f16 1024 + (b+128);
//   one packed f16 subtract of 1152 leaves b.  x enters as hi + lo f16 halves (two MFMAs, ~22 bits),
//   converted once per workgroup into LDS in operand order (whole rows: a pass is a few rows at most).
//   The waves of a workgroup split k; a wave requests the activations first, then two chunks of
//   its weight blocks (all of them for k = 6144) before it waits for anything, and the partial sums
//   meet in LDS in a fixed order (no atomics: the result does not depend on timing).
// gemv_q8_digits_kernel: one to eight rows; gemv_q8_units_kernel, gemv_q8_blocks_kernel: more (all further down).

#include "q8_weights.h"

#include <type_traits>

namespace hipml {

// 8 f32 -> hi and lo f16 halves with hi + lo = x to ~22 bits (up to 65,504; beyond, lo holds what it can, and from 131,008
// on the sum stays there).
__device__ __forceinline__ void split_hi_lo(const float4v &a, const float4v &b, half8 &hi, half8 &lo)
{
    uint4v h, l;
    float d[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float x0 = j < 2 ? a[2 * j] : b[2 * j - 4];
        const float x1 = j < 2 ? a[2 * j + 1] : b[2 * j - 3];
        h[j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x0, x1));
        // x - h (exact: h holds the leading bits of x) by the instruction that reads the f16 half in place: one per value
        // where the compiler makes a conversion and a subtraction
        asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d[2 * j]) : "v"(h[j]), "v"(x0));
        asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d[2 * j + 1]) : "v"(h[j]), "v"(x1));
    }
    // To f16, to nearest, with MODE bit 23 on: an overflow gives +-65,504 and not infinity (which a weight of 0 makes NaN).
    // For these conversions alone: under it an MFMA of infinities gives large finite numbers.  us over 5120 x 6144 and 24 /
    // 40 / 128 rows: 18.4 / 28.9 / 55.5; without the bit 18.3 / 28.0 / 53.4, the rounded difference by v_fma_mixlo_f16 and
    // v_fma_mixhi_f16 18.5 / 28.5 / 54.4, x clamped by v_med3_f32 first 19.3 / 30.7 / 58.4.
    asm("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 1\n\t"
        "v_cvt_pk_f16_f32 %0, %4, %5\n\t"
        "v_cvt_pk_f16_f32 %1, %6, %7\n\t"
        "v_cvt_pk_f16_f32 %2, %8, %9\n\t"
        "v_cvt_pk_f16_f32 %3, %10, %11\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 0"
        : "=&v"(l[0]), "=&v"(l[1]), "=&v"(l[2]), "=&v"(l[3])
        : "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "v"(d[4]), "v"(d[5]), "v"(d[6]), "v"(d[7]));
    hi = __builtin_bit_cast(half8, h);
    lo = __builtin_bit_cast(half8, l);
}

// One chunk of a wave's steps, as fetched.  A step is a pair of blocks of one weight row (68 bytes,
// dword aligned): the fetch lane of k quarter g holds bytes 8g..8g+11 of the pair (the even block's
// quarter sits 2 bytes in; g = 0 also catches the even scale, g = 3 the odd one) and the odd block's
// quarter, which is aligned.
template <int TILES, int CH>
struct GemvChunk {
    uint3a4 e[CH][TILES];
    uint2a4 o[CH][TILES];
};

constexpr int kGemvMaxRows = 2;        // activation rows per pass (their operands live in LDS)
constexpr int kGemvLdsBudget = 128 << 10;

// Activation rows per pass for a given k: as many (up to kGemvMaxRows) as keep the hi/lo operands of
// the whole rows, 4 bytes per element, inside the LDS budget; 0 = k too large.
__host__ __device__ inline int gemv_rows_per_pass(int k)
{
    const int fit = kGemvLdsBudget / (4 * k);
    return fit > kGemvMaxRows ? kGemvMaxRows : fit;
}
static_assert(kGemvLdsBudget / 4 / 8 / 512 <= 8, "a pass is staged in one round of at most 8 groups per thread");

// LDS: x operands [k/32 blocks][2*rp A rows: hi of rows 0..rp-1, then lo][4 quarters][8 x f16], then
// the partial sums [WAVES][TILES][32 lanes] float4.  The hi and the lo halves are different rows of
// ONE A operand: A rows 0..3 carry hi, rows 4..7 lo, so a block is one MFMA and the two partial
// products come out in lanes 0..15 (hi) and 16..31 (lo) of the C tile.
template <int WAVES, int TILES, int CH, int XG>
__global__ void __launch_bounds__(64 * WAVES, TILES == 1 ? 2 : 1) gemv_q8_rows_kernel(const uint8_t *__restrict__ w,
                                                                const float *__restrict__ x,
                                                                float *__restrict__ y, int m, int k,
                                                                int rows, int rp)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lm = lane & 15, lg = lane >> 4; // MFMA operand lane: weight row lm, k quarter lg
    const int fr = lane >> 2, fg = lane & 3;  // fetch lane: weight row fr, k quarter fg
    const int pull = (lm * 4 + lg) * 4;       // byte address of the fetch lane that holds this lane's operand
    const int nb = k >> 5;
    const size_t row_bytes = (size_t)nb * kQ8Block;
    const int m0 = blockIdx.x * (16 * TILES);
    const int r0 = blockIdx.y * rp;
    const int nrows = rows - r0 < rp ? rows - r0 : rp;
    const int nu = nb >> 1; // steps: pairs of blocks
    const int u_lo = (int)((long)wave * nu / WAVES), u_hi = (int)((long)(wave + 1) * nu / WAVES);
    float4v *red = reinterpret_cast<float4v *>(lds + (size_t)nb * rp * 128);
    const int per_row = k >> 3; // 8-element groups of one activation row

    // ---- 1. this thread's share of the activations, requested first (they are waited for first) --
    // group e = 8 consecutive k of one row; (row, e) pairs are dealt round-robin to the threads
    const int groups = nrows * (k >> 3);
    // XG groups in flight per thread and round; a thread with fewer left wraps around to groups that
    // are not its own (loaded, not stored) rather than all such threads asking for one address
    float4v xa[XG], xb[XG];
    auto x_issue = [&](int g0) {
#pragma unroll
        for (int i = 0; i < XG; i++) {
            int g = g0 + i * 64 * WAVES;
            g = g < groups ? g : g % groups;
            const float *p = x + (size_t)r0 * k + (size_t)g * 8; // rows are contiguous: group g of the pass

            xa[i] = *reinterpret_cast<const float4v *>(p);
            xb[i] = *reinterpret_cast<const float4v *>(p + 4);
        }
    };
    auto x_store = [&](int g0) {
#pragma unroll
        for (int i = 0; i < XG; i++) {
            const int g = g0 + i * 64 * WAVES;
            if (g < groups) {
                const int r = rp == 1 ? 0 : g / per_row, e = g - r * per_row;
                half8 hi, lo;
                split_hi_lo(xa[i], xb[i], hi, lo);
                uint8_t *blk = lds + (size_t)(e >> 2) * rp * 128 + (e & 3) * 16;
                *reinterpret_cast<half8 *>(blk + r * 64) = hi;
                *reinterpret_cast<half8 *>(blk + (rp + r) * 64) = lo;
            }
        }
    };
    x_issue(threadIdx.x);
    // every wave's activation requests enter the CU's memory pipeline before any wave's weight
    // requests: the pipeline serves them in order, and the first barrier below waits for the last
    // wave's activations
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);

    // ---- 2. the first two chunks of this wave's weight blocks ------------------------------------
    // rows past the end are clamped: they load (and compute) a duplicate that is never stored
    const uint8_t *wp[TILES];
#pragma unroll
    for (int t = 0; t < TILES; t++) {
        const int row = m0 + t * 16 + fr < m ? m0 + t * 16 + fr : m - 1;
        wp[t] = w + (size_t)row * row_bytes;
    }
    typedef GemvChunk<TILES, CH> Chunk;
    auto fetch = [&](Chunk &c, int u0) {
#pragma unroll
        for (int i = 0; i < CH; i++) {
            int uc = u0 + i < u_hi ? u0 + i : u_hi - 1;
            uc = uc < 0 ? 0 : uc;
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                const uint8_t *unit = wp[t] + (size_t)uc * (2 * kQ8Block);
                c.e[i][t] = *reinterpret_cast<const uint3a4 *>(unit + fg * 8);
                c.o[i][t] = *reinterpret_cast<const uint2a4 *>(unit + 36 + fg * 8);
            }
        }
    };
    Chunk A, B;
    fetch(A, u_lo);
    fetch(B, u_lo + CH);
    __builtin_amdgcn_sched_barrier(0);

    // ---- 3. activations to LDS as MFMA operands -----------------------------------------------
    x_store(threadIdx.x); // XG covers every group: the launcher sizes the pass for that
    __syncthreads();

    // ---- 4. the block steps --------------------------------------------------------------------
    float4v acc[TILES];
#pragma unroll
    for (int t = 0; t < TILES; t++)
        acc[t] = (float4v){0, 0, 0, 0};
    // A row lm: hi of activation row lm for lm < 4, lo of row lm - 4 for 4 <= lm < 8; the rest, and
    // rows past the live ones, repeat a valid slot (their products are never read)
    const int ar = (lm & 3) < nrows ? (lm & 3) : nrows - 1;
    const uint8_t *xop = lds + ((size_t)(((lm >> 2) & 1) * rp + ar) * 4 + lg) * 16;
    // One step = operands staged (realign, gather scales, move to the MFMA lanes, read x), then the
    // arithmetic; a step's staging is issued before the previous step's arithmetic so the LDS
    // round trips are covered, and the scheduler may not move anything across a step: a step waits
    // for its own two loads only.
    struct Staged {
        uint32_t q[TILES][4];
        uint32_t ds[TILES];
        half8 x0, x1;
    };
    auto stage = [&](Staged &s, const Chunk &c, int i, int u) {
        const int uc = u < u_hi ? u : u_hi - 1;
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            const uint3a4 e = c.e[i][t];
            // in the fetch lane: the even quarter realigned; both scales gathered in the quad's lane 0
            const int e2_of_g3 = __builtin_amdgcn_update_dpp(0, (int)e[2], 0xFF, 0xf, 0xf, true);
            const int sc = (int)((e[0] & 0xffffu) | ((uint32_t)e2_of_g3 & 0xffff0000u));
            s.q[t][0] = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)__builtin_amdgcn_alignbit(e[1], e[0], 16));
            s.q[t][1] = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)__builtin_amdgcn_alignbit(e[2], e[1], 16));
            s.q[t][2] = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)c.o[i][t][0]);
            s.q[t][3] = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)c.o[i][t][1]);
            s.ds[t] = (uint32_t)__builtin_amdgcn_ds_bpermute(lm * 16, sc);
        }
        s.x0 = *reinterpret_cast<const half8 *>(xop + (size_t)uc * rp * 256);
        s.x1 = *reinterpret_cast<const half8 *>(xop + (size_t)uc * rp * 256 + rp * 128);
    };
    auto math = [&](const Staged &s, int u) {
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            const float d0 = u < u_hi ? (float)__builtin_bit_cast(_Float16, (uint16_t)(s.ds[t] & 0xffffu)) : 0.0f;
            const float d1 = u < u_hi ? (float)__builtin_bit_cast(_Float16, (uint16_t)(s.ds[t] >> 16)) : 0.0f;
            const half8 w0 = int8x8_to_f16(s.q[t][0], s.q[t][1]), w1 = int8x8_to_f16(s.q[t][2], s.q[t][3]);
            float4v p0 = {0, 0, 0, 0}, p1 = {0, 0, 0, 0};
            p0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.x0, w0, p0, 0, 0, 0);
            p1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.x1, w1, p1, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[t][j] = fmaf(d1, p1[j], fmaf(d0, p0[j], acc[t][j]));
        }
    };
    auto compute = [&](const Chunk &c, int u0) {
        Staged s0, s1;
        stage(s0, c, 0, u0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < CH; i += 2) {
            if (i + 1 < CH)
                stage(s1, c, i + 1, u0 + i + 1);
            __builtin_amdgcn_sched_barrier(0);
            math(s0, u0 + i);
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < CH) {
                if (i + 2 < CH)
                    stage(s0, c, i + 2, u0 + i + 2);
                __builtin_amdgcn_sched_barrier(0);
                math(s1, u0 + i + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // The first two chunks (all of a wave's steps up to k = 64 * 2 * CH * WAVES) are straight-line
    // code, so each step waits for exactly its own loads while the rest are still in flight.
    // Longer rows continue in a loop that fetches and consumes two chunks per turn; nothing is
    // carried in registers from one turn to the next (carried chunks made the compiler copy them at
    // the loop head, behind a wait for every outstanding load).
    if (u_hi > u_lo) {
        compute(A, u_lo);
        compute(B, u_lo + CH);
        for (int u = u_lo + 2 * CH; u < u_hi; u += 2 * CH) {
            fetch(A, u);
            fetch(B, u + CH);
            compute(A, u);
            compute(B, u + CH);
        }
    }

    // ---- 5. the k slices meet in a fixed order: lanes 0..15 hold the hi products of activation
    // rows 0..3, lanes 16..31 the lo products ---------------------------------------------------
    if (lg < 2) {
#pragma unroll
        for (int t = 0; t < TILES; t++)
            red[(wave * TILES + t) * 32 + lane] = acc[t];
    }
    __syncthreads();
    if (threadIdx.x < 16 * TILES) {
        const int t = threadIdx.x >> 4, l = threadIdx.x & 15;
        float4v hi = red[t * 32 + l], lo = red[t * 32 + 16 + l];
#pragma unroll
        for (int u = 1; u < WAVES; u++) {
            hi += red[(u * TILES + t) * 32 + l];
            lo += red[(u * TILES + t) * 32 + 16 + l];
        }
        const float4v s = hi + lo;
        const int row = m0 + t * 16 + l;
        if (row < m) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j < nrows)
                    y[(size_t)(r0 + j) * m + row] = s[j];
        }
    }
}

// ---- gemv_q8_digits_kernel: one to eight activation rows, int8 matrix instructions over the weights as they are ----
//
// (a result) = sum over blocks of d * (sum of q x over the block).  The activations of a block become whole numbers: x =
// s X with s a power of two and |X| < 2^30, so that the block's largest value keeps all its 24 bits and every other one is
// cut at 2^-30 of it; X = X0 + 256 X1 + 65536 X2 + 2^24 X3 with digits in [-128, 127].  v_mfma_i32_16x16x64_i8 then
// multiplies the weight bytes as they lie in memory with the digits, exactly, and a block's four digit sums become one
// float.  Compared with f16 operands (x = hi + lo, the bytes made f16 numbers first) that is a third of the vector
// instructions for one row and half of them for four.
//
// B operand (weights): lane (lm, lg) holds 16 bytes of weight row lm, block lg of a group of four, so that a lane reads its
// whole block at once (9 dwords from the first dword boundary, realigned by v_perm_b32; the scale is among them).  A operand
// (activations): row 4 b + i is digit i of block b and holds zeros for the other three blocks, so that the contraction
// over the lanes lg keeps the blocks apart: C row 4 lg + j, digit j of block lg, meets in lane (lm, lg) the block's scale
// that this lane has read.  A lane's sum is thus one float for its weight row, its blocks and an activation row.
// Three and four activation rows fill the operand without zeros: v_mfma_i32_16x16x32_i8 over one block, A row 4 r + i digit
// i of row r, lane (lm, lg) holding 8 bytes of weight row lm and, in C, the digit sums of activation row lg; it adds the
// blocks 0 .. 3 of a group of four apart, as the lanes lg above do, so that a row's bits are the same.  Five to eight rows are
// two such operands over the same weight registers, or two passes of four (gemv_digits_cut): a wave makes the second set's
// digits in the place of the first's, whose operands it holds by then.
//
// A workgroup takes `ng` groups of GR weight rows (up to 16).  Wave v of V owns the runs v, v + V, ... of 512 values of k (544
// bytes of each row: with runs of 272 a pass over 12288 x 5120 reads 1 us slower) for all of them, makes the digits of its
// activations while its first weights travel, and then streams the groups' rows of its run through a place of its own by
// global_load_lds_dwordx4: a group's bytes move to registers, the next group is asked for, and the registers are
// multiplied.  Nothing is shared between the waves until their sums meet, so there is no barrier before that.
// A result is the sum over the waves in order, of which each adds its runs in order, blocks 0 .. 3 of a group of four apart
// and (0 + 2) + (1 + 3) behind them; V follows from k: the same operations in the same order whatever R is and whichever rows travel with it, so a
// verify group's rows have the bits of their plain decodes (crates/hipml-kernels/src/attn_gpu.rs:930-932).
constexpr int kChunkBytes = 8 * kQ8Block; // 272: a row's share of 256 values, which starts and ends at a 16-byte boundary
constexpr int kRunBytes = 2 * kChunkBytes;
constexpr int kDigitLds = 160 << 10;
constexpr int kDigitMaxWaves = 12;

typedef int int4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef uint32_t uint4a4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint32_t proj_lds_address(const void *p)
{
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

// 64 lanes x 16 bytes from base + voff (per lane) to LDS address lds_at + 16 * lane.  ONCE: non-temporal.
// gemv_q8_digits_kernel asks for its weights so (runs of 544 bytes of a row, read once; from HBM 12288 x 5120 over 1 / 3 rows
// 13.0 / 15.4 us with the hint, 13.8 / 15.7 without).  Where a request ends inside a cache line whose rest another one wants it
// costs a second fetch: gemv_q8_units_kernel over 1024 x 5120 and 24 rows 8.8 and 7.6, gemv_q8_blocks_kernel over 12288 x 5120
// and 9 / 16 rows 19.2 / 19.9 and 18.2 / 18.8.
// gemv_q8_blocks_kernel asks with it from 17 rows on, whatever the size of the matrix, and also where the workgroups of further
// activation rows, from 65 on, read the weights again.  To the call by itself it is a loss: us with / without over 12288 x 5120
// from HBM and 24 / 32 / 48 / 64 / 65 / 128 rows 22.2 / 24.5 / 31.6 / 34.4 / 57.0 / 67.8 and 21.7 / 23.6 / 31.5 / 35.4 / 53.2 / 65.0,
// with all weights in the last-level cache 24.1 / 26.5 / 33.7 / 36.6 / 59.3 / 70.7 and 22.9 / 23.8 / 28.1 / 34.6 / 49.8 / 64.5;
// 6400 x 1024 over 32 / 128 rows 6.7 / 17.3 and 6.7 / 15.5.  What it buys is that the weights do not push out of that cache what the
// next calls find there, which shows only while a few layers are all that runs: a layer over 32 short / 20 short / 24 deeper
// sequences, three layers in turn (333 MB of weights) 86.6 / 75.1 / 90.5 with and 89.5 / 77.9 / 94.8 without, sixteen, whose W_o
// comes from HBM either way, 90.7 / 78.9 / 93.4 and 89.2 / 77.8 / 93.0, one layer again and again 90.6 / 79.9 / 94.3 and 84.4 /
// 75.9 / 91.7.
template <bool ONCE>
__device__ __forceinline__ void proj_dma16(uint32_t lds_at, const uint8_t *base, uint32_t voff)
{
    if (ONCE)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                     :
                     : "s"(lds_at), "v"(voff), "s"(base)
                     : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(lds_at), "v"(voff), "s"(base)
                     : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// LDS of a wave: a group's rows of a run; the digits of its activations of the run, 2 KB a row of a set (eight rows are two
// sets of four, one after the other in the same place), beside one and two rows their scales, whose place takes the wave's
// sums when they are in registers, unless a wave has several runs; behind the waves 64 zero bytes.
constexpr int gemv_digit_set(int r) { return r > 4 ? 4 : r; }
constexpr int gemv_digit_x(int r) { return (r > 2 ? 2048 : 2048 + 64) * gemv_digit_set(r); }
constexpr int gemv_digit_wave(int r, int gr, int ng, bool more)
{
    const int sums = ng * r * 64, x = gemv_digit_x(r);
    return gr * kRunBytes + (more ? x + sums : (x > sums ? x : sums));
}
static_assert(kDigitMaxWaves * gemv_digit_wave(4, 4, 11, true) + 64 <= kDigitLds, "groups of four rows always fit");

// acc + ds * (p[0] + 2^8 p[1] + 2^16 p[2] + 2^24 p[3]); a digit sum is at most 2^19, so that both pairs are exact
__device__ __forceinline__ float add_digits(const int4v &p, float ds, float acc)
{
    const float lo = (float)(p[0] + p[1] * 256), hi = (float)(p[2] + p[3] * 256);
    return fmaf(fmaf(hi, 65536.0f, lo), ds, acc);
}

// s + the s of lane ^ 16, and of lane ^ 32
__device__ __forceinline__ float sum_lanes16(float s)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, s), __builtin_bit_cast(uint32_t, s), false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float sum_lanes32(float s)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, s), __builtin_bit_cast(uint32_t, s), false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

template <int R, int GR>
__global__ void __launch_bounds__(64 * kDigitMaxWaves) gemv_q8_digits_kernel(const uint8_t *__restrict__ w,
                                                                             const float *__restrict__ x,
                                                                             float *__restrict__ y, int m, int k, int rows,
                                                                             int ng)
{
    constexpr int kPerRow = kRunBytes / 16, kPieces = GR * kPerRow; // 16-byte pieces of a unit: a group's rows of a run
    constexpr int NI = (kPieces + 63) / 64;
    constexpr int S = gemv_digit_set(R), kSets = R / S; // activation rows of a set, and sets
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int waves = (int)(blockDim.x >> 6);
    const int lane = threadIdx.x & 63;
    const int lm = lane & 15, lg = lane >> 4;
    const int nchunk = k >> 8, nrun = (nchunk + 1) >> 1;
    const uint32_t row_bytes = (uint32_t)(k >> 5) * kQ8Block;
    const int m0 = blockIdx.x * (ng * GR);
    const int r0 = blockIdx.y * R;
    const int nrows = rows - r0 < R ? rows - r0 : R;
    const bool more = nrun > waves;
    const int area = gemv_digit_wave(R, GR, ng, more);
    uint8_t *const place = lds + wave * area;
    // one and two rows: [chunk][row][block][digit][32], then the scales [chunk][row][block]; more: [chunk][row][block][four
    // values][digit][4], a lane's own 16 bytes (one write without bank conflicts for four that took four times as long: 0.4 us
    // of a call over four rows), the scales by ds_bpermute
    uint8_t *const xdig = place + kPieces * 16;
    uint32_t *const scales = reinterpret_cast<uint32_t *>(xdig + 2048 * S);
    auto sums_of = [&](int v) { return reinterpret_cast<float *>(lds + v * area + kPieces * 16 + (more ? gemv_digit_x(R) : 0)); };
    uint8_t *const zeros = lds + waves * area;
    const uint32_t place_at = proj_lds_address(place), xdig_at = proj_lds_address(xdig);
    const uint8_t *const xb = reinterpret_cast<const uint8_t *>(x + (size_t)r0 * k);

    // ---- requests (a chunk past the end of k repeats the one before it: never used; rows past the live ones are not asked
    // for, and what is made of their places is not stored) ----
    auto issue_x = [&](int run, int set) {
#pragma unroll
        for (int cc = 0; cc < 2; cc++) {
            const int c = 2 * run + cc < nchunk ? 2 * run + cc : nchunk - 1;
#pragma unroll
            for (int r = 0; r < S; r++)
                if (set * S + r < nrows)
                    proj_dma16<false>(xdig_at + (cc * S + r) * 1024u, xb + (size_t)(set * S + r) * ((size_t)k * 4) + (size_t)c * 1024,
                                      lane * 16u);
        }
    };
    // piece p = 64 j + lane of a unit: row p / kPerRow of the group, 16 bytes p % kPerRow of its run
    uint32_t woff[NI];
#pragma unroll
    for (int j = 0; j < NI; j++) {
        const uint32_t p = (uint32_t)(j * 64 + lane), pr = p / (uint32_t)kPerRow;
        woff[j] = pr * row_bytes + (p - pr * kPerRow) * 16u;
    }
    const uint8_t *const w_last = w + (size_t)m * row_bytes - 16;
    auto issue_w = [&](int run, int g) {
        const int row = m0 + g * GR < m ? m0 + g * GR : m - 1;
        const uint8_t *const src = w + (size_t)row * row_bytes + (size_t)run * kRunBytes;
        // pieces past the matrix repeat its last one; a run cut short by the end of k goes on into the next row (never used)
        const size_t room = (size_t)(w_last - src);
        const uint32_t most = room < 0xfffffff0u ? (uint32_t)room : 0xfffffff0u;
#pragma unroll
        for (int j = 0; j < NI; j++)
            if ((j + 1) * 64 <= kPieces || j * 64 + lane < kPieces)
                proj_dma16<true>(place_at + j * 1024, src, woff[j] < most ? woff[j] : most);
    };
    if (wave < nrun) {
        issue_x(wave, 0);
        issue_w(wave, 0);
    }
    if (lane < 16) // (every wave writes the same zeros)
        reinterpret_cast<uint32_t *>(zeros)[lane] = 0;

    constexpr bool kDense = R > 2;
    // (not dense) lanes lg = 0 .. 3 take the blocks 0, 2, 1, 3 of a group of four: their first dwords then start in different
    // banks; payload dwords start 2 bytes into the first dword, or at the next; A row lm is a digit of the block of lanes
    // lm / 4.  (Rows past a group's repeat its last: never stored.)
    const uint32_t odd = (uint32_t)lg >> 1;
    const int blk = 2 * (lg & 1) + (int)odd;
    const uint32_t pick = odd ? 0x07060504u : 0x05040302u;
    const bool live = (lm >> 2) == lg;
    const uint8_t *const wrow = place + (lm < GR ? lm : GR - 1) * kRunBytes;
    const uint8_t *const wlane = kDense ? wrow + lg * 8 : wrow + blk * kQ8Block - 2 * (int)odd;
    const uint8_t *const xlane = kDense  ? xdig + ((lm >> 2) < S ? lm >> 2 : S - 1) * 1024 + (lm & 3) * 4 + lg * 32
                                 : live ? xdig + blk * 128 + (lm & 3) * 32
                                        : zeros;
    const int xstep = kDense || live ? 1 : 0;

    for (int run = wave; run < nrun; run += waves) {
        const bool two = 2 * run + 1 < nchunk; // (the last run may be one chunk)
        int4v a[kDense ? 1 : 2 * R][2][2];
        uint2v ad[kDense ? kSets : 1][2][8];
        float sx[kDense ? 2 : 2 * R][kDense ? 8 : 2];
        uint32_t pair[kSets][8]; // (dense) the scales of a block of either chunk, as the upper halves of their floats
#pragma unroll
        for (int set = 0; set < kSets; set++) {
            if (set > 0) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (the set before is in registers)
                issue_x(run, set);
            }
            if (run == wave && set == 0)
                wait_vm<NI>(); // (the first weights are still travelling)
            else
                wait_vm<0>();
            // ---- digits, in place: four values a lane, eight lanes a block ------------------------------------------
            float4v f[2 * S];
#pragma unroll
            for (int e = 0; e < 2 * S; e++)
                f[e] = *reinterpret_cast<const float4v *>(xdig + e * 1024 + lane * 16);
            asm volatile("" ::: "memory"); // (one wave: every lane has read before any writes)
            __builtin_amdgcn_wave_barrier();
            uint32_t scale_of[2] = {0, 0}; // (dense) of block lane / 8 and row lane % 8
#pragma unroll
            for (int e = 0; e < 2 * S; e++) {
                if (kDense && set * S + e % S >= nrows)
                    continue;
                uint32_t b[4];
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    v[i] = f[e][i]; // (__builtin_bit_cast of a vector's element itself takes element 0)
                    b[i] = __builtin_bit_cast(uint32_t, v[i]) & 0x7fffffffu;
                }
                // the block's largest magnitude, as bits (infinities and NaN above all numbers)
                uint32_t top = b[0] > b[1] ? b[0] : b[1];
                top = top > b[2] ? top : b[2];
                top = top > b[3] ? top : b[3];
                uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0xB1, 0xf, 0xf, true); // lane ^ 1
                top = o > top ? o : top;
                o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x4E, 0xf, 0xf, true); // lane ^ 2
                top = o > top ? o : top;
                o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x141, 0xf, 0xf, true); // lane 7 - i of eight
                top = o > top ? o : top;
                const uint32_t most = 0x47ffe000u; // 131,008: beyond it activations count as that much
                uint32_t bad = 0;
                if (__builtin_amdgcn_ballot_w64(top > most) != 0) { // (in no block of the wave, as a rule)
                    bad = top >= 0x7f800000u ? 0x7fc00000u : 0u;
                    top = top < most ? top : most;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        v[i] = __builtin_amdgcn_fmed3f(v[i], -131008.0f, 131008.0f);
                }
                uint32_t ex = top & 0x7f800000u; // |x| < 2^(ex - 126)
                ex = ex > (30u << 23) ? ex : 30u << 23;
                const float up = __builtin_bit_cast(float, (283u << 23) - ex); // 2^(156 - ex)
                uint32_t z[4];
#pragma unroll
                for (int i = 0; i < 4; i++) // X + 0x808080: the three low digits, each 128 up, and the fourth
                    z[i] = (uint32_t)(int)fmaf(v[i], up, 8421504.0f);
                const uint32_t p0 = __builtin_amdgcn_perm(z[1], z[0], 0x05010400u), p1 = __builtin_amdgcn_perm(z[3], z[2], 0x05010400u);
                const uint32_t p2 = __builtin_amdgcn_perm(z[1], z[0], 0x07030602u), p3 = __builtin_amdgcn_perm(z[3], z[2], 0x07030602u);
                const uint4v digit = {__builtin_amdgcn_perm(p1, p0, 0x05040100u) ^ 0x80808080u,
                                      __builtin_amdgcn_perm(p1, p0, 0x07060302u) ^ 0x80808080u,
                                      __builtin_amdgcn_perm(p3, p2, 0x05040100u) ^ 0x80808080u,
                                      __builtin_amdgcn_perm(p3, p2, 0x07060302u)}; // each of four values
                if (kDense) {
                    *reinterpret_cast<uint4v *>(xdig + e * 1024 + lane * 16) = digit;
                } else {
                    uint32_t *const dst = reinterpret_cast<uint32_t *>(xdig + e * 1024 + (lane >> 3) * 128 + (lane & 7) * 4);
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        dst[8 * i] = digit[i];
                }
                const uint32_t scale = (ex - (29u << 23)) | bad; // 2^(ex - 156), or NaN
                if (kDense)
                    scale_of[e / S] = (lane & 7) == e % S ? scale : scale_of[e / S];
                else if ((lane & 7) == 0)
                    scales[e * 8 + (lane >> 3)] = scale;
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            if constexpr (kDense) {
                const uint32_t both = __builtin_amdgcn_perm(scale_of[1], scale_of[0], 0x07060302u);
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    pair[set][q] = (uint32_t)__builtin_amdgcn_ds_bpermute(q * 32 + lg * 4, (int)both); // of row lg
#pragma unroll
                    for (int cc = 0; cc < 2; cc++) {
                        const uint32_t *const src = reinterpret_cast<const uint32_t *>(xlane + cc * (S * 1024) + q * 128);
                        ad[set][cc][q] = (uint2v){src[0], src[4]};
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 2 * R; e++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
#pragma unroll
                        for (int j = 0; j < 2; j++)
                            a[e][h][j] = *reinterpret_cast<const int4v *>(xlane + (e * 1024 + h * 512) * xstep + j * 16);
                        sx[e][h] = __builtin_bit_cast(float, scales[e * 8 + h * 4 + blk]);
                    }
            }
        }
        auto scale_at = [&](int set, int cc, int q) {
            return __builtin_bit_cast(float, cc == 0 ? pair[set][q] << 16 : pair[set][q] & 0xffff0000u);
        };
        if constexpr (kDense && kSets == 1) { // (two sets have no registers for them)
#pragma unroll
            for (int cc = 0; cc < 2; cc++)
#pragma unroll
                for (int q = 0; q < 8; q++)
                    sx[cc][q] = scale_at(0, cc, q);
        }
        // ---- the groups ---------------------------------------------------------------------------------------------
#pragma unroll 1
        for (int g = 0; g < ng; g++) {
            wait_vm<0>();
            auto ask = [&]() { // the unit, and the activations before it, are in registers
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (g + 1 < ng) {
                    issue_w(run, g + 1);
                } else if (run + waves < nrun) {
                    int next = run + waves;
                    asm volatile("" : "+s"(next)); // (or its addresses are made ahead of the loop and held through it)
                    issue_x(next, 0);
                    issue_w(next, 0);
                }
            };
            if constexpr (kDense) {
                float acc[kSets][4] = {}; // blocks 0 .. 3 of a group of four
                if constexpr (kSets > 1) { // (or they are taken apart ahead of the loop, into 32 registers)
#pragma unroll
                    for (int e = 0; e < 8 * kSets; e++)
                        asm volatile("" : "+v"(pair[e >> 3][e & 7]));
                }
#pragma unroll
                for (int cc = 0; cc < 2; cc++) {
                    uint32_t q0[8], q1[8], q2[4];
                    _Float16 dh[8];
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        const uint8_t *const src = wlane + cc * kChunkBytes + q * kQ8Block;
                        if ((q & 1) == 0) { // (the lane's 8 bytes start 2 bytes past a dword boundary)
                            const uint3a4 v = *reinterpret_cast<const uint3a4 *>(src);
                            q0[q] = v[0];
                            q1[q] = v[1];
                            q2[q >> 1] = v[2];
                        } else {
                            const uint2a4 v = *reinterpret_cast<const uint2a4 *>(src + 2);
                            q0[q] = v[0];
                            q1[q] = v[1];
                        }
                        dh[q] = *reinterpret_cast<const _Float16 *>(wrow + cc * kChunkBytes + q * kQ8Block);
                    }
                    if (cc == 1) {
                        ask();
                        if (!two)
                            break;
                    }
                    int4v p[8][kSets];
                    auto multiply = [&](int q) {
                        uint2v v = {q0[q], q1[q]};
                        if ((q & 1) == 0) {
                            v[0] = __builtin_amdgcn_alignbit(q1[q], q0[q], 16);
                            v[1] = __builtin_amdgcn_alignbit(q2[q >> 1], q1[q], 16);
                        }
                        if (kSets > 1)
                            asm volatile("" : "+v"(v));
#pragma unroll
                        for (int set = 0; set < kSets; set++) {
                            p[q][set] = (int4v){0, 0, 0, 0};
                            p[q][set] = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, ad[set][cc][q]),
                                                                              __builtin_bit_cast(long, v), p[q][set], 0, 0, 0);
                        }
                    };
                    auto add = [&](int q) {
#pragma unroll
                        for (int set = 0; set < kSets; set++) {
                            const float of = kSets == 1 ? sx[cc][q] : scale_at(set, cc, q);
                            float &to = acc[set][q & 3];
                            to = add_digits(p[q][set], (float)dh[q] * of, to);
                            if (kSets > 1)
                                asm volatile("" : "+v"(to));
                        }
                    };
                    // (two sets: the empty statements keep the products of three blocks in registers at a time; the compiler
                    // puts all of a chunk's matrix instructions first)
                    multiply(0);
                    multiply(1);
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        if (q + 2 < 8)
                            multiply(q + 2);
                        add(q);
                    }
                }
#pragma unroll
                for (int set = 0; set < kSets; set++) {
                    const float s = (acc[set][0] + acc[set][2]) + (acc[set][1] + acc[set][3]);
                    float *const to = sums_of(wave) + (g * R + set * S + lg) * 16 + lm;
                    if (lg < S)
                        *to = run == wave ? s : *to + s;
                }
            } else {
                float acc[R];
#pragma unroll
                for (int r = 0; r < R; r++)
                    acc[r] = 0.0f;
#pragma unroll
                for (int cc = 0; cc < 2; cc++) {
                    uint4v d0[2], d1[2];
                    uint32_t d2[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const uint8_t *const src = wlane + cc * kChunkBytes + h * (4 * kQ8Block);
                        d0[h] = *reinterpret_cast<const uint4a4 *>(src);
                        d1[h] = *reinterpret_cast<const uint4a4 *>(src + 16);
                        d2[h] = *reinterpret_cast<const uint32_t *>(src + 32);
                    }
                    if (cc == 1) {
                        ask();
                        if (!two)
                            break;
                    }
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const uint4v u0 = d0[h], u1 = d1[h];
                        int4v w0, w1;
                        w0[0] = (int)__builtin_amdgcn_perm(u0[1], u0[0], pick);
                        w0[1] = (int)__builtin_amdgcn_perm(u0[2], u0[1], pick);
                        w0[2] = (int)__builtin_amdgcn_perm(u0[3], u0[2], pick);
                        w0[3] = (int)__builtin_amdgcn_perm(u1[0], u0[3], pick);
                        w1[0] = (int)__builtin_amdgcn_perm(u1[1], u1[0], pick);
                        w1[1] = (int)__builtin_amdgcn_perm(u1[2], u1[1], pick);
                        w1[2] = (int)__builtin_amdgcn_perm(u1[3], u1[2], pick);
                        w1[3] = (int)__builtin_amdgcn_perm(d2[h], u1[3], pick);
                        const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(u0[0] >> (odd * 16)));
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            const int e = cc * R + r;
                            int4v p = {0, 0, 0, 0};
                            p = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[e][h][0], w0, p, 0, 0, 0);
                            p = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[e][h][1], w1, p, 0, 0, 0);
                            acc[r] = add_digits(p, d * sx[e][h], acc[r]);
                        }
                    }
                }
                // the lane's four fellows of a weight row: blocks (0 + 2) + (1 + 3)
#pragma unroll
                for (int r = 0; r < R; r++) {
                    float s = acc[r];
                    s = sum_lanes16(s);
                    s = sum_lanes32(s);
                    float *const to = sums_of(wave) + (g * R + r) * 16 + lm;
                    if (lg == 0)
                        *to = run == wave ? s : *to + s;
                }
            }
        }
    }
    __syncthreads();
    const int used = nrun < waves ? nrun : waves;
    for (int e = threadIdx.x; e < ng * R * 16; e += 64 * waves) {
        const int wr = e & 15, e4 = e >> 4, g = e4 / R, r = e4 - g * R;
        float s = sums_of(0)[e];
        for (int v = 1; v < used; v++)
            s += sums_of(v)[e];
        const int row = m0 + g * GR + wr;
        if (wr < GR && row < m && r < nrows)
            y[(size_t)(r0 + r) * m + row] = s;
    }
}

// ---- 9 to 128 activation rows (verify groups, batched decode): two kernels ---------------------------------------
//
// More rows than the kernel above holds operands for.  In both, a workgroup takes RW weight rows and XT tiles of 16
// activation rows; weights and f32 activations travel by global_load_lds as they lie in memory, into a ring, and from
// there to registers while what came before them is multiplied.  A lane (row lm, quarter lg) splits its 8 floats of a
// tile and block into hi and lo halves; a block and pair of tiles is two chained MFMAs (hi, then lo into the same fp32
// sums), the weights exactly as f16 integers (1024 + u trick), the block scale applied to the fp32 dot product.  The
// 16-byte pieces of an activation row lie in LDS at piece ^ row, so that the rows of a tile start in different banks
// without padding.  A result is a sum over eight chains of blocks in fixed order: its bits depend on the shape of W
// (which picks the kernel), not on the number of rows, tiles and weight rows per workgroup.
//
// What bounds them: vector instructions (bytes to f16, hi / lo split, scaling of block products: a single wave issues
// one per 8 cycles, so a SIMD needs two), requests (~16 cycles of a CU each, whatever their size), and ~4 us of launch,
// first data and final sum.
//
// gemv_q8_units_kernel (m up to 6,144; any k of whole 64-value units, W at a 4-byte boundary): no barrier, a wave
// streams units of its own.  gemv_q8_blocks_kernel (more rows, k of whole 256-value chunks, W at a 16-byte boundary):
// the workgroup walks chunks together and shares its requests for the weights.  us over 9 / 16 / 24 / 32 / 40 / 48 / 64 / 128
// rows, units (by 16-byte requests) and blocks, each with its best tile, the weights from HBM (k 5120, for 2,048 and 4,096
// weight rows 4096, for 5,120 6144):
//    1,024 weight rows  6.8 13.1 |  7.5 13.4 |  7.4 13.2 |  7.3 13.3 |  8.8 13.3 |  9.6 13.4 |  9.5 13.5 | 11.9 13.5
//    2,048              6.2 11.3 |  6.6 11.3 |  7.6 11.4 |  8.4 11.4 |  9.9 11.4 | 10.7 11.5 | 10.5 11.8 | 13.8 15.0
//    4,096              7.9 11.4 |  9.2 11.6 | 11.4 12.0 | 11.2 11.8 | 13.2 14.5 | 13.6 14.7 | 14.7 15.1 | 26.4 24.8
//    5,120              12.9 15.8 | 14.3 16.2 | 18.0 19.5 | 19.6 19.0 | 22.6 22.3 | 23.2 22.8 | 25.7 24.9 | 45.8 38.5
//    6,144              12.3 13.7 | 13.6 14.4 | 16.8 16.8 | 16.9 16.7 | 19.8 21.3 | 20.4 21.3 | 22.9 22.0 | 41.2 33.8
//    7,168              15.3 14.0 | 15.8 15.0 | 18.4 17.5 | 20.8 18.7 | 29.2 23.2 | 29.8 27.5 | 34.2 31.1 | 59.5 52.1
//    8,192              15.7 15.7 | 16.4 15.4 | 19.2 17.9 | 21.2 19.1 | 30.5 23.5 | 31.4 27.9 | 35.6 31.5 | 61.0 56.1
//   12,288              20.9 19.7 | 21.1 19.4 | 24.3 22.2 | 27.4 24.7 | 39.6 28.2 | 40.9 32.1 | 46.0 36.0 | 83.8 64.8
// What a workgroup asks for adds up, wherever it comes from: a CU takes 36 bytes a cycle out of L2 however many CUs ask and
// whatever the pattern, and what comes from HBM waits in the same queue.  12288 x 5120 over 32 rows: weights alone 12 us,
// activations (every workgroup reads all of them) 8 more.
// The choice must not depend on the number of rows (their bits would), so the line lies where the row counts of verify
// groups and batched decode, 9 to 40, change sides; over more rows the blocks would win from 5,120 weight rows on.

template <int XT, int RW, bool HALF>
struct BlocksShape {
    static constexpr int kMT = (RW + 15) / 16;              // weight tiles
    static constexpr int kXRows = 16 * XT - (HALF ? 8 : 0); // activation rows that are fetched
    static constexpr int kWBytes = RW * kChunkBytes;
    static constexpr int kXWave = kXRows * 128;             // one wave's block of them
    static constexpr int kSlot = kWBytes + 8 * kXWave;
    static constexpr int kFit = (160 << 10) / kSlot;
    // Chunks on the way, at most three: 12288 x 5120 over 9 / 16 rows with five / three / two 19.4 / 18.2 / 20.9 and 20.1 / 18.8 /
    // 22.0 us, over 24 / 32 with three / two 22.1 / 24.2 and 23.8 / 27.8, from HBM; 8192 x 5120 over 16 with five / three 16.8 /
    // 15.6 from the last-level cache.
    static constexpr int kMost = 3;
    static constexpr int kDepth = kFit < kMost ? kFit : kMost; // chunks on the way
    static constexpr int kSums = 8 * XT * kMT * 1024;
    static constexpr int kRead = HALF ? 1024 : 0; // (a HALF tile's dead rows are read past the wave's block)
    static constexpr int kLds = (kDepth * kSlot > kSums ? kDepth * kSlot : kSums) + kRead;
    static_assert(kDepth >= 2 && kLds <= 160 << 10, "");
};

// Wave w multiplies block w of a chunk of 256 values.  One barrier per chunk: behind it chunk c + 1 has arrived for
// everybody, and everybody has moved chunk c to registers, so that its place is asked for anew at once.  HALF: the last
// tile has at most 8 live rows; the other 8 are never fetched, hold whatever the LDS held, and are never stored.
template <int XT, int RW, bool HALF>
__global__ void __launch_bounds__(512, 2) gemv_q8_blocks_kernel(const uint8_t *__restrict__ w,
                                                                const float *__restrict__ x, float *__restrict__ y,
                                                                int m, int k, int rows)
{
    typedef BlocksShape<XT, RW, HALF> S;
    constexpr int MT = S::kMT, D = S::kDepth;
    constexpr int NX = S::kXRows / 8;                     // activation requests per chunk and wave: eight rows each
    constexpr int NW = (RW * 17 + 63) / 64;               // weight requests per chunk
    constexpr int NWMost = (NW + 7) / 8;                  // of a wave, or one less
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int lm = lane & 15, lg = lane >> 4;
    const int nb = k >> 5, nchunk = nb >> 3;
    const uint32_t row_bytes = (uint32_t)nb * kQ8Block;
    const int m0 = blockIdx.x * RW, r0 = blockIdx.y * (16 * XT);
    const int nrows = rows - r0 < 16 * XT ? rows - r0 : 16 * XT;
    const uint32_t ring_at = proj_lds_address(lds);
    const uint8_t *wb = w + (size_t)m0 * row_bytes;
    const uint8_t *xb = reinterpret_cast<const uint8_t *>(x + (size_t)r0 * k);

    // piece p of a chunk of weights: row p / 17, 16 bytes p % 17 of its 272; rows past the matrix repeat the last
    constexpr int kPieces = RW * 17;
    uint32_t woff[NWMost], xoff[NX];
    int wreq = 0;
#pragma unroll
    for (int j = 0; j < NWMost; j++) {
        const int p = (wave + 8 * j) * 64 + lane;
        const int pr = p / 17, pq = p - pr * 17;
        woff[j] = (uint32_t)(m0 + pr < m ? pr : m - 1 - m0) * row_bytes + (uint32_t)pq * 16u;
        wreq += wave + 8 * j < NW ? 1 : 0;
    }
#pragma unroll
    for (int j = 0; j < NX; j++) { // rows past the live ones repeat the last
        const int r = 8 * j + (lane >> 3);
        xoff[j] = (uint32_t)(r < nrows ? r : nrows - 1) * (uint32_t)k * 4u + (uint32_t)(((lane ^ r) & 7) * 16);
    }
    auto issue = [&](int c) {
        const uint32_t at = ring_at + (uint32_t)((c % D) * S::kSlot);
        const uint8_t *xs = xb + (size_t)(8 * c + wave) * 128;
#pragma unroll
        for (int j = 0; j < NX; j++)
            proj_dma16<false>(at + S::kWBytes + wave * S::kXWave + j * 1024, xs, xoff[j]);
#pragma unroll
        for (int j = 0; j < NWMost; j++) {
            const int q = wave + 8 * j;
            if (q < NW && (kPieces % 64 == 0 || q * 64 + lane < kPieces))
                proj_dma16<(XT > 1)>(at + q * 1024, wb, woff[j] + (uint32_t)c * kChunkBytes);
        }
    };
    // chunk c has arrived: only the chunks asked for behind it, `most` of them, are outstanding
    auto wait_chunk = [&](int c, int most) {
        const int newer = nchunk - 1 - c < most ? nchunk - 1 - c : most;
        constexpr int a = NX + NWMost, b = NX + NWMost - 1; // requests of a chunk
        static_assert(2 * a < 64 && S::kMost <= 3, "vmcnt has six bits");
        switch (newer) {
        case 2: return wreq == NWMost ? wait_vm<2 * a>() : wait_vm<2 * b>();
        case 1: return wreq == NWMost ? wait_vm<a>() : wait_vm<b>();
        default: return wait_vm<0>();
        }
    };

    struct Regs {
        float4v x[XT][2];
        uint32_t q[MT][3];
        uint16_t d[MT];
    };
    // block w: the lane's 8 bytes sit 2 bytes past a dword boundary in even blocks (three dwords, realigned below) and
    // at one in odd blocks; rows of the last tile past RW repeat the last (never stored)
    const uint32_t shift = wave & 1 ? 0 : 16;
    int wrow[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
        wrow[t] = (t * 16 + lm < RW ? t * 16 + lm : RW - 1) * kChunkBytes + wave * kQ8Block;
    auto load = [&](Regs &g, int c) {
        const uint8_t *buf = lds + (c % D) * S::kSlot;
        const uint8_t *xa = buf + S::kWBytes + wave * S::kXWave + lm * 128;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const uint8_t *blk = buf + wrow[t];
            const uint32_t *q = reinterpret_cast<const uint32_t *>(blk + (wave & 1) * 2 + lg * 8);
#pragma unroll
            for (int j = 0; j < 3; j++)
                g.q[t][j] = q[j];
            g.d[t] = *reinterpret_cast<const uint16_t *>(blk);
        }
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                g.x[xt][h] = *reinterpret_cast<const float4v *>(xa + xt * 2048 + (((lg * 2 + h) ^ lm) & 7) * 16);
    };
    float4v acc[XT][MT];
#pragma unroll
    for (int xt = 0; xt < XT; xt++)
#pragma unroll
        for (int t = 0; t < MT; t++)
            acc[xt][t] = (float4v){0, 0, 0, 0};
    auto multiply = [&](const Regs &g) {
        half8 wv[MT], hi[XT], lo[XT];
        float d[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            wv[t] = int8x8_to_f16(__builtin_amdgcn_alignbit(g.q[t][1], g.q[t][0], shift),
                                  __builtin_amdgcn_alignbit(g.q[t][2], g.q[t][1], shift));
            d[t] = (float)__builtin_bit_cast(_Float16, g.d[t]);
        }
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
            split_hi_lo(g.x[xt][0], g.x[xt][1], hi[xt], lo[xt]);
        float4v p[XT][MT];
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                p[xt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[xt], wv[t], (float4v){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                p[xt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[xt], wv[t], p[xt][t], 0, 0, 0);
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[xt][t][j] = fmaf(d[t], p[xt][t][j], acc[xt][t][j]);
    };
#pragma unroll
    for (int c = 0; c < D; c++)
        if (c < nchunk)
            issue(c);
    Regs even, odd;
    wait_chunk(0, D - 1);
    __syncthreads();
    load(even, 0);
    // chunk c is in `now`
    auto turn = [&](Regs &now, Regs &next, int c) {
        // (lgkmcnt(0), through the builtin: the compiler then knows that `now` is there and does not hold up its use for
        // the reads of `next`, of which there are more than lgkmcnt can count)
        __builtin_amdgcn_s_waitcnt(0xc07f);
        if (c + 1 < nchunk)
            wait_chunk(c + 1, D - 2);
        __syncthreads();
        if (c + D < nchunk)
            issue(c + D);
        if (c + 1 < nchunk)
            load(next, c + 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(now);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int c = 0; c < nchunk; c += 2) {
        turn(even, odd, c);
        if (c + 1 < nchunk)
            turn(odd, even, c + 1);
    }

    // ---- the waves' sums meet in wave order (the ring is free: the last turn's barrier stood behind its last reads) --
    float4v *red = reinterpret_cast<float4v *>(lds);
#pragma unroll
    for (int xt = 0; xt < XT; xt++)
#pragma unroll
        for (int t = 0; t < MT; t++)
            red[((wave * XT + xt) * MT + t) * 64 + lane] = acc[xt][t];
    __syncthreads();
    for (int e = threadIdx.x; e < XT * MT * 64; e += 512) {
        const int l = e & 63, xt = (e >> 6) / MT, t = (e >> 6) - xt * MT;
        float4v s = red[e];
#pragma unroll
        for (int u = 1; u < 8; u++)
            s += red[u * (XT * MT * 64) + e];
        const int wr = t * 16 + (l & 15);
        if (wr < RW && m0 + wr < m) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int r = xt * 16 + (l >> 4) * 4 + j;
                if (r < nrows)
                    y[(size_t)(r0 + r) * m + m0 + wr] = s[j];
            }
        }
    }
}

// WIDE (k of whole 256-value chunks, W at a 16-byte boundary): weights by 16-byte requests, the five pieces that a row's 68
// bytes of a unit lie in.  By dwords a row takes 17, and the requests cost a CU more than the activations': 1024 x 5120 over
// 24 rows 10.1 -> 7.6 us, 5120 x 6144 over 9 / 24 rows 14.3 / 19.3 -> 12.8 / 18.5, with the depths and tiles below.  Tried on
// it: a block of 34 bytes a turn instead of two (20 % slower: a turn costs 0.2 us beside its work), two blocks 256 values apart,
// as gemv_q8_blocks_kernel sums them (10 %: twice the lines), the sums of a unit's second block taken a turn later (no gain),
// weights asked for in front of the activations (2 % slower).
template <int XT, int RW, bool HALF, bool WIDE>
struct UnitsShape {
    static constexpr int kMT = (RW + 15) / 16;              // weight tiles
    static constexpr int kXRows = 16 * XT - (HALF ? 8 : 0); // activation rows that are fetched
    static constexpr int kXBytes = kXRows * 256;
    static constexpr int kWRow = WIDE ? 80 : 68;            // a weight row's bytes of a unit, as they are fetched
    static constexpr int kSlot = kXBytes + (RW * kWRow + 15) / 16 * 16; // a unit
    static constexpr int kRead = HALF ? 2048 : 0;           // (a HALF tile's dead rows are read past the activations)
    static constexpr int kRoom = (160 << 10) - kRead;
    static constexpr int kWaves = kRoom / (8 * kSlot) >= 2 ? 8 : 4;
    // Units of a wave on the way.  More only lengthen the queue that everybody's first ones wait in: 1024 x 5120 over 24 rows
    // with 4 / 3 / 2 of them 8.7 / 8.4 / 7.6 us from HBM and 7.4 / 7.3 / 6.7 from the last-level cache, 5120 x 6144 over 9 rows
    // with 3 / 2 13.8 / 12.8 from HBM.  By dwords as well, where it was up to four: over k 5184 from HBM and 3 / 9 / 24 / 64 / 128
    // rows 1,024 weight rows 8.5 / 9.9 / 10.2 / 10.8 / 14.4 -> 7.5 / 9.3 / 9.6 / 10.0 / 13.3, 5,120 11.3 / 12.4 / 16.9 / 26.9 / 49.3 ->
    // 10.0 / 11.6 / 16.7 / 25.5 / 45.3, 12,288 19.0 / 19.8 / 24.9 / 52.7 / 98.1 -> 18.2 / 19.8 / 24.8 / 49.8 / 91.7 (with
    // the order of a turn below); 216 shapes from 512 to 12,288 weight rows 12 % less to 1 % more.
    static constexpr int kDepth = 2;
    static constexpr int kLds = kWaves * kDepth * kSlot + kRead;
    static constexpr int kChains = 8 / kWaves; // of a wave
    static_assert(kLds <= 160 << 10 && kDepth * kSlot >= kChains * XT * kMT * 1024, "");
};
template <int XT, int RW, bool HALF, bool WIDE>
constexpr int kUnitsThreads = 64 * UnitsShape<XT, RW, HALF, WIDE>::kWaves;

__device__ __forceinline__ void proj_dma4(uint32_t lds_at, const uint8_t *base, uint32_t voff)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds_at), "v"(voff), "s"(base)
                 : "memory");
}

// Wave w of WV streams units (pairs of blocks, 64 values of k) w, w + WV, ... of its rows through a ring of its own; unit
// u belongs to chain u % 8, so four waves keep two sets of sums each.  HALF: as above.
// (One wave a SIMD may use all 512 registers: held to 256, two sets of 2 x 3 tiles spill, 200 us instead of 28.)
template <int XT, int RW, bool HALF, bool WIDE>
__global__ void __launch_bounds__((kUnitsThreads<XT, RW, HALF, WIDE>), (UnitsShape<XT, RW, HALF, WIDE>::kWaves / 4))
    gemv_q8_units_kernel(const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y, int m, int k, int rows)
{
    typedef UnitsShape<XT, RW, HALF, WIDE> S;
    constexpr int MT = S::kMT, D = S::kDepth, WV = S::kWaves;
    constexpr int NX = S::kXRows / 4;          // activation requests per unit: four rows of 256 bytes each
    constexpr int kPer = WIDE ? 5 : 17;        // pieces of a weight row in a unit, of 16 or 4 bytes
    constexpr int NW = (RW * kPer + 63) / 64;  // weight requests: 64 pieces each
    constexpr int REQ = NX + NW;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int lm = lane & 15, lg = lane >> 4;
    const int nunits = k >> 6;
    const uint32_t row_bytes = (uint32_t)(k >> 5) * kQ8Block;
    const int m0 = blockIdx.x * RW, r0 = blockIdx.y * S::kXRows;
    const int nrows = rows - r0 < S::kXRows ? rows - r0 : S::kXRows;
    const int mine = wave < nunits ? (nunits - wave + WV - 1) / WV : 0;
    uint8_t *ring = lds + wave * (D * S::kSlot);
    const uint32_t ring_at = proj_lds_address(ring);
    const uint8_t *wb = w + (size_t)m0 * row_bytes;
    const uint8_t *xb = reinterpret_cast<const uint8_t *>(x + (size_t)r0 * k);
    // a unit begins 4 (u % 4) bytes into a piece, the same for all of a wave's
    const uint32_t lead = WIDE ? 4u * (wave & 3) : 0u;
    static_assert(!WIDE || WV % 4 == 0, "");
    uint32_t woff[NW], xoff[NX]; // rows past the matrix, and past the live activation rows, repeat the last
#pragma unroll
    for (int j = 0; j < NW; j++) {
        const int p = j * 64 + lane;
        const int pr = p / kPer, pd = p - pr * kPer;
        woff[j] = (uint32_t)(m0 + pr < m ? pr : m - 1 - m0) * row_bytes + (uint32_t)pd * (WIDE ? 16u : 4u);
    }
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int r = 4 * j + lg;
        xoff[j] = (uint32_t)(r < nrows ? r : nrows - 1) * (uint32_t)k * 4u + (uint32_t)((lm ^ (r & 15)) * 16);
    }
    auto issue = [&](int i) {
        const uint32_t at = ring_at + (uint32_t)((i % D) * S::kSlot);
        const uint32_t u = (uint32_t)(wave + WV * i);
        const uint8_t *xs = xb + (size_t)u * 256, *ws = wb + (size_t)u * (2 * kQ8Block) - lead;
#pragma unroll
        for (int j = 0; j < NX; j++)
            proj_dma16<false>(at + j * 1024, xs, xoff[j]);
#pragma unroll
        for (int j = 0; j < NW; j++) {
            if ((j + 1) * 64 <= RW * kPer || j * 64 + lane < RW * kPer) {
                if (WIDE)
                    proj_dma16<false>(at + S::kXBytes + j * 1024, ws, woff[j]);
                else
                    proj_dma4(at + S::kXBytes + j * 256, ws, woff[j]);
            }
        }
    };
    // unit i has arrived: only the one asked for behind it is outstanding
    static_assert(D == 2 && REQ < 64, "vmcnt has six bits");
    auto wait_unit = [&](int i) {
        if (i + 1 < mine)
            wait_vm<REQ>();
        else
            wait_vm<0>();
    };
    struct Regs {
        float4v x[XT][2][2];
        uint32_t e[MT][3], o[MT][2];
        uint16_t d[MT][2];
    };
    int wrow[MT]; // (rows of the last tile past RW repeat the last: never stored)
#pragma unroll
    for (int t = 0; t < MT; t++)
        wrow[t] = (t * 16 + lm < RW ? t * 16 + lm : RW - 1) * S::kWRow + (int)lead;
    auto load = [&](Regs &g, int i) {
        const uint8_t *buf = ring + (i % D) * S::kSlot;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const uint8_t *unit = buf + S::kXBytes + wrow[t];
            const uint32_t *e = reinterpret_cast<const uint32_t *>(unit + lg * 8);
#pragma unroll
            for (int j = 0; j < 3; j++)
                g.e[t][j] = e[j];
#pragma unroll
            for (int j = 0; j < 2; j++)
                g.o[t][j] = e[9 + j];
            g.d[t][0] = *reinterpret_cast<const uint16_t *>(unit);
            g.d[t][1] = *reinterpret_cast<const uint16_t *>(unit + kQ8Block);
        }
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    g.x[xt][b][h] = *reinterpret_cast<const float4v *>(buf + (xt * 16 + lm) * 256 + ((b * 8 + lg * 2 + h) ^ lm) * 16);
    };
    float4v acc[S::kChains][XT][MT];
#pragma unroll
    for (int s = 0; s < S::kChains; s++)
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                acc[s][xt][t] = (float4v){0, 0, 0, 0};
    auto multiply = [&](const Regs &g, float4v (&sum)[XT][MT]) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            half8 wv[MT], hi[XT], lo[XT];
            float d[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const uint32_t q0 = b == 0 ? __builtin_amdgcn_alignbit(g.e[t][1], g.e[t][0], 16) : g.o[t][0];
                const uint32_t q1 = b == 0 ? __builtin_amdgcn_alignbit(g.e[t][2], g.e[t][1], 16) : g.o[t][1];
                wv[t] = int8x8_to_f16(q0, q1);
                d[t] = (float)__builtin_bit_cast(_Float16, g.d[t][b]);
            }
#pragma unroll
            for (int xt = 0; xt < XT; xt++)
                split_hi_lo(g.x[xt][b][0], g.x[xt][b][1], hi[xt], lo[xt]);
            float4v p[XT][MT];
#pragma unroll
            for (int xt = 0; xt < XT; xt++)
#pragma unroll
                for (int t = 0; t < MT; t++)
                    p[xt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[xt], wv[t], (float4v){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int xt = 0; xt < XT; xt++)
#pragma unroll
                for (int t = 0; t < MT; t++)
                    p[xt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[xt], wv[t], p[xt][t], 0, 0, 0);
#pragma unroll
            for (int xt = 0; xt < XT; xt++)
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        sum[xt][t][j] = fmaf(d[t], p[xt][t][j], sum[xt][t][j]);
        }
    };
#pragma unroll
    for (int i = 0; i < D; i++)
        if (i < mine)
            issue(i);
    Regs even, odd;
    if (mine > 0) {
        wait_unit(0);
        load(even, 0);
    }
    // Unit i is in `now`.  Its place is asked for anew at once and its products stand in front of the wait for unit i + 1: behind
    // that wait they held up the next request as well.  us before / now over 1024 x 5120 and 9 / 24 / 32 rows 7.2 / 7.6 / 7.7 and
    // 6.9 / 7.4 / 7.4, 4096 x 4096 and 24 rows 11.7 and 11.5, 5120 x 6144 and 16 / 24 / 40 rows 14.8 / 18.7 / 23.1 and 14.5 / 18.6
    // / 22.8, from HBM.  (gemv_q8_blocks_kernel so: no gain.)
    auto turn = [&](Regs &now, Regs &next, float4v (&sum)[XT][MT], int i) {
        __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0), as above: unit i's place in the ring has been read
        asm volatile("" ::: "memory");
        if (i + D < mine)
            issue(i + D);
        __builtin_amdgcn_sched_barrier(0);
        multiply(now, sum);
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < mine) {
            wait_unit(i + 1);
            load(next, i + 1);
        }
    };
    for (int i = 0; i < mine; i += 2) {
        turn(even, odd, acc[0], i);
        if (i + 1 < mine)
            turn(odd, even, acc[S::kChains - 1], i + 1);
    }

    // ---- the chains' sums meet in their order (a wave leaves its own at the head of its ring, which it has read) ------
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    constexpr int kTiles = XT * MT * 64;
#pragma unroll
    for (int s = 0; s < S::kChains; s++)
#pragma unroll
        for (int xt = 0; xt < XT; xt++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                reinterpret_cast<float4v *>(ring)[s * kTiles + (xt * MT + t) * 64 + lane] = acc[s][xt][t];
    __syncthreads();
    for (int e = threadIdx.x; e < kTiles; e += 64 * WV) {
        const int l = e & 63, xt = (e >> 6) / MT, t = (e >> 6) - xt * MT;
        float4v s = reinterpret_cast<const float4v *>(lds)[e];
#pragma unroll
        for (int c = 1; c < 8; c++)
            s += reinterpret_cast<const float4v *>(lds + (c % WV) * (D * S::kSlot))[(c / WV) * kTiles + e];
        const int wr = t * 16 + (l & 15);
        if (wr < RW && m0 + wr < m) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int r = xt * 16 + (l >> 4) * 4 + j;
                if (r < nrows)
                    y[(size_t)(r0 + r) * m + m0 + wr] = s[j];
            }
        }
    }
}

template <int WAVES, int TILES, int CH, int XG>
static int launch_gemv_xg(hipStream_t st, const uint8_t *w, const float *x, float *y, int m, int k,
                          int rows, int rp)
{
    const size_t lds = (size_t)(k >> 5) * rp * 128 + (size_t)WAVES * TILES * 32 * sizeof(float4v);
    auto kern = gemv_q8_rows_kernel<WAVES, TILES, CH, XG>;
    const dim3 grid((unsigned)((m + 16 * TILES - 1) / (16 * TILES)), (unsigned)((rows + rp - 1) / rp), 1);
    HIPML_LAUNCH(kern, grid, dim3(64 * WAVES, 1, 1), lds, st, w, x, y, m, k, rows, rp);
    return launched("gemv_q8_0_rows");
}

template <int WAVES, int TILES, int CH>
static int launch_gemv_variant(hipStream_t st, const uint8_t *w, const float *x, float *y, int m, int k,
                               int rows, int rp)
{
    // 8-element groups of the activations per thread
    const int need = (rp * (k >> 3) + 64 * WAVES - 1) / (64 * WAVES);
    if (need <= 2)
        return launch_gemv_xg<WAVES, TILES, CH, 2>(st, w, x, y, m, k, rows, rp);
    if (need <= 4)
        return launch_gemv_xg<WAVES, TILES, CH, 4>(st, w, x, y, m, k, rows, rp);
    // rp * k <= 32,768 (the LDS budget), so 8 groups per thread always cover a pass
    return launch_gemv_xg<WAVES, TILES, CH, 8>(st, w, x, y, m, k, rows, rp);
}

// How a call of `rows` activation rows is cut: R rows a pass, waves, ng groups of gr weight rows per workgroup, and rounds of
// the chip (ng = 0: no group fits the LDS).
struct DigitsCut {
    int r, waves, gr, ng, lds, rounds, n;
};
// One round of the chip's 256 CUs, every CU the same bytes, up to 48 weight rows per workgroup (44 where a wave has several
// runs and keeps its sums apart) and several such rounds beyond: n rows a workgroup.  A unit is what a wave has in flight
// and has a fixed share of work: of the groups that fit the LDS the one for which the units cost least, as two rows more
// than they have (over 60 matrices of 256 to 14,336 weight rows and k of 2,560 to 8,192 the mean call takes 0.1 to 0.6 %
// longer than with its best group; the group that pads least, which this rule replaced, 4 to 7 %, 7168 x 5120 over three
// rows 14.2 us with seven units of four rows, 12.1 with three of ten).  Four rows only for a workgroup that has no more, or
// where nothing else fits.
static const int kDigitGroups[] = {12, 8, 10, 4};
static constexpr bool gemv_digit_group(int r, int gr) { return r <= 2 ? gr < 12 : r <= 4 || gr > 4; }
static DigitsCut gemv_digits_cut_of(int m, int k, int rows, int r)
{
    DigitsCut c = {r, 0, 0, 0, 0, 0, 0};
    // (the waves follow from k alone: a row's bits depend on them)
    const int nrun = ((k >> 8) + 1) >> 1, passes = (nrun + kDigitMaxWaves - 1) / kDigitMaxWaves;
    c.waves = (nrun + passes - 1) / passes;
    const long long all = (long long)m * ((rows + r - 1) / r), most = 256 * (passes > 1 ? 44 : 48);
    c.rounds = (int)((all + most - 1) / most);
    c.n = (int)((all + 256LL * c.rounds - 1) / (256LL * c.rounds));
    for (int gr : kDigitGroups) {
        const int ng = (c.n + gr - 1) / gr;
        const int lds = c.waves * gemv_digit_wave(r, gr, ng, passes > 1) + 64;
        if (lds > kDigitLds || !gemv_digit_group(r, gr))
            continue;
        if (c.ng == 0 || (gr == 4 ? c.n <= 4 : ng * (gr + 2) < c.ng * (c.gr + 2))) {
            c.gr = gr;
            c.ng = ng;
            c.lds = lds;
        }
    }
    return c;
}
// Five to eight rows: one pass over W with two sets of operands, or two passes of four rows.  One pass wherever two have more
// rounds (12288 x 5120 over 5 / 8 rows: one 19.6 / 21.4 us, two 28.0 / 28.7; 7168 x 5120: one 16.2 / 17.5, two 22 / 24).
// Within one round two passes read W twice but leave the second set's digits to other workgroups (1024 x 5120: one 9.6 /
// 10.7, two 7.5 / 7.6); up to six rows and from about 4,600 weight rows on the bytes tell (5120 x 6144 over 5 / 6 / 8 rows:
// one 14.7 / 15.3 / 16.2, two 15.5 / 15.5 / 15.6).
static DigitsCut gemv_digits_cut(int m, int k, int rows)
{
    const DigitsCut c = gemv_digits_cut_of(m, k, rows, rows < 4 ? rows : 4);
    if (rows > 4) {
        const DigitsCut one = gemv_digits_cut_of(m, k, rows, 8);
        if (one.ng > 0 && (c.rounds > one.rounds || (rows <= 6 && c.n > 36)))
            return one;
    }
    return c;
}

// Calls f with the kernel of (R, GR).
template <int R, typename F>
static void with_gemv_digits_kernel(int gr, F &&f)
{
    auto is = [&](auto g) {
        constexpr int GR = decltype(g)::value;
        if constexpr (gemv_digit_group(R, GR))
            if (gr == GR)
                f(&gemv_q8_digits_kernel<R, GR>);
    };
    is(std::integral_constant<int, 4>{});
    is(std::integral_constant<int, 8>{});
    is(std::integral_constant<int, 10>{});
    is(std::integral_constant<int, 12>{});
}

// Which kernel a call takes, and its variant: kRows: -; kDigits: activation rows a pass, weight rows of a group, -; kBlocks
// and kUnits: activation tiles, weight rows per workgroup, whether the last tile is half dead.
struct RowsPick {
    enum { kRows, kDigits, kBlocks, kUnits } kernel;
    int a, b, c;
};

// Calls f with the kernel of (XT, RW, HALF), its threads and its LDS bytes.
template <typename F>
static void with_gemv_blocks_kernel(int xt, int rw, bool half, F &&f)
{
#define HIPML_BLOCKS(X, R)                                                                                      \
    if (xt == X && rw == R)                                                                                     \
        return half ? f(&gemv_q8_blocks_kernel<X, R, true>, 512, BlocksShape<X, R, true>::kLds)                 \
                    : f(&gemv_q8_blocks_kernel<X, R, false>, 512, BlocksShape<X, R, false>::kLds)
    if (xt == 1) // (nine rows and more: never half dead)
        return rw == 32 ? f(&gemv_q8_blocks_kernel<1, 32, false>, 512, BlocksShape<1, 32, false>::kLds)
                        : f(&gemv_q8_blocks_kernel<1, 48, false>, 512, BlocksShape<1, 48, false>::kLds);
    HIPML_BLOCKS(2, 32);
    HIPML_BLOCKS(2, 48);
    HIPML_BLOCKS(3, 32);
    HIPML_BLOCKS(3, 48);
    HIPML_BLOCKS(4, 32);
    HIPML_BLOCKS(4, 48);
#undef HIPML_BLOCKS
}
// The tiles that any call with 16-byte requests would take (the others lose to one of them at every shape).
static constexpr bool wide_units_tile(int xt, int rw, bool half)
{
    return half ? xt == 2 || rw == 16 || rw == 32 : xt == 1 || (rw != 20 && rw != 24);
}

template <typename F>
static void with_gemv_units_kernel(int xt, int rw, bool half, bool wide, F &&f)
{
    auto pick = [&](auto x, auto r, auto h, auto w16) {
        constexpr int X = decltype(x)::value, R = decltype(r)::value;
        constexpr bool H = decltype(h)::value, W = decltype(w16)::value;
        if constexpr (!W || wide_units_tile(X, R, H))
            f(&gemv_q8_units_kernel<X, R, H, W>, kUnitsThreads<X, R, H, W>, UnitsShape<X, R, H, W>::kLds);
    };
    const std::true_type yes;
    const std::false_type no;
#define HIPML_UNITS(X, R)                                                                                       \
    if (xt == X && rw == R) {                                                                                   \
        const std::integral_constant<int, X> x;                                                                 \
        const std::integral_constant<int, R> r;                                                                 \
        return half ? (wide ? pick(x, r, yes, yes) : pick(x, r, yes, no))                                       \
                    : (wide ? pick(x, r, no, yes) : pick(x, r, no, no));                                        \
    }
    HIPML_UNITS(1, 16);
    HIPML_UNITS(1, 20);
    HIPML_UNITS(1, 24);
    HIPML_UNITS(1, 32);
    HIPML_UNITS(1, 48);
    HIPML_UNITS(2, 16);
    HIPML_UNITS(2, 20);
    HIPML_UNITS(2, 24);
    HIPML_UNITS(2, 32);
    HIPML_UNITS(2, 48);
#undef HIPML_UNITS
}
static const int kBlocksRw[2] = {32, 48}, kUnitsRw[5] = {16, 20, 24, 32, 48};

static RowsPick pick_tiles(int m, int k, int rows, bool w16)
{
    // by the shape of W alone: a row has the same bits however many travel with it
    const bool wide = k % 256 == 0 && w16, blocks = m > 6144 && wide;
    // The tile that costs least, in rounds of 256 workgroups x the cost of a unit.
    // Units by 16-byte requests, where a workgroup may also take 8 or 24 rows, whatever comes behind them: weight tiles, their
    // products with activation tiles, and requests; fewer workgroups over the same weight rows where that is a tie.  Picks the
    // fastest tile or one within 3 % at 63 shapes (512 to 6,144 weight rows, k 4096 to 6144, 9 to 128 rows), by the mean of
    // its times with the weights in HBM and in the last-level cache.  A workgroup's own bytes are what it waits for: 1024 x
    // 5120 over 16 / 24 / 32 rows by 16 rows 8.0 / 7.6 / 8.0 us (last-level cache), by 8 7.0 / 7.3 / 7.5; 6144 x 5120 over 40
    // rows by 32 rows 22.1, by 24 18.2.
    // The others: the cycles of a unit in the eight waves of a CU, as the sum of its vector instructions (two waves a SIMD,
    // 4 cycles each) and its requests (16 cycles); blocks of 7,168 to 12,288 weight rows over 9 to 128 rows: the fastest
    // tile or one within 6 %.
    RowsPick best = {blocks ? RowsPick::kBlocks : RowsPick::kUnits, 0, 0, 0};
    long long best_cost = 0;
    for (int xt = 1; xt <= (blocks ? 4 : 2) && 16 * (xt - 1) < rows; xt++)
        for (int rw : kUnitsRw)
            for (int half = wide && !blocks ? 1 : 0; half >= 0; half--) {
                if (blocks ? rw < 32 : wide && !wide_units_tile(xt, rw, half != 0))
                    continue;
                const int mt = (rw + 15) / 16, step = 16 * xt - 8 * half;
                const long long rounds = ((long long)((m + rw - 1) / rw) * ((rows + step - 1) / step) + 255) / 256;
                long long cost;
                if (wide && !blocks) {
                    cost = rounds * (mt + mt * xt + step / 4 + (rw * 5 + 63) / 64) * 128 + (rows + step - 1) / step;
                } else {
                    const int valu = 26 * mt + 28 * xt + 8 * mt * xt + 20;
                    const int requests = 4 * xt + (rw * 17 + 63) / 64 / (blocks ? 4 : 1);
                    cost = rounds * (8 * valu + 8 * 16 * requests);
                }
                if (best_cost == 0 || cost < best_cost) {
                    best_cost = cost;
                    best.a = xt;
                    best.b = rw;
                    best.c = wide && !blocks ? half : rows <= 16 * xt - 8 ? 1 : 0;
                }
            }
    return best;
}

static RowsPick pick_rows(int m, int k, int rows, bool w16)
{
    // Up to eight rows over the digits kernel: weight rows of whole 256-value chunks at 16-byte boundaries.
    if (rows <= 8 && k % 256 == 0 && w16) {
        const DigitsCut c = gemv_digits_cut(m, k, rows);
        return {RowsPick::kDigits, c.r, c.gr, 0};
    }
    return rows > kGemvMaxRows ? pick_tiles(m, k, rows, w16) : RowsPick{RowsPick::kRows, 0, 0, 0};
}

template <int R>
static void launch_gemv_digits(hipStream_t st, const uint8_t *w, const float *x, float *y, int m, int k, int rows)
{
    const DigitsCut c = gemv_digits_cut(m, k, rows);
    const dim3 grid((unsigned)((m + c.ng * c.gr - 1) / (c.ng * c.gr)), (unsigned)((rows + R - 1) / R), 1);
    with_gemv_digits_kernel<R>(c.gr, [&](auto kernel) {
        HIPML_LAUNCH(kernel, grid, dim3(64 * c.waves, 1, 1), (size_t)c.lds, st, w, x, y, m, k, rows, c.ng);
    });
}

static bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// (x at a 16-byte boundary: the caller has checked it)
int launch_gemv_q8_rows(hipStream_t st, const uint8_t *w, const float *x, float *y, int m, int k, int rows)
{
    const RowsPick p = pick_rows(m, k, rows, aligned16(w));
    if (p.kernel == RowsPick::kRows) {
        int rp = gemv_rows_per_pass(k);
        if (rp < 1)
            return fail(HIPML_ATTN_E_RANGE, "k %d: one activation row does not fit the LDS operand buffer", k);
        rp = rows < rp ? rows : rp;
        // One 16-row weight tile per workgroup keeps the kernel inside 128 registers, so two workgroups
        // share a CU and the 320 workgroups of a 5120-row matrix start together (workgroups start in
        // windows of as many as fit the chip; a second window opens when the first has drained).
        return launch_gemv_variant<8, 1, 6>(st, w, x, y, m, k, rows, rp);
    }
    if (p.kernel == RowsPick::kDigits) {
        switch (p.a) {
        case 1: launch_gemv_digits<1>(st, w, x, y, m, k, rows); break;
        case 2: launch_gemv_digits<2>(st, w, x, y, m, k, rows); break;
        case 3: launch_gemv_digits<3>(st, w, x, y, m, k, rows); break;
        case 4: launch_gemv_digits<4>(st, w, x, y, m, k, rows); break;
        default: launch_gemv_digits<8>(st, w, x, y, m, k, rows);
        }
        return launched("gemv_q8_0_rows");
    }
    const int xt = p.a, rw = p.b;
    const int step = 16 * xt - 8 * p.c; // activation rows of a workgroup
    const dim3 grid((unsigned)((m + rw - 1) / rw), (unsigned)((rows + step - 1) / step), 1);
    auto go = [&](auto kernel, int threads, int lds) {
        HIPML_LAUNCH(kernel, grid, dim3((unsigned)threads, 1, 1), (size_t)lds, st, w, x, y, m, k, rows);
    };
    if (p.kernel == RowsPick::kBlocks)
        with_gemv_blocks_kernel(xt, rw, p.c, go);
    else
        with_gemv_units_kernel(xt, rw, p.c, k % 256 == 0 && aligned16(w), go);
    return launched("gemv_q8_0_rows");
}

// For tests and the benchmark: the kernel that a call takes, as kernel * 10^6 + a * 10^4 + b * 100 + c of its RowsPick.
extern "C" int hipml_dbg_rows_kernel(int m, int k, int rows, int w_aligned16)
{
    const RowsPick p = pick_rows(m, k, rows, w_aligned16 != 0);
    return p.kernel * 1000000 + p.a * 10000 + p.b * 100 + p.c;
}

template <int WAVES, int TILES, int CH>
static hipError_t raise_gemv_lds()
{
    hipError_t e = hipSuccess;
    auto raise = [&](const void *f) {
        if (e == hipSuccess)
            e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10);
    };
    raise(reinterpret_cast<const void *>(&gemv_q8_rows_kernel<WAVES, TILES, CH, 2>));
    raise(reinterpret_cast<const void *>(&gemv_q8_rows_kernel<WAVES, TILES, CH, 4>));
    raise(reinterpret_cast<const void *>(&gemv_q8_rows_kernel<WAVES, TILES, CH, 8>));
    return e;
}

int proj_init()
{
    hipError_t e = raise_gemv_lds<8, 1, 6>();
    auto raise = [&](const void *f) {
        if (e == hipSuccess)
            e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10);
    };
    auto raise_digits = [&](auto r) {
        for (int gr : kDigitGroups)
            with_gemv_digits_kernel<decltype(r)::value>(
                gr, [&](auto kernel) { raise(reinterpret_cast<const void *>(kernel)); });
    };
    raise_digits(std::integral_constant<int, 1>{});
    raise_digits(std::integral_constant<int, 2>{});
    raise_digits(std::integral_constant<int, 3>{});
    raise_digits(std::integral_constant<int, 4>{});
    raise_digits(std::integral_constant<int, 8>{});
    for (int xt = 1; xt <= 4; xt++)
        for (bool half : {false, true}) {
            auto up = [&](auto kernel, int, int) { raise(reinterpret_cast<const void *>(kernel)); };
            for (int rw : kBlocksRw)
                with_gemv_blocks_kernel(xt, rw, half, up);
            for (int rw : kUnitsRw)
                for (bool wide : {false, true})
                    with_gemv_units_kernel(xt, rw, half, wide, up);
        }
    if (e != hipSuccess)
        return fail((int)e, "hipFuncSetAttribute(projection LDS) failed: %d (%s)", (int)e, hipGetErrorString(e));
    return 0;
}

} // namespace hipml
