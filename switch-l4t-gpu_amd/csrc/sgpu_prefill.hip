// sgpu_prefill.hip -- the Qwen2.5 prompt's products on the fp16 matrix cores (gfx950).
//
// The layer weights are fp16, so only x has to be cut to fit the fp16 matrix instructions, and
// it keeps its 24 bits: the kernels that produce an x (RMSNorm, attention, SwiGLU) write it as
// three fp16 pieces x * 2^s = p0 + p1 + p2 (11 + 11 + 2 of the 24 mantissa bits), s one power of
// two per row and 64 consecutive values, chosen so that the largest of them lies in
// [2^14, 2^15).  Every product of a weight and a piece is exact in the fp32 accumulators, and
// an fp32 dot product costs three fp16 MFMAs instead of sixteen fp32 ones' time.  A value less
// than 2^-16 of its block's largest keeps fewer than 24 bits: the pieces' error is at most
// 2^-39 of the block's largest value (half an fp16 subnormal step, 2^-25, over 2^14).
//
// Piece layout ("planes"): row t holds K codes of p0, K of p1, K of p2; beside them one float
// 2^-s per row and 64-block.  Non-finite values go to p0 as they are (p1 = p2 = 0) and s is
// chosen over the finite ones.
//
// Measured against the same layers on fp32 MFMA tiles (sgpu_pf_gemm, 32x32 per block): a prompt
// of 500 rows of the Qwen2.5-0.5B sizes 6.08 -> 3.30 ms, of 3001 rows 39.5 -> 11.1-11.5 ms; distance
// of the logits from a 64-bit forward 1.1e-6 -> 6.2e-7 and 9.3e-7 -> 7.0e-7.
//
// This code object keeps fp16 subnormals (the pieces use them).  The reference reads subnormal
// weights as +0: the engine clears those codes once, where it uploads the weights
// (sgpu_h16_flush).
#include "gemv_core.h"

namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int G = 64;                                  // values per scale

// |x|'s bits if x is finite, else 0: the maximum of these over a block picks its scale.
__device__ __forceinline__ uint32_t mag_bits(float x) {
    const uint32_t b = __float_as_uint(x) & 0x7fffffffu;
    return b < 0x7f800000u ? b : 0u;
}
// 2^s and 2^-s for a block whose largest magnitude has bits m: s = 14 - exponent, at most 126
// (so that 2^-s stays a normal number).
__device__ __forceinline__ void block_scale(uint32_t m, float& up, float& down) {
    const int s = min(141 - (int)(m >> 23), 126);
    up = __uint_as_float((uint32_t)(s + 127) << 23);
    down = __uint_as_float((uint32_t)(127 - s) << 23);
}
__device__ __forceinline__ void split3(const float (&x)[4], float up, f16x4& p0, f16x4& p1, f16x4& p2) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float y = x[i] * up;
        p0[i] = (_Float16)y;
        float r = y - (float)p0[i];
        r = __builtin_isfinite(y) ? r : 0.0f;
        p1[i] = (_Float16)r;
        p2[i] = (_Float16)(r - (float)p1[i]);
    }
}

// y[k] of row t as the pieces hold it.
__device__ __forceinline__ float plane_at(const uint16_t* row, const float* down, int K, int k) {
    float v = 0.0f;
    for (int p = 2; p >= 0; p--) v += (float)__builtin_bit_cast(_Float16, row[(size_t)p * K + k]);
    return v * down[k / G];
}
// A dot product again, serially and with the reference's own decode of the weight codes: for
// the sums that come out non-finite (a code of exponent 31 is a finite value in the reference).
__device__ __noinline__ float recompute(const uint16_t* __restrict__ w, const uint16_t* __restrict__ row,
                                        const float* __restrict__ down, int K) {
    float acc = 0.0f;
    for (int k = 0; k < K; k++) acc = __builtin_fmaf(sgpu_h2f(w[k]), plane_at(row, down, K, k), acc);
    return acc;
}

enum { EPI_STORE, EPI_SWIGLU };

// Y[t][n] = X[t] . W[n] + bias?[n] (EPI_STORE; accum != 0: added to Y), or silu(gate) * up as
// pieces for the next product (EPI_SWIGLU: W holds N gate rows, then N up rows).
//
// Bound: the matrix cores, and below some 1000 rows the steps' loads.  (These cores reach 2.0
// PFLOP/s on random operands, 2.26 on zeros, by bin/sgemm_floor; gate|up at 3001 rows runs at 1.04 PFLOP/s of piece
// products, 1.4 with its loads taken out.)  A block of 2x2 waves computes 64*TF tokens x 64*NF weight rows, a
// wave 32*TF x 32*NF of them in 16x16 tiles.  Per step of 64 k the block's pieces and weights go straight into
// LDS (16 bytes a lane, no registers; a row's eight 16-byte chunks are stored at chunk ^ (row / 2
// % 8), so that the operand reads of sixteen consecutive rows use all banks); there is one buffer,
// and the two or more blocks on a CU cover each other's loads.  The products run transposed
// (weights as A), so a lane holds one token per 16x16 tile and scales its step's sum with one
// factor; four consecutive n per lane make 16-byte stores.  Within a step the smallest pieces
// are summed first.
// S > 1: K split over S blocks per tile by the hand-off of sgpu_device.h; ws holds S * tiles
// records of 4096*TF*NF floats, cnt one zeroed counter per tile.
// Preconditions (launcher): blockDim 256, K % 64 == 0, N % 64 == 0, operands 16-byte aligned,
// N * K (twice that for SwiGLU) and 3 * T * K below 2^30 codes, grid = tiles * S blocks.
template <int TF, int NF, int EPI>
__device__ __forceinline__ void pf_mm(const uint16_t* __restrict__ W, const uint16_t* __restrict__ X,
                                      const float* __restrict__ xd, const float* __restrict__ bias,
                                      float* __restrict__ Y, uint16_t* __restrict__ P, float* __restrict__ pd, int K,
                                      int N, int T, int S, float* __restrict__ ws, unsigned* __restrict__ cnt,
                                      int accum) {
    constexpr int TT = 64 * TF, NR = 64 * NF;              // tokens and weight rows per block
    constexpr int TM = 2 * TF, NM = 2 * NF;                // a wave's 16x16 tiles
    constexpr int NC = EPI == EPI_SWIGLU ? NR / 2 : NR;    // output columns per block
    static_assert(EPI == EPI_STORE || NF == 4, "a wave's SwiGLU columns are one 64-block");
    __shared__ __attribute__((aligned(1024))) uint16_t xs[3 * TT * G];
    __shared__ __attribute__((aligned(1024))) uint16_t wsm[NR * G];
    int& last_s = *reinterpret_cast<int*>(xs);             // after the k loop, whose last barrier frees xs
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, quarter = lane >> 4, wt = wave >> 1, wn = wave & 1;
    const int ntt = (T + TT - 1) / TT, ntn = (N + NC - 1) / NC, ntiles = ntt * ntn;
    // Blocks are dealt round-robin to the 8 XCDs: each XCD takes a contiguous run of tiles, eight
    // token tiles by all columns at a time, so that the blocks on one XCD share about as many
    // pieces as weight rows in its L2.
    const int total = ntiles * S, xcd = blockIdx.x % 8;
    const int unit = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
    const int tile = unit % ntiles, sp = unit / ntiles;
    const int band = tile / (8 * ntn), bt = min(8, ntt - 8 * band), in = tile - band * 8 * ntn;
    const int t0 = (8 * band + in % bt) * TT, n0 = (in / bt) * NC;
    const int ng = K / G, g0 = sp * ng / S, g1 = (sp + 1) * ng / S;

    // Loads: each wave instruction brings eight rows of 128 bytes.  Rows past T or N repeat a
    // valid row and are never stored.
    const int lr = lane >> 3, lc = 16 * ((lane & 7) ^ (4 * (wave & 1) + (lr >> 1)));
    int xo[2 * TF], wo[2 * NF];
#pragma unroll
    for (int q = 0; q < 2 * TF; q++) xo[q] = min(t0 + 32 * q + 8 * wave + lr, T - 1) * (6 * K) + lc;
#pragma unroll
    for (int q = 0; q < 2 * NF; q++) {
        const int r = 32 * q + 8 * wave + lr;
        int n;
        if constexpr (EPI == EPI_SWIGLU) {                 // wave column wn: 64 gate rows, then their 64 up rows
            const int c = min(n0 + 64 * (r / 128) + r % 64, N - 1);
            n = r % 128 < 64 ? c : N + c;
        } else {
            n = min(n0 + r, N - 1);
        }
        wo[q] = n * (2 * K) + lc;
    }
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)X, (short)0, T * (6 * K), 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)W, (short)0, (EPI == EPI_SWIGLU ? 2 * N : N) * (2 * K), 0x00020000);
    int tok[TM];                                           // this lane's tokens, clamped
#pragma unroll
    for (int f = 0; f < TM; f++) tok[f] = min(t0 + 32 * TF * wt + 16 * f + l16, T - 1);

    // acc[f][j]: tokens 16 * f.., weight rows 16 * j.. of the wave's part
    sgpu_f32x4 acc[TM][NM];
#pragma unroll
    for (int f = 0; f < TM; f++)
#pragma unroll
        for (int j = 0; j < NM; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[f][j][r] = 0.0f;
    const int lrow = (lane & 15) * G, sw = (lane & 15) >> 1;      // operand reads: row lane % 16, swizzled chunk
    const uint16_t* const xl = xs + 32 * TF * wt * G + lrow;
    const uint16_t* const wl = wsm + 32 * NF * wn * G + lrow;
    auto read_w = [&](int j, f16x8 (&w)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; s++) w[s] = *reinterpret_cast<const f16x8*>(wl + 16 * j * G + 8 * ((4 * s + quarter) ^ sw));
    };

    for (int g = g0; g < g1; g++) {
        const int kb = g * (2 * G);
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int q = 0; q < 2 * TF; q++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(xs + (p * TT + 32 * q + 8 * wave) * G), 16, xo[q],
                                                         p * 2 * K + kb, 0, 0);
#pragma unroll
        for (int q = 0; q < 2 * NF; q++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wsm + (32 * q + 8 * wave) * G), 16, wo[q], kb, 0, 0);
        float down[TM];
#pragma unroll
        for (int f = 0; f < TM; f++) down[f] = xd[(size_t)tok[f] * ng + g];
        __builtin_amdgcn_s_waitcnt(0);                     // this wave's rows are in LDS
        __syncthreads();
        f16x8 w[2][2], x[2][3][2];
        auto read_x = [&](int f) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 2; p >= 0; p--)
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        x[u][p][s] = *reinterpret_cast<const f16x8*>(xl + (p * TT + 16 * (f + u)) * G +
                                                                     8 * ((4 * s + quarter) ^ sw));
        };
        read_w(0, w[0]);
        read_x(0);
        // one column of two 16x16 tiles per round: the next column's weights are read and the
        // last one's sums are scaled under this one's products
        sgpu_f32x4 c[2][2];
#pragma unroll
        for (int i = 0; i <= TF * NM; i++) {
            const int f = 2 * (i / NM), j = i % NM;
            if (i < TF * NM) {
                if (i + 1 < TF * NM) read_w((j + 1) % NM, w[(i + 1) % 2]);
#pragma unroll
                for (int u = 0; u < 2; u++) c[i % 2][u] = sgpu_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int p = 2; p >= 0; p--)
#pragma unroll
                    for (int s = 0; s < 2; s++)
#pragma unroll
                        for (int u = 0; u < 2; u++)
                            c[i % 2][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[i % 2][s], x[u][p][s], c[i % 2][u], 0, 0, 0);
                if (j == NM - 1 && i + 1 < TF * NM) read_x(f + 2);   // as the last products free their registers
            }
            if (i > 0) {
                const int f1 = 2 * ((i - 1) / NM), j1 = (i - 1) % NM;
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        acc[f1 + u][j1][r] = __builtin_fmaf(c[(i - 1) % 2][u][r], down[f1 + u], acc[f1 + u][j1][r]);
            }
            // rounds stay in order: the wave keeps within half a SIMD's registers
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();                                   // reads done before the next step's rows land
    }

    // Accumulator r of tile (f, j): token tok[f], weight row 32 * NF * wn + 16 * j + 4 * quarter + r
    // of the block.
    if (EPI == EPI_STORE && S > 1) {
        constexpr int REC = 4096 * TF * NF;
        float* rec = ws + (size_t)(sp * ntiles + tile) * REC + tid;
#pragma unroll
        for (int f = 0; f < TM; f++)
#pragma unroll
            for (int j = 0; j < NM; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    __hip_atomic_store(rec + ((f * NM + j) * 4 + r) * 256, acc[f][j][r], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);                     // this wave's partial stores are acknowledged
        __syncthreads();
        if (tid == 0) {
            last_s = __hip_atomic_fetch_add(cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
            if (last_s) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // before the others' partials
        }
        __syncthreads();
        if (!last_s) return;
        // all splits in order, this block's own among them, 16 loads issued before the first add
        for (int s2 = 0; s2 < S; s2++) {
            const float* src = ws + (size_t)(s2 * ntiles + tile) * REC + tid;
#pragma unroll
            for (int f = 0; f < TM; f++)
#pragma unroll
                for (int j = 0; j < NM; j += (NM < 4 ? NM : 4)) {
                    sgpu_f32x4 v[NM < 4 ? NM : 4];
#pragma unroll
                    for (int i = 0; i < (NM < 4 ? NM : 4); i++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            v[i][r] = __hip_atomic_load(src + ((f * NM + j + i) * 4 + r) * 256, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int i = 0; i < (NM < 4 ? NM : 4); i++)
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[f][j + i][r] = s2 == 0 ? v[i][r] : acc[f][j + i][r] + v[i][r];
                }
        }
        if (tid == 0) __hip_atomic_store(cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int tl = t0 + 32 * TF * wt + l16;
    uint32_t top = 0;                                      // some sum non-finite: looked at once for the wave
#pragma unroll
    for (int f = 0; f < TM; f++)
#pragma unroll
        for (int j = 0; j < NM; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) top = max(top, __float_as_uint(acc[f][j][r]) & 0x7fffffffu);
    const bool redo = __any(top >= 0x7f800000u);
    if constexpr (EPI == EPI_STORE) {
        const int nl = n0 + 32 * NF * wn + 4 * quarter;
#pragma unroll
        for (int f = 0; f < TM; f++) {
            const int t = tl + 16 * f;
            if (t >= T) continue;
#pragma unroll
            for (int j = 0; j < NM; j++) {
                const int n = nl + 16 * j;
                if (n >= N) continue;
                sgpu_f32x4 v = acc[f][j];
                if (redo) {
                    for (int e = 0; e < 4; e++)
                        if (!__builtin_isfinite(v[e]))
                            v[e] = recompute(W + (size_t)(n + e) * K, X + (size_t)t * 3 * K, xd + (size_t)t * ng, K);
                }
                sgpu_f32x4* y = reinterpret_cast<sgpu_f32x4*>(Y + (size_t)t * N + n);
                if (bias) v += *reinterpret_cast<const sgpu_f32x4*>(bias + n);
                if (accum) v = *y + v;
                *y = v;
            }
        }
    } else {
#pragma clang fp contract(off)
        const int c0 = n0 + 64 * wn;                       // the wave's 64 columns (whole: N % 64 == 0)
#pragma unroll
        for (int f = 0; f < TM; f++) {
            const int t = tl + 16 * f;
            uint32_t m = 0;
            if (redo) {
#pragma unroll
                for (int j = 0; j < NM; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (!__builtin_isfinite(acc[f][j][r])) {
                            const int n = min(c0 + 16 * (j % 4) + 4 * quarter + r, N - 1);
                            acc[f][j][r] = recompute(W + (size_t)(j < 4 ? n : N + n) * K, X + (size_t)min(t, T - 1) * 3 * K,
                                                     xd + (size_t)min(t, T - 1) * ng, K);
                        }
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float gt = acc[f][j][r], v = (gt / (1.0f + expf(-gt))) * acc[f][j + 4][r];
                    acc[f][j][r] = v;
                    m = max(m, mag_bits(v));
                }
            m = max(m, (uint32_t)__shfl_xor((int)m, 16));
            m = max(m, (uint32_t)__shfl_xor((int)m, 32));
            float up, down;
            block_scale(m, up, down);
            // through LDS (the wave's own 6 KB, free after the k loop) so that a row's 64 codes of
            // a piece leave as one 128-byte line: 8-byte stores straight from the accumulators
            // took 311 us instead of 299 at 3001 rows and K 1792 (172 either way at K 896)
            uint16_t* const st = xs + wave * (3 * 16 * G);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float x[4] = {acc[f][j][0], acc[f][j][1], acc[f][j][2], acc[f][j][3]};
                f16x4 p[3];
                split3(x, up, p[0], p[1], p[2]);
#pragma unroll
                for (int q = 0; q < 3; q++)
                    *reinterpret_cast<f16x4*>(st + (16 * q + l16) * G + 8 * ((2 * j + quarter / 2) ^ sw) + 4 * (quarter & 1)) = p[q];
            }
            sgpu::wave_sync();
            if (t < T && c0 < N && quarter == 0) pd[(size_t)t * (N / G) + c0 / G] = down;
#pragma unroll
            for (int q = 0; q < 3; q++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int r = 8 * i + lr, tr = t0 + 32 * TF * wt + 16 * f + r, ch = lane & 7;
                    const sgpu_u32x4 v = *reinterpret_cast<const sgpu_u32x4*>(st + (16 * q + r) * G + 8 * (ch ^ (r >> 1)));
                    if (tr < T && c0 < N)
                        *reinterpret_cast<sgpu_u32x4*>(P + (size_t)tr * 3 * N + (size_t)q * N + c0 + 8 * ch) = v;
                }
            sgpu::wave_sync();
        }
    }
}

// Causal attention for prompt rows on the fp32 matrix cores: T query rows at positions pos0..
// (row t's q rotated in place in its qkv vector of length QKVD) over cached positions
// 0..pos0+t, one block per query head and 32 query rows.  Output row t: NH*HD floats of out, or
// (P given, HD % 64 == 0) its pieces for the next product.
//
// Bound: the matrix cores (4*HD flop per query, key and head).  The keys are taken in tiles of
// 32, dealt to the block's four waves (wave w: tiles w, w+4, ..); each wave keeps its own
// running maximum, sum and output over its tiles (online softmax) and the four are merged once
// through LDS at the end, so the key loop has no barrier and a short prompt still fills the
// CUs' SIMDs.  Both products are laid out so that no operand passes through LDS:
//  * scores transposed, S^T = K Q^T: lane (l32, h) feeds key l32's dims 8*v + 4*h.. as A and query
//    l32's as B (16-byte loads, the halves' side by side; the k order of a dot product is free:
//    with dims HD/2*h.. each load touched twice the cache lines), so accumulator r of a
//    lane is key 8*(r/4) + 4*h + r%4 of query l32 and the softmax over keys is in-lane, plus
//    one exchange between the lane halves;
//  * O^T = V^T P^T: step r multiplies the keys the lanes hold in accumulator r, so P is the B
//    operand where it lies, and A is V[that key][NB*l32 + j] for dim block j (NB = HD/32
//    consecutive dims per lane: one 4*NB-byte load per step).
// K and V of the wave's next tile are loaded while this tile's softmax and second product run.
// Loads go through buffer resources that end at the last valid key row: rows past it read as
// zero and are masked.  In tiles that reach past some row's own position, non-finite values of V are
// taken out of the product (0 times an infinity is a NaN) and added at the end to the rows that see them.  The heavy blocks (last rows) are dispatched first.
// Sums are kept short, as the vector-ALU form's were: four accumulators for a score's dims, and a
// tile's output summed by itself before it is added (logits against 64 bits, GPT-2, mean of 16 seeds:
// 300 rows 5.64e-7 -> 5.59e-7, 1000 rows 6.25e-7 -> 6.17e-7, vector ALUs 5.61e-7 and 6.13e-7; Qwen, 3001
// rows 7.9e-7 -> 7.0e-7; the time stays, 11.18 -> 11.10 ms, as long as the wave keeps to half a
// SIMD's registers: 308 of them took 11.99).
// Measured against one block per head and row on the vector ALUs, which read K and V once per
// row, 14 query and 2 KV heads of 64: 50 -> 16 us a launch at 500 rows, 1390 -> 172 us for 3001 rows
// (194 with expf and with a lane's dims of K in one run).
template <int HD>
__device__ __forceinline__ void pf_attn(const float* __restrict__ qkv, const float* __restrict__ kc,
                                        const float* __restrict__ vc, float* __restrict__ out, uint16_t* __restrict__ P,
                                        float* __restrict__ pd, int pos0, int T, int NH, int NKV, float scale,
                                        int QKVD) {
    constexpr int HH = HD / 2, NB = HD / 32, PITCH = HD + 1;
    typedef uint32_t vseg __attribute__((ext_vector_type(NB)));
    __shared__ float part[4][32][PITCH];
    __shared__ float ml[4][2][32];
    __shared__ int odd[4];                            // per wave: some V was taken out
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int head = blockIdx.x % NH, q0 = ((T + 31) / 32 - 1 - blockIdx.x / NH) * 32;
    const int KVD = NKV * HD, g = head / (NH / NKV);
    const int n = pos0 + min(T, q0 + 32);             // keys that some row of the block reads
    const int ntile = (n + 31) / 32, qpos = pos0 + q0 + l32;

    float qv[HH];
    {
        const float* qr = qkv + (size_t)min(q0 + l32, T - 1) * QKVD + (size_t)head * HD + 4 * h;
#pragma unroll
        for (int v = 0; v < HH / 4; v++) {
            const sgpu_f32x4 a = *reinterpret_cast<const sgpu_f32x4*>(qr + 8 * v);
#pragma unroll
            for (int e = 0; e < 4; e++) qv[4 * v + e] = a[e];
        }
    }
    sgpu_f32x4 kr[HH / 4];
    vseg vr[16];
    const int koff = (l32 * KVD + 4 * h) * 4, voff = (4 * h * KVD + NB * l32) * 4;
    auto tile_rsrc = [&](const float* c, int t) __attribute__((always_inline)) {
        const int rows = max(n - 32 * t, 0);
        return __builtin_amdgcn_make_buffer_rsrc((void*)(c + (size_t)g * HD + (size_t)t * 32 * KVD), (short)0,
                                                 rows > 0 ? (min(rows, 32) * KVD - (KVD - HD)) * 4 : 0, 0x00020000);
    };
    auto load_k = [&](int t) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(kc, t);
#pragma unroll
        for (int v = 0; v < HH / 4; v++)
            kr[v] = __builtin_bit_cast(sgpu_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, koff + 32 * v, 0, 0));
    };
    auto load_v = [&](int t) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(vc, t);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int o = voff + (8 * (r / 4) + r % 4) * KVD * 4;
            if constexpr (NB == 1) vr[r][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
            else if constexpr (NB == 2) vr[r] = __builtin_bit_cast(vseg, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
            else vr[r] = __builtin_bit_cast(vseg, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
        }
    };

    // The softmax in powers of two: a weight is one FMA and one v_exp_f32, exp2(score * scale2 - max).  The
    // product is not rounded before the subtraction, so weights near the maximum, which carry the sum,
    // are exact to v_exp_f32's own rounding however large the scores are.
    const float scale2 = scale * 1.44269504088896340736f;
    f32x16 o[NB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[j][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    bool taken = false;                               // non-finite V taken out of a tile
    load_k(wave);
    load_v(wave);
    for (int t = wave; t < ntile; t += 4) {
        f32x16 s4[4], s;
#pragma unroll
        for (int r = 0; r < 16; r++) s4[0][r] = s4[1][r] = s4[2][r] = s4[3][r] = 0.0f;
#pragma unroll
        for (int k = 0; k < HH; k++)                  // four accumulators: no MFMA waits for the one before it
            s4[k % 4] = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[k / 4][k % 4], qv[k], s4[k % 4], 0, 0, 0);
        load_k(t + 4);
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = (s4[0][r] + s4[1][r]) + (s4[2][r] + s4[3][r]);
        const bool past = 32 * t + 31 > pos0 + q0;    // the tile reaches past some row's own position
        if (past) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (32 * t + 8 * (r / 4) + 4 * h + r % 4 > qpos) s[r] = -INFINITY;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32)) * scale2);
        const float base = mx == -INFINITY ? 0.0f : mx;   // every key so far masked: weights are all zero
        const float al = __builtin_amdgcn_exp2f(m - base);
        m = mx;
        float sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale2, -base));
            sum += s[r];
        }
        l = l * al + sum;
        if (past) {                                   // a weight of zero must not meet an infinity or a NaN
#pragma unroll
            for (int r = 0; r < 16; r++)
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    const bool odd = (vr[r][j] & 0x7f800000u) == 0x7f800000u;
                    taken |= odd;
                    vr[r][j] = odd ? 0u : vr[r][j];
                }
        }
        // the tile's sum by itself, then added: chains of 32 keys instead of all of the wave's
        f32x16 c[NB];
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) c[j][r] = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                c[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(vr[r][j]), s[r], c[j], 0, 0, 0);
        load_v(t + 4);
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[j][r] = __builtin_fmaf(o[j][r], al, c[j][r]);
    }
    l += __shfl_xor(l, 32);
    taken = __any(taken);
    if (lane == 0) odd[wave] = taken;
    if (h == 0) {
        ml[wave][0][l32] = m;
        ml[wave][1][l32] = l;
    }
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) part[wave][l32][NB * (8 * (r / 4) + 4 * h + r % 4) + j] = o[j][r];
    __syncthreads();
    // Merge: 8 threads per query row, HD/8 dims each; the four waves in order.
    const int q = threadIdx.x / 8, d0 = (threadIdx.x % 8) * (HD / 8);
    if (q0 + q >= T) return;
    float M = ml[0][0][q];
#pragma unroll
    for (int w = 1; w < 4; w++) M = fmaxf(M, ml[w][0][q]);
    if (M == -INFINITY) M = 0.0f;
    float wt[4], L = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        wt[w] = __builtin_amdgcn_exp2f(ml[w][0][q] - M);
        L = __builtin_fmaf(ml[w][1][q], wt[w], L);
    }
    float v[HD / 8];
    uint32_t mag = 0;
#pragma unroll
    for (int e = 0; e < HD / 8; e++) {
        float a = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) a = __builtin_fmaf(part[w][q][d0 + e], wt[w], a);
        v[e] = a / L;
        mag = max(mag, mag_bits(v[e]));
    }
    const size_t C = (size_t)NH * HD, t = q0 + q, c = (size_t)head * HD + d0;
    if (odd[0] | odd[1] | odd[2] | odd[3]) {          // the V taken out, to the rows that see them
        for (int k = (pos0 + q0 + 1) / 32 * 32; k <= pos0 + (int)t; k++) {
            const size_t kv = (size_t)k * KVD + (size_t)g * HD;
            bool any = false;
            for (int e = 0; e < HD / 8; e++) any |= !__builtin_isfinite(vc[kv + d0 + e]);
            if (!any) continue;
            float s = 0.0f;
            for (int d = 0; d < HD; d++) s = __builtin_fmaf(qkv[t * QKVD + (size_t)head * HD + d], kc[kv + d], s);
            const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(s, scale2, -M)) / L;
#pragma unroll
            for (int e = 0; e < HD / 8; e++) {
                const float x = vc[kv + d0 + e];
                v[e] = __builtin_isfinite(x) ? v[e] : __builtin_fmaf(w, x, v[e]);
            }
        }
        mag = 0;
#pragma unroll
        for (int e = 0; e < HD / 8; e++) mag = max(mag, mag_bits(v[e]));
    }
    if constexpr (HD >= G) {
        if (P) {                                      // block-uniform; a 64-block is 8 or 4 threads of one row
#pragma unroll
            for (int o = 1; o < 8 * G / HD; o *= 2) mag = max(mag, (uint32_t)__shfl_xor((int)mag, o));
            float up, down;
            block_scale(mag, up, down);
            if (d0 % G == 0) pd[t * (C / G) + c / G] = down;
            uint16_t* row = P + t * 3 * C + c;
#pragma unroll
            for (int e = 0; e < HD / 8; e += 4) {
                const float x[4] = {v[e], v[e + 1], v[e + 2], v[e + 3]};
                f16x4 p0, p1, p2;
                split3(x, up, p0, p1, p2);
                *reinterpret_cast<f16x4*>(row + e) = p0;
                *reinterpret_cast<f16x4*>(row + C + e) = p1;
                *reinterpret_cast<f16x4*>(row + 2 * C + e) = p2;
            }
            return;
        }
    }
#pragma unroll
    for (int e = 0; e < HD / 8; e++) out[t * C + c + e] = v[e];
}

}  // namespace

extern "C" {

// fp16 subnormal codes of w become +0, as the reference reads them (n codes, n % 8 == 0, 16-byte
// aligned).
__global__ void __launch_bounds__(256) sgpu_h16_flush(sgpu_u32x4* __restrict__ w, size_t n) {
    const size_t nv = n / 8, stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < nv; i += stride) {
        sgpu_u32x4 v = w[i];
        bool any = false;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uint32_t u = v[e];
            if (!(u & 0x7c00u)) u &= 0xffff0000u;
            if (!(u & 0x7c000000u)) u &= 0xffffu;
            any |= u != v[e];
            v[e] = u;
        }
        if (any) w[i] = v;
    }
}

// RMSNorm of row blockIdx.x (rmsnorm's arithmetic) written as pieces: n % 64 == 0, 256 threads,
// four consecutive values a thread and pass, so sixteen lanes hold a 64-block.
__global__ void __launch_bounds__(256) sgpu_pf_rms(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                   uint16_t* __restrict__ P, float* __restrict__ pd, int n, float eps) {
#pragma clang fp contract(off)
    __shared__ float red[4];
    const int tid = threadIdx.x;
    const size_t t = blockIdx.x;
    x += t * n;
    P += t * 3 * n;
    pd += t * (n / G);
    // the thread's first four values and gains stay in registers, both loaded before the reduction
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const int k4 = min(4 * tid, n - 4);
    const sgpu_f32x4 x4 = *reinterpret_cast<const sgpu_f32x4*>(x + k4);
    const u16x4 w4 = *reinterpret_cast<const u16x4*>(w + k4);
    float local = 4 * tid < n ? (x4[0] * x4[0] + x4[1] * x4[1]) + (x4[2] * x4[2] + x4[3] * x4[3]) : 0.0f;
    for (int k = 4 * tid + 1024; k < n; k += 1024) {
        const sgpu_f32x4 v = *reinterpret_cast<const sgpu_f32x4*>(x + k);
        local += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    }
    local = sgpu_group_sum<64>(local);
    if ((tid & 63) == 63) red[tid >> 6] = local;
    __syncthreads();
    const float ss = ((red[0] + red[1]) + (red[2] + red[3])) / (float)n;
    const float inv = 1.0f / __builtin_sqrtf(ss + eps);
    for (int k0 = 0; k0 < n; k0 += 1024) {                 // whole waves stay in the loop for the exchanges
        const int k = k0 + 4 * tid;
        const bool ok = k < n;
        float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t m = 0;
        if (ok) {
            const sgpu_f32x4 v = k0 == 0 ? x4 : *reinterpret_cast<const sgpu_f32x4*>(x + k);
            const u16x4 g = k0 == 0 ? w4 : *reinterpret_cast<const u16x4*>(w + k);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                y[e] = v[e] * inv * sgpu_h2f(g[e]);
                m = max(m, mag_bits(y[e]));
            }
        }
#pragma unroll
        for (int o = 1; o < 16; o *= 2) m = max(m, (uint32_t)__shfl_xor((int)m, o));
        if (!ok) continue;
        float up, down;
        block_scale(m, up, down);
        f16x4 p0, p1, p2;
        split3(y, up, p0, p1, p2);
        *reinterpret_cast<f16x4*>(P + k) = p0;
        *reinterpret_cast<f16x4*>(P + n + k) = p1;
        *reinterpret_cast<f16x4*>(P + 2 * n + k) = p2;
        if (tid % 16 == 0) pd[k / G] = down;
    }
}

}  // extern "C"

#define SGPU_PF_ATTN(HD)                                                                                              \
    extern "C" __global__ void __launch_bounds__(256, (HD) <= 64 ? 2 : 1) sgpu_pf_attn##HD(                                               \
        const float* __restrict__ qkv, const float* __restrict__ kc, const float* __restrict__ vc,                    \
        float* __restrict__ out, uint16_t* __restrict__ P, float* __restrict__ pd, int pos0, int T, int NH, int NKV,   \
        float scale, int QKVD) {                                                                                      \
        pf_attn<HD>(qkv, kc, vc, out, P, pd, pos0, T, NH, NKV, scale, QKVD);                                           \
    }
SGPU_PF_ATTN(32)
SGPU_PF_ATTN(64)
SGPU_PF_ATTN(128)

#define SGPU_PF_MM(TF, NF)                                                                                            \
    extern "C" __global__ void __launch_bounds__(256, 2) sgpu_pf_mm_##TF##NF(                                         \
        const uint16_t* __restrict__ W, const uint16_t* __restrict__ X, const float* __restrict__ xd,                 \
        const float* __restrict__ bias, float* __restrict__ Y, int K, int N, int T, int S, float* __restrict__ ws,    \
        unsigned* __restrict__ cnt, int accum) {                                                                      \
        pf_mm<TF, NF, EPI_STORE>(W, X, xd, bias, Y, nullptr, nullptr, K, N, T, S, ws, cnt, accum);                    \
    }
// 64 tokens and 128 SwiGLU columns a block.  128 tokens a block were slower at every prompt length
// (Qwen2.5-0.5B: 36 us against 53 at 500 rows, 151 against 156 at 3001): a CU holds two blocks
// of either, and the smaller one's step waits for 56 KB instead of 80.
extern "C" __global__ void __launch_bounds__(256, 2) sgpu_pf_gateup(
    const uint16_t* __restrict__ W, const uint16_t* __restrict__ X, const float* __restrict__ xd,
    uint16_t* __restrict__ P, float* __restrict__ pd, int K, int N, int T) {
    pf_mm<1, 4, EPI_SWIGLU>(W, X, xd, nullptr, nullptr, P, pd, K, N, T, 1, nullptr, nullptr, 0);
}
SGPU_PF_MM(1, 1)
SGPU_PF_MM(1, 2)
SGPU_PF_MM(2, 2)
