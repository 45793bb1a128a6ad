// sgpu_pieces.hip -- the large fp32 SGEMM on the bf16 matrix cores (gfx950).
//
// C = A B (row-major fp32) for problems of many 128x128 tiles.  The fp32 matrix instructions
// reach 157 TFLOP/s, and the members built on them run at 94% of that; bf16 ones are sixteen
// times as fast.  Every operand is cut into three bf16 pieces x = p0 + p1 + p2 (8 + 8 + 8 mantissa
// bits, the first two rounded to nearest, the third what is left), and the product is the sum of the
// six piece products p_i q_j with i + j <= 2.  |p1| <= 2^-8 |x| and |p2| <= 2^-17 |x|, so the three left
// out are at most 2^-24 of |x y|, what rounding a product to fp32 may take (rms 0.09 x 2^-24; products
// of random operands, each rounded once more at the end: 0.433 x 2^-24 rms and 1.70 at most, where
// one fp32 rounding has 0.424 and 1.0).  A product of pieces is exact in the fp32 accumulators.  p0 q0
// has accumulators of its own and the five small products share a second set, so the long sum is
// rounded once per 32 k: sums of many terms end closer to the exact ones than fp32 FMA chains do
// (4096^3 3.8e-7 against 5.7e-7), those of a single term up to 2 x 2^-24 away.  All eight that reach
// 2^-32 would cost 24% at 4096^3 (748 us against 602) and leave that error as it is.
//
// bf16 pieces end at 2^-133 (their subnormals count), so numbers below 2^-110 may lose bits that fp32
// keeps, and the largest round up to infinity.  A wave's part of a tile is computed again on the fp32
// matrix cores where it holds
//  * a sum that came out non-finite (an infinity, a NaN, an operand that rounded up to infinity);
//  * an element whose row of A or column of B lost bits, if it is below K 2^-108 times the other
//    operand's largest magnitude there: what was lost, 2^-133 a number, could pass 2^-25 of it;
//  * an element whose row and column are nonzero with the product of their largest magnitudes below
//    2^-110 (products of pieces end at 2^-149).
// A product all of which is computed again: 2048^3 110 -> 285-308 us (fp32 members 151), 4096^3 0.67 ->
// 1.9-2.1 ms (1.1); with one NaN in A 180 us and 1.13 ms.  By a serial dot product per element 2048^3
// took 12.2 ms and 0.8.
#include "sgpu_device.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int TM = 128, KS = 32;                       // tile rows, k per step

template <bool V>
struct bool_c {
    constexpr operator bool() const { return V; }
};

// The three pieces of two numbers, packed: two rounded to nearest, then the upper halves of what is
// left (8 bits at most), which one v_perm takes for two numbers.  What that drops (numbers below
// 2^-110 only) is seen in the lower halves.
__device__ __forceinline__ void cut2(float x0, float x1, uint32_t (&p)[3], uint32_t& lost) {
    p[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x0, x1}, bf16x2));
    x0 -= __uint_as_float(p[0] << 16);
    x1 -= __uint_as_float(p[0] & 0xffff0000u);
    p[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x0, x1}, bf16x2));
    x0 -= __uint_as_float(p[1] << 16);
    x1 -= __uint_as_float(p[1] & 0xffff0000u);
    p[2] = __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
    lost |= __float_as_uint(x0) | __float_as_uint(x1);
}
constexpr float kTiny = 0x1p-55f;                      // rows and columns from here on need no look at their products
__device__ __forceinline__ float max3abs(float m, float a, float b) { return fmaxf(fmaxf(m, fabsf(a)), fabsf(b)); }

// The wave's part of a tile again on the fp32 matrix cores, from memory: a points at the lane's first
// row of A (its others 16 rows on), b at its first column of B.  Lane quarter q takes k 4 q.. of each
// 16 (the k order within an MFMA is free), so operands are whole vectors; the next 16 k are loaded under
// this one's MFMAs.
template <int NJ>
__device__ __forceinline__ void fp32_tile(const float* __restrict__ a, const float* __restrict__ b, int K, int N, int quarter,
                                          f32x4 (&acc)[4][NJ]) {
    typedef float rowv __attribute__((ext_vector_type(NJ)));
    typedef float rowv_a4 __attribute__((ext_vector_type(NJ), aligned(4)));
    a += 4 * quarter;
    b += (size_t)(4 * quarter) * N;
    f32x4 av[2][4], sum[4][NJ];
    rowv bv[2][4];
    // slice s of 16 k; the last starts at K - 16 (K >= 32), its k already summed are set to zero
    auto load = [&](int s, int u) __attribute__((always_inline)) {
        const int k = min(16 * s, K - 16);
#pragma unroll
        for (int i = 0; i < 4; i++) av[u][i] = *reinterpret_cast<const sgpu_f32x4_a4*>(a + (size_t)(16 * i) * K + k);
#pragma unroll
        for (int t = 0; t < 4; t++) bv[u][t] = *reinterpret_cast<const rowv_a4*>(b + (size_t)(k + t) * N);
    };
    auto mul = [&](int s, int u) __attribute__((always_inline)) {
        const int done = 16 * s - (K - 16);
        if (done > 0) {
#pragma unroll
            for (int t = 0; t < 4; t++)
                if (4 * quarter + t < done) {
#pragma unroll
                    for (int i = 0; i < 4; i++) av[u][i][t] = 0.0f;
#pragma unroll
                    for (int j = 0; j < NJ; j++) bv[u][t][j] = 0.0f;
                }
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u][i][t], bv[u][t][j], sum[i][j], 0, 0, 0);
    };
    const int ns = (K + 15) / 16;
    load(0, 0);
    for (int s0 = 0; s0 < ns; s0 += 16) {                  // sums of 256 k, added up
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) sum[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int s = s0; s < min(s0 + 16, ns); s += 2) {
            load(s + 1, 1);
            mul(s, 0);
            load(s + 2, 0);
            mul(s + 1, 1);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = s0 == 0 ? sum[i][j] : acc[i][j] + sum[i][j];
    }
}

// Bound: the matrix cores.  A block of 2x4 waves computes a tile of 128 x 64 NJ, a wave 64 x 16 NJ of
// it in 16x16 tiles.  Operands pass through two LDS buffers of 32 k: while the matrix cores run on
// one, the waves cut the next 32 k (read into registers half a step or more earlier) into the
// other, their VALU work and LDS writes dealt out between the MFMAs, so that a step has one
// barrier; two waves a SIMD fill each other's waits.  A's rows and B's columns hold their 32 k of
// a piece in 64 bytes (16-byte chunk c at c ^ (-(row / 4) % 4): a read serves lanes 0-3, 12-15, 20-23
// and 24-27 and the like together, and these then use all 64 banks).  B's column n is kept in LDS
// row n % NJ * 64 + n / NJ, so that a lane ends with NJ consecutive columns of C.
// Measured at 4096^3: 8 waves and 128x256 590-602 us, 128x128 691; 4 waves and 128x128 822; one LDS
// buffer and two blocks of 4 waves a CU 672; the fp32 members 926.  With chunk order c ^ (row / 4 % 4),
// which puts two of a read's rows on the same banks, 610 and 724.
// A last row or column of tiles that would pass M or N ends at M or N and is stored from its first
// new row or column on: the tile before it owns the overlap (one of the two may be split over K and
// the other not, whose sums round differently).  A last step that would pass K starts at K - 32 with
// the k already summed set to zero: no load needs a bound.  Operands of any float alignment.
// The first `full` tiles are one block each; those that are left, too few for a round of all CUs, are
// split over S blocks of consecutive slices each, whose sums meet by the hand-off of
// sgpu_device.h: ws holds one record of 128 * TN + 128 + TN floats per block (its tile, then its
// rows' and columns' largest magnitudes), cnt one zeroed counter per split tile.
// Preconditions (launcher): M >= 128, N >= 64 NJ, K >= 32, 4-byte aligned operands, blockDim 512,
// 1 <= S <= slices of 32 k, grid = full + (tiles - full) * S.
template <int NJ>
__device__ __forceinline__ void sgemm_pieces(const float* __restrict__ A, const float* __restrict__ B,
                                             float* __restrict__ C, int M, int N, int K, int full, int S,
                                             float* __restrict__ ws, unsigned* __restrict__ cnt) {
    constexpr int TN = 64 * NJ, REC = TM * TN + TM + TN;
    typedef float rowv __attribute__((ext_vector_type(NJ)));
    typedef float rowv_a4 __attribute__((ext_vector_type(NJ), aligned(4)));
    __shared__ __attribute__((aligned(1024))) uint16_t as[2][3 * TM * KS], bs[2][3 * TN * KS];
    __shared__ int look;                                   // some row or column lost bits or is tiny
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, quarter = lane >> 4, wm = wave >> 2, wn = wave & 3;
    // Blocks are dealt round-robin to the 8 XCDs: of the unsplit tiles each XCD takes a contiguous
    // run, eight tile rows by all columns at a time, so that its blocks share operands in its L2.
    const int ntm = (M + TM - 1) / TM, ntn = (N + TN - 1) / TN, rest = ntm * ntn - full, xcd = blockIdx.x % 8;
    const bool whole = (int)blockIdx.x < full;
    const int u = (int)blockIdx.x - full, part = whole ? 0 : u % rest, sp = whole ? 0 : u / rest;
    const int tile = whole ? xcd * (full / 8) + min(xcd, full % 8) + blockIdx.x / 8 : full + part;
    const int band = tile / (8 * ntn), bm = min(8, ntm - 8 * band), in = tile - band * 8 * ntn;
    const int mt = (8 * band + in % bm) * TM, nt = (in / bm) * TN;         // first row and column of its own
    const int m0 = min(mt, M - TM), n0 = min(nt, N - TN);

    // A thread's part of a slice: A rows r and r + 64, k 4 q..; B rows k 4 q + i, columns NJ r...
    const int r = tid >> 3, q = tid & 7;
    const float* ap = A + (size_t)(m0 + r) * K + 4 * q;
    const float* bp = B + (size_t)(4 * q) * N + n0 + NJ * r;
    f32x4 av[2];
    rowv bv[4];
    auto load_a = [&](int s) __attribute__((always_inline)) {
        const int k0 = min(KS * s, K - KS);
#pragma unroll
        for (int i = 0; i < 2; i++) av[i] = *reinterpret_cast<const sgpu_f32x4_a4*>(ap + (size_t)(64 * i) * K + k0);
    };
    auto load_b = [&](int s) __attribute__((always_inline)) {
        const int k0 = min(KS * s, K - KS);
#pragma unroll
        for (int i = 0; i < 4; i++) bv[i] = *reinterpret_cast<const rowv_a4*>(bp + (size_t)(k0 + i) * N);
    };
    // k of slice s that are summed already: set to zero
    auto mask = [&](int s) __attribute__((always_inline)) {
        const int done = KS * s - (K - KS);
        if (done <= 0) return;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (4 * q + e >= done) continue;
            av[0][e] = av[1][e] = 0.0f;
#pragma unroll
            for (int c = 0; c < NJ; c++) bv[e][c] = 0.0f;
        }
    };
    uint32_t lost_a = 0, lost_b = 0;
    float amax[2] = {0.0f, 0.0f}, bmax[NJ];
#pragma unroll
    for (int c = 0; c < NJ; c++) bmax[c] = 0.0f;
    const int wo = r * KS + 8 * ((q >> 1) ^ (-(r >> 2) & 3)) + 4 * (q & 1);
    auto cut_a = [&](int buf, int i) __attribute__((always_inline)) {
        uint32_t lo[3], hi[3];
        cut2(av[i][0], av[i][1], lo, lost_a);
        cut2(av[i][2], av[i][3], hi, lost_a);
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<u32x2*>(as[buf] + wo + (p * TM + 64 * i) * KS) = u32x2{lo[p], hi[p]};
        amax[i] = max3abs(max3abs(amax[i], av[i][0], av[i][1]), av[i][2], av[i][3]);
    };
    auto cut_b = [&](int buf, int c) __attribute__((always_inline)) {
        uint32_t lo[3], hi[3];
        cut2(bv[0][c], bv[1][c], lo, lost_b);
        cut2(bv[2][c], bv[3][c], hi, lost_b);
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<u32x2*>(bs[buf] + wo + (p * TN + 64 * c) * KS) = u32x2{lo[p], hi[p]};
        bmax[c] = max3abs(max3abs(bmax[c], bv[0][c], bv[1][c]), bv[2][c], bv[3][c]);
    };
    f32x4 acc[4][NJ], low[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = low[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int ch = 8 * (quarter ^ (-(l16 >> 2) & 3));
    const int aro = (64 * wm + l16) * KS + ch, bro = (16 * wn + l16) * KS + ch;

    const int ns = (K + KS - 1) / KS;                      // this block's slices: s0..nk-1
    const int s0 = whole ? 0 : sp * ns / S, nk = whole ? ns : (sp + 1) * ns / S;
    // Step s on LDS buffer `buf`: slice s + 1 cut into the other one, slice s + 2 read.  What is cut past
    // the block's last slice is not used.
    auto step = [&](int s, int buf) __attribute__((always_inline)) {
        mask(s + 1);
        bf16x8 b[NJ][3];
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int p = 0; p < 3; p++) b[j][p] = *reinterpret_cast<const bf16x8*>(bs[buf] + bro + (p * TN + 64 * j) * KS);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            bf16x8 a[3];
#pragma unroll
            for (int p = 0; p < 3; p++) a[p] = *reinterpret_cast<const bf16x8*>(as[buf] + aro + (p * TM + 16 * i) * KS);
            constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int t = 0; t < 6; t++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    f32x4& d = t < 5 ? low[i][j] : acc[i][j];
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[pa[t]], b[j][pb[t]], d, 0, 0, 0);
                }
            if (i < 2) {
#pragma unroll
                for (int c = 0; c < NJ / 2; c++) cut_b(buf ^ 1, NJ / 2 * i + c);
                if (i == 1) load_b(s + 2);
            } else {
                cut_a(buf ^ 1, i - 2);
                if (i == 3) load_a(s + 2);
            }
        }
        __syncthreads();
    };
    if (tid == 0) look = 0;
    load_a(s0);
    load_b(s0);
    mask(s0);
#pragma unroll
    for (int c = 0; c < NJ; c++) cut_b(0, c);
    load_b(s0 + 1);
    cut_a(0, 0);
    cut_a(0, 1);
    load_a(s0 + 1);
    __syncthreads();
    for (int s = s0; s < nk; s += 2) {
        step(s, 0);
        if (s + 1 < nk) step(s + 1, 1);
    }

    // The largest magnitude of each of the tile's rows and columns, through LDS; negative where bits
    // were lost.
    float* const rmax = reinterpret_cast<float*>(as[0]);   // 128 rows, then TN columns
    auto put_max = [&](int at, float m, uint32_t lost) __attribute__((always_inline)) {
#pragma unroll
        for (int o = 1; o < 8; o *= 2) m = fmaxf(m, __shfl_xor(m, o));
        lost = (lost & 0xffffu) != 0u;
        if (q == 0) rmax[at] = lost ? -m : m;
        if (lost || (m < kTiny && m > 0.0f)) look = 1;
    };
#pragma unroll
    for (int o = 1; o < 8; o *= 2) {
        lost_a |= (uint32_t)__shfl_xor((int)lost_a, o);
        lost_b |= (uint32_t)__shfl_xor((int)lost_b, o);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) put_max(r + 64 * i, amax[i], lost_a);
#pragma unroll
    for (int c = 0; c < NJ; c++) put_max(TM + NJ * r + c, bmax[c], lost_b);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] += low[i][j];
    __syncthreads();
    if (!whole && S > 1) {
        float* const rec = ws + (size_t)(sp * rest + part) * REC;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    __hip_atomic_store(rec + ((i * NJ + j) * 4 + e) * 512 + tid, acc[i][j][e], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        if (tid < TM + TN)
            __hip_atomic_store(rec + TM * TN + tid, rmax[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);                     // this wave's partial stores are acknowledged
        int& last_s = *reinterpret_cast<int*>(bs[0]);
        __syncthreads();
        if (tid == 0) {
            last_s = __hip_atomic_fetch_add(cnt + part, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
            if (last_s) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // before the others' partials
        }
        __syncthreads();
        if (!last_s) return;
        // all parts in order, this block's own among them; a tile's (narrow: two tiles') loads are
        // issued before the first add
        constexpr int U = 4 / NJ;
        float big = 0.0f;
        bool lost = false;
        for (int s2 = 0; s2 < S; s2 += U) {
            f32x4 v[U][4][NJ];
            float m[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float* src = ws + (size_t)(min(s2 + u, S - 1) * rest + part) * REC;
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            v[u][i][j][e] = __hip_atomic_load(src + ((i * NJ + j) * 4 + e) * 512 + tid, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT);
                m[u] = tid < TM + TN ? __hip_atomic_load(src + TM * TN + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (s2 + u >= S) break;
                big = fmaxf(big, fabsf(m[u]));
                lost |= m[u] < 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) acc[i][j] = s2 + u == 0 ? v[u][i][j] : acc[i][j] + v[u][i][j];
            }
        }
        if (tid < TM + TN) rmax[tid] = lost ? -big : big;
        if (lost || (big < kTiny && big > 0.0f)) look = 1;
        if (tid == 0) __hip_atomic_store(cnt + part, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
    }
    // Accumulator e of tile (i, j): row 64 wm + 16 i + 4 quarter + e, column NJ (16 wn + l16) + j.
    const int lc = NJ * (16 * wn + l16), n = n0 + lc;
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) top = max(top, __float_as_uint(acc[i][j][e]) & 0x7fffffffu);
    bool again = top >= 0x7f800000u;
    if (look) {
        const float least = (float)K * 0x1p-108f;
        for (int j = 0; j < NJ; j++) {
            const float cm = rmax[TM + lc + j], ca = fabsf(cm);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float rm = rmax[64 * wm + 16 * i + 4 * quarter + e], ra = fabsf(rm);
                    float v = 0.0f;
#pragma unroll
                    for (int jj = 0; jj < NJ; jj++) v = jj == j ? fabsf(acc[i][jj][e]) : v;
                    again |= (rm < 0.0f && v < least * ca) || (cm < 0.0f && v < least * ra) ||
                             (ra > 0.0f && ca > 0.0f && ra * ca < 0x1p-110f);
                }
        }
    }
    if (__any(again)) fp32_tile<NJ>(A + (size_t)(m0 + 64 * wm + l16) * K, B + n, K, N, quarter, acc);
    auto store = [&](auto shifted) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = m0 + 64 * wm + 16 * i + 4 * quarter + e;
                if (shifted && m < mt) continue;
                rowv v;
#pragma unroll
                for (int j = 0; j < NJ; j++) v[j] = acc[i][j][e];
                float* const c = C + (size_t)m * N + n;
                if (!shifted || n >= nt) {
                    *reinterpret_cast<rowv_a4*>(c) = v;
                } else {
#pragma unroll
                    for (int j = 0; j < NJ; j++)
                        if (n + j >= nt) c[j] = v[j];
                }
            }
    };
    if (m0 == mt && n0 == nt) store(bool_c<false>{});
    else store(bool_c<true>{});
}

}  // namespace

extern "C" __global__ void __launch_bounds__(512) sgpu_sgemm_pieces(const float* __restrict__ A, const float* __restrict__ B,
                                                                    float* __restrict__ C, int M, int N, int K, int full,
                                                                    int S, float* __restrict__ ws,
                                                                    unsigned* __restrict__ cnt) {
    sgemm_pieces<2>(A, B, C, M, N, K, full, S, ws, cnt);
}
extern "C" __global__ void __launch_bounds__(512) sgpu_sgemm_pieces_wide(const float* __restrict__ A,
                                                                         const float* __restrict__ B, float* __restrict__ C,
                                                                         int M, int N, int K, int full, int S,
                                                                         float* __restrict__ ws,
                                                                         unsigned* __restrict__ cnt) {
    sgemm_pieces<4>(A, B, C, M, N, K, full, S, ws, cnt);
}
