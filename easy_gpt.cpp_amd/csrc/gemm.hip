// out[m, n] = sum_k x[m, k] * w[n, k] + bias[n]: the linear layer y = x W^T + b with W stored [out, in]
// (/root/reference/src/ops.cpp:101-118).
//
// gemm_tiled: plain FMA tiles in float32 arithmetic for every element type, the fallback for sizes the MFMA kernels refuse.
// gemm_f32_mfma, gemm_f32_rows: the float32 product on the matrix cores, for few rows and for many.
#include "api.h"
#include "common.h"

namespace egpt {

constexpr int BM = 64, BN = 64, BK = 16;

template <typename TIn, typename TOut>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(const TIn* __restrict__ x, const TIn* __restrict__ w,
                                                         const TIn* __restrict__ bias, TOut* __restrict__ out,
                                                         int m, int n, int k) {
    __shared__ float xs[BK][BM + 4];
    __shared__ float ws[BK][BN + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int ty = tid / 16, tx = tid % 16;  // 16 x 16 threads, 4 x 4 outputs each
    float acc[4][4] = {};
    for (int k0 = 0; k0 < k; k0 += BK) {
        // each thread loads 4 elements of each tile: tile row = idx / BK, column = idx % BK
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + i * 256;
            const int r = idx / BK, c = idx % BK;
            const int gm = m0 + r, gn = n0 + r, gk = k0 + c;
            xs[c][r] = (gm < m && gk < k) ? to_float(x[static_cast<size_t>(gm) * k + gk]) : 0.f;
            ws[c][r] = (gn < n && gk < k) ? to_float(w[static_cast<size_t>(gn) * k + gk]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int gm = m0 + ty * 4 + i;
        if (gm >= m) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int gn = n0 + tx * 4 + j;
            if (gn >= n) continue;
            const float v = acc[i][j] + (bias ? to_float(bias[gn]) : 0.f);
            out[static_cast<size_t>(gm) * n + gn] = from_float<TOut>(v);
        }
    }
}

template <typename TIn, typename TOut>
int launch_tiled(const void* x, const void* w, const void* bias, void* out, int m, int n, int k, hipStream_t s) {
    dim3 grid((n + BN - 1) / BN, (m + BM - 1) / BM);
    gemm_tiled_kernel<TIn, TOut><<<grid, 256, 0, s>>>(static_cast<const TIn*>(x), static_cast<const TIn*>(w),
                                                      static_cast<const TIn*>(bias), static_cast<TOut*>(out), m, n,
                                                      k);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

// ----------------------------------------------------------------------------- float32 on the matrix cores
// The float32 product on the bfloat16 matrix instructions, with no less than float32's precision: every operand is the sum of three
// bfloat16 numbers, 2^24 x = h + m + l, each the nearest to what the ones before leave (8 + 8 + 8 bits: nothing is left), and of
// the nine products the six largest are added up; the three others are below 2^-25 of the product and of either sign.  The
// power of two keeps the parts of the smallest numbers in bfloat16's range: the last bit of any float32 number, 2^-149, becomes
// 2^-125, while without it the parts of 2^-116 lose bits (an error of 2.3e-6 instead of 1.1e-7, and 2.3e-3 at 2^-126).  The
// six products of a block of 32 values of k are one chain of v_mfma_f32_16x16x32_bf16 that begins at zero, and the block's sum
// is taken back by 2^48 and added to the element's in float32.  Error against 64 bits (2-norm, k = 896 / 4,864): 1.1e-7 / 2.4e-7,
// with v_mfma_f32_16x16x4_f32, which took its operands as they are and rounded after every fourth product, 5.4e-7 / 1.25e-6; with
// one chain over all blocks 4.5e-7 / 1.1e-6.  (The power of two is a product per operand: nothing with up to 64 rows, 5 to 8 % of
// a tile of 128 rows: 1,811 and 4,096 rows of 9,728 x 896 in 235 and 480 us, 219 and 452 without it.)
// Values that have no such three parts (infinities, NaN, from 2^104 on) and block sums beyond 2^80 leave an element that is no
// finite number.  A wavefront that holds one adds its tile up again with v_mfma_f32_16x16x4_f32, which takes
// float32 operands whole, and takes those elements from there.  (1,811 rows of 9,728 x 896, us: 251, 280 with one row of NaN,
// 737 with nothing else; 8 rows 8.7 and 15.0.)
//
// Every element of the result is the same sequence of operations whatever m is and wherever its row lies in x, in all
// kernels here: block after block of 32 values within a range of k, ranges of k one after the other.  So a token's values do not
// depend on what else is in the batch, to the bit.
constexpr int kBlockF = 32;                   // values of k per block
constexpr int kStepF = 64;                    // ranges of k are multiples of this
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 f_bf16x8;

constexpr float kUp = 0x1p24f;                // what operands are multiplied by
constexpr float kDown = 0x1p-48f;             // and block sums

struct Parts {                                // eight values of k, times kUp, as three bfloat16 numbers each
    f_bf16x8 h, m, l;
};
typedef __attribute__((ext_vector_type(2))) __bf16 f_bf16x2;
// What is left of two values when a pair of bfloat16 numbers is taken away: one instruction each (a dot product with -1 and
// 0, exact here) instead of a conversion and a subtraction.  The constants stand in registers: as an inline constant
// -1.0 would be float32's, whose bfloat16 pair is (0, -1).
__device__ __forceinline__ void take_away(f_bf16x2 pair, float& a, float& b) {
#if defined(__HIP_DEVICE_COMPILE__)
    unsigned low = 0x0000bf80u, high = 0xbf800000u;
    asm("" : "+s"(low), "+s"(high));
    a = __builtin_amdgcn_fdot2_f32_bf16(pair, __builtin_bit_cast(f_bf16x2, low), a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(pair, __builtin_bit_cast(f_bf16x2, high), b, false);
#endif
}
__device__ __forceinline__ Parts split_parts(const f32x4& a, const f32x4& b) {
    Parts p;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        float x = kUp * (i < 4 ? a[i] : b[i - 4]), y = kUp * (i < 4 ? a[i + 1] : b[i - 3]);
        f_bf16x2 h{static_cast<__bf16>(x), static_cast<__bf16>(y)};
        take_away(h, x, y);
        f_bf16x2 m{static_cast<__bf16>(x), static_cast<__bf16>(y)};
        take_away(m, x, y);
        p.h[i] = h[0], p.h[i + 1] = h[1];
        p.m[i] = m[0], p.m[i + 1] = m[1];
        p.l[i] = static_cast<__bf16>(x), p.l[i + 1] = static_cast<__bf16>(y);
    }
    return p;
}
// The sums of N blocks, w[j] with x[j] (or with x[0], X = 1), as chains that go forward side by side: a product waits for the
// one before it in its chain, not for its neighbours.
template <int N, int X>
__device__ __forceinline__ void block_sums(const Parts* w, const Parts* x, f32x4* t) {
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].l, x[j % X].h, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].h, x[j % X].l, t[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].m, x[j % X].m, t[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].m, x[j % X].h, t[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].h, x[j % X].m, t[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].h, x[j % X].h, t[j], 0, 0, 0);
}
// The sums of N tiles of 16 x 16 elements over values [k0, k1) of k (multiples of four) without parts, straight from memory: x and
// w[j] are the lane's rows li of the operands; v_mfma_f32_16x16x4_f32, sixteen values of k after the other, the i-th instruction of
// each sixteen the i-th values of the four lanes' quadruples.
template <int N>
__device__ __forceinline__ void whole_sums(const float* x, const float* const (&w)[N], int lg, int k0, int k1, f32x4 (&t)[N]) {
    const f32x4 none{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < N; ++j) t[j] = none;
#pragma unroll 1
    for (int b = k0; b < k1; b += 16) {
        const int at = b + lg * 4;
        const f32x4 xv = at < k1 ? *reinterpret_cast<const f32x4*>(x + at) : none;
        f32x4 wv[N];
#pragma unroll
        for (int j = 0; j < N; ++j) wv[j] = at < k1 ? *reinterpret_cast<const f32x4*>(w[j] + at) : none;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < N; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][i], xv[i], t[j], 0, 0, 0);
    }
}
__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }
// Whether all of a wavefront's elements of N tiles are finite numbers.
template <int N>
__device__ __forceinline__ bool all_finite(const f32x4 (&t)[N]) {
    bool good = true;
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) good &= finite(t[j][v]);
    return __all(good);
}
// In place of the elements that are no finite number those of whole_sums.
template <int N>
__device__ __forceinline__ void mend(const float* x, const float* const (&w)[N], int lg, int k0, int k1, f32x4 (&t)[N]) {
    if (all_finite(t)) return;
    f32x4 whole[N];
    whole_sums(x, w, lg, k0, k1, whole);
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (!finite(t[j][v])) t[j][v] = whole[j][v];
}

// Up to 64 rows of x to a workgroup (further groups of rows: blockIdx.z).  A wavefront owns 16 rows of w (16 columns of the
// result) and streams them once, as they are (four steps of 64 values ahead: with few rows the kernel is a stream of w, and a
// stream one step deep was a chain of round trips, 1.1 TB/s on a 17 MB matrix), and splits them in registers; the rows of x
// are split on their way to LDS, CH steps at a time, and shared by the wavefronts: four steps for up to 16 rows, where a barrier
// a step was a quarter of the time of a short range, one for more rows, whose LDS would keep workgroups off a CU.  A lane's four
// values of a row of the result are one store (as four they cost 64 rows of 9,728 columns 2.6 us of 25.7).  The k range may be
// split over workgroups (blockIdx.y) into partial sums out[split][m][n].
// us for 8 / 64 rows, each with the ranges that the callers take: 1,152 x 896 4.8 / 8.3, 9,728 x 896 11.3 / 23.1, 896 x 4,864 10.1 /
// 17.7, 151,936 x 896 109 / 184; with v_mfma_f32_16x16x4_f32 4.8 / 8.5, 12.9 / 23.6, 10.6 / 18.5 and 114 / 210.

template <int MT, int CH, int NW>
__global__ __launch_bounds__(NW * 64) void gemm_f32_mfma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ bias, float* __restrict__ out,
                                                            int m, int n, int k, int steps_per_split) {
    __shared__ __attribute__((aligned(16))) __bf16 xs[2][3][MT * 16][CH * kStepF + 8];   // (16 bytes of padding to a row)
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int li = lane % 16, lg = lane / 16;
    const int split = blockIdx.y;
    const int m0 = blockIdx.z * 64;                       // first row of this group
    const int n0 = (blockIdx.x * NW + wave) * 16;
    const int total_steps = (k + kStepF - 1) / kStepF;
    const int step_begin = split * steps_per_split;
    const int step_end = min(total_steps, step_begin + steps_per_split);
    // lane (li, lg) takes eight values of row li per block of 32: 128 contiguous bytes of each row an instruction pair
    const float* wp = w + static_cast<size_t>(min(n0 + li, n - 1)) * k + lg * 8;
    auto load_w = [&](f32x4* av, int step) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int at = step * kStepF + q / 2 * kBlockF + q % 2 * 4;
            av[q] = at + lg * 8 < k ? *reinterpret_cast<const f32x4*>(wp + at) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // eight values of a row of x per thread and load: MT * 16 rows x 8 * CH pieces
    constexpr int PC = CH * 8, XP = MT * 16 * PC, XN = (XP + NW * 64 - 1) / (NW * 64);
    constexpr int XS = CH == 1 ? 2 : 1;                   // stagings on their way
    f32x4 xr[XS][XN][2];
    auto x_load = [&](int set, int step) {
#pragma unroll
        for (int j = 0; j < XN; ++j) {
            const int c = tid + j * NW * 64, r = m0 + c / PC, kc = step * kStepF + c % PC * 8;
#pragma unroll
            for (int u = 0; u < 2; ++u)
                xr[set][j][u] = (c < XP && r < m && kc + u * 4 < k)
                                    ? *reinterpret_cast<const f32x4*>(x + static_cast<size_t>(r) * k + kc + u * 4)
                                    : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    auto x_store = [&](int set, int buf) {
#pragma unroll
        for (int j = 0; j < XN; ++j) {
            const int c = tid + j * NW * 64;
            if (c >= XP) break;
            const Parts p = split_parts(xr[set][j][0], xr[set][j][1]);
            *reinterpret_cast<f_bf16x8*>(&xs[buf][0][c / PC][c % PC * 8]) = p.h;
            *reinterpret_cast<f_bf16x8*>(&xs[buf][1][c / PC][c % PC * 8]) = p.m;
            *reinterpret_cast<f_bf16x8*>(&xs[buf][2][c / PC][c % PC * 8]) = p.l;
        }
    };
    f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int kAhead = 4;
    f32x4 a[kAhead][4];     // (a native vector type: arrays of it stay in registers across the loop's back edge)
    x_load(0, step_begin);
    if (XS > 1 && step_begin + CH < step_end) x_load(XS - 1, step_begin + CH);
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
        if (step_begin + u < step_end) load_w(a[u], step_begin + u);
    x_store(0, 0);
    if (step_begin + XS * CH < step_end) x_load(0, step_begin + XS * CH);
    __syncthreads();
    for (int step0 = step_begin; step0 < step_end; step0 += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int step = step0 + u;
            if (step >= step_end) break;
            // (kAhead is a multiple of CH; of 2 * CH it is not where a staging is four steps: the count of stagings then)
            const int buf = CH * 2 <= kAhead ? u / CH & 1 : (step0 - step_begin) / CH & 1;
            const int in = u % CH * kStepF;
            const Parts wv[2] = {split_parts(a[u][0], a[u][1]), split_parts(a[u][2], a[u][3])};
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                Parts xv[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    xv[q].h = *reinterpret_cast<const f_bf16x8*>(&xs[buf][0][t * 16 + li][in + q * kBlockF + lg * 8]);
                    xv[q].m = *reinterpret_cast<const f_bf16x8*>(&xs[buf][1][t * 16 + li][in + q * kBlockF + lg * 8]);
                    xv[q].l = *reinterpret_cast<const f_bf16x8*>(&xs[buf][2][t * 16 + li][in + q * kBlockF + lg * 8]);
                }
                f32x4 sums[2];
                block_sums<2, 2>(wv, xv, sums);
                acc[t] += kDown * sums[0];
                acc[t] += kDown * sums[1];
            }
            if (step + kAhead < step_end) load_w(a[u], step + kAhead);
            if ((u + 1) % CH == 0 && step + 1 < step_end) {
                const int set = (u + 1) & (XS - 1);
                x_store(set, buf ^ 1);
                if (step + 1 + XS * CH < step_end) x_load(set, step + 1 + XS * CH);
                __syncthreads();
            }
        }
    }
    // D layout: lane (li, lg) holds rows lg*4 + v of the 16 x 16 tile (an n index) at column li (an m index)
    const bool whole = n % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;   // four values are one store
    const float* const wrow[1] = {w + static_cast<size_t>(min(n0 + li, n - 1)) * k};
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int mm = m0 + t * 16 + li, nn = n0 + lg * 4;
        f32x4 sums[1] = {acc[t]};
        mend(x + static_cast<size_t>(min(mm, m - 1)) * k, wrow, lg, step_begin * kStepF, min(k, step_end * kStepF), sums);
        if (mm >= m || nn >= n) continue;
        f32x4 val = sums[0];
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (bias && nn + v < n) val[v] += bias[nn + v];
        float* to = out + (static_cast<size_t>(split) * m + mm) * n + nn;
        if (whole) {
            *reinterpret_cast<f32x4*>(to) = val;
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (nn + v < n) to[v] = val[v];
        }
    }
}

// Many rows of x: tiles of 128 rows of x and 128 of w, both split on their way to LDS (a thread eight values of each a block, loaded
// two blocks ahead), eight wavefronts of 32 x 64.  A block's parts lie in LDS as rows of 64 bytes whose four pieces of 16
// bytes are exchanged by the row's number (piece p of row r in place p ^ (r / 2 & 3)), so that the lanes that read one
// piece of many rows hit different banks; two buffers, one barrier a block.
// With 64 rows of x the workgroup is half as large and a CU holds two (LDS, and up to 256 registers): 1,811 and 4,096 rows of 9,728 x
// 896 in 224 and 489 us, one to a CU 271 and 593 (each lane had more than 256 registers); with 128 rows 235 and 480.
// FOLD: a workgroup walks all ranges of k and adds their sums up in their order, which is what a reader of partial sums does:
// the same bits, without the partial sums' traffic.
// TAIL: k is no multiple of a block (its end is filled with zeros).
// GATED: w = [gate; up] of n rows each, and what leaves is act(x gate^T) * (x up^T), the bits that an activation kernel makes of the
// product: a wavefront's columns are 32 gates and the up columns of the same numbers.  1,811 rows of 9,728 x 896: 218 us and 21 for
// the activation kernel, 215 so (71 MB less written, 71 less read, and the activation under the other workgroup's products).
template <int WM, bool FOLD, bool TAIL, bool GATED>
__global__ __launch_bounds__(WM * 128) void gemm_f32_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ bias, float* __restrict__ out,
                                                            int m, int n, int k, int blocks_per_split, int act) {
    constexpr int TM = 2, TN = 4;                          // 16 x 16 tiles of a wavefront
    constexpr int BM = WM * 32, NT = WM * 128, WL = 512 / NT;   // rows of x; threads; pieces of w that a thread stages
    constexpr int kPartX = BM * 64, kPartW = 128 * 64;     // bytes of a part of an operand's block
    __shared__ __attribute__((aligned(128))) char lds[2][3 * (kPartX + kPartW)];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int li = lane % 16, lg = lane / 16;
    const int wm = wave % WM, wn = wave / WM;
    // a die gets a contiguous range of tiles, rows of x fastest
    constexpr int kCols = GATED ? 64 : 128;                // columns of the result
    const int mt = (m + BM - 1) / BM, tiles = mt * ((n + kCols - 1) / kCols);
    int tile = blockIdx.x;
    {
        const int q = tiles / 8, r = tiles % 8, d = tile % 8, i = tile / 8;
        tile = d * q + (d < r ? d : r) + i;
    }
    const int m0 = tile % mt * BM, n0 = tile / mt * kCols;
    auto w_row = [&](int r) {                              // the row of w that is row r of the tile (beyond the last one any)
        if (!GATED) return w + static_cast<size_t>(min(n0 + r, n - 1)) * k;
        return w + static_cast<size_t>(min(n0 + r / 64 * 32 + r % 32, n - 1) + (r % 64 < 32 ? 0 : n)) * k;
    };
    const int total = (k + kBlockF - 1) / kBlockF;
    const int first = FOLD ? 0 : blockIdx.y * blocks_per_split;
    const int last = FOLD ? total : min(total, first + blocks_per_split);
    // ---- staging: a thread's row and its eight values of k
    const int srow = tid / 4, piece = tid % 4;
    const float* xp = x + static_cast<size_t>(min(m0 + srow, m - 1)) * k + piece * 8;
    const float* wp[WL];
#pragma unroll
    for (int o = 0; o < WL; ++o) wp[o] = w_row(srow + o * (NT / 4)) + piece * 8;
    f32x4 raw[2][1 + WL][2];                               // [set][x, w ..][halves]
    auto load = [&](int set, int block) {                  // (beyond the last block the last one again, which nobody reads)
        const int at = min(block, last - 1) * kBlockF;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool in = !TAIL || at + piece * 8 + u * 4 < k;
            const int offset = in ? at + u * 4 : -piece * 8;
            raw[set][0][u] = *reinterpret_cast<const f32x4*>(xp + offset);
#pragma unroll
            for (int o = 0; o < WL; ++o) raw[set][1 + o][u] = *reinterpret_cast<const f32x4*>(wp[o] + offset);
            if (TAIL && !in)
#pragma unroll
                for (int o = 0; o < 1 + WL; ++o) raw[set][o][u] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    const int place = srow * 64 + (piece ^ (srow / 2 & 3)) * 16;          // (the same for srow + a multiple of 8)
    auto store = [&](int set, int buf) {
#pragma unroll
        for (int o = 0; o < 1 + WL; ++o) {
            const Parts p = split_parts(raw[set][o][0], raw[set][o][1]);
            char* to = lds[buf] + (o == 0 ? place : 3 * kPartX + place + (o - 1) * (NT / 4) * 64);
            constexpr int parts[2] = {kPartX, kPartW};
            *reinterpret_cast<f_bf16x8*>(to) = p.h;
            *reinterpret_cast<f_bf16x8*>(to + parts[o > 0]) = p.m;
            *reinterpret_cast<f_bf16x8*>(to + 2 * parts[o > 0]) = p.l;
        }
    };
    const int read_at = li * 64 + (lg ^ (li / 2 & 3)) * 16;
    auto piece_of = [&](const char* from) { return *reinterpret_cast<const f_bf16x8*>(from); };
    f32x4 acc[TM][TN], sum[FOLD ? TM : 1][FOLD ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (FOLD) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    const int row0 = m0 + wm * 32 + li, col0 = n0 + wn * (kCols / 2) + lg * 4;
    // the end of a range [b0, b1) of blocks: elements that are no finite number
    auto mend_range = [&](int b0, int b1) {
        const float* wrow[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) wrow[j] = w_row(wn * 64 + j * 16 + li);
#pragma unroll
        for (int i = 0; i < TM; ++i) mend(x + static_cast<size_t>(min(row0 + i * 16, m - 1)) * k, wrow, lg, b0 * kBlockF, min(k, b1 * kBlockF), acc[i]);
    };
    load(0, first);
    load(1, first + 1);
    store(0, 0);
    load(0, first + 2);
    int range_begin = first, in_range = 0;
#pragma unroll 1
    for (int b0 = first; b0 < last; b0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int b = b0 + u;
            if (b >= last) break;
            __syncthreads();                               // block b is in buffer u, buffer 1 - u has been read
            // block b + 1 is split by one of the two wavefronts of a SIMD before its products and by the other behind them:
            // the vector unit and the matrix cores work at the same time
            if (wn == 0) {
                store(1 - u, 1 - u);
                load(1 - u, b + 3);
            }
            const char* xs = lds[u] + wm * 2048 + read_at;
            const char* ws = lds[u] + 3 * kPartX + wn * 4096 + read_at;
            Parts wv[TN], xv[TM];
#pragma unroll
            for (int j = 0; j < TN; ++j) wv[j].h = piece_of(ws + j * 1024);
            xv[0].h = piece_of(xs);
#pragma unroll
            for (int j = 0; j < TN; ++j) wv[j].m = piece_of(ws + j * 1024 + kPartW);
            xv[0].m = piece_of(xs + kPartX);
#pragma unroll
            for (int j = 0; j < TN; ++j) wv[j].l = piece_of(ws + j * 1024 + 2 * kPartW);
            xv[0].l = piece_of(xs + 2 * kPartX);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if (i + 1 < TM) {
                    xv[i + 1].h = piece_of(xs + (i + 1) * 1024);
                    xv[i + 1].m = piece_of(xs + (i + 1) * 1024 + kPartX);
                    xv[i + 1].l = piece_of(xs + (i + 1) * 1024 + 2 * kPartX);
                }
                f32x4 sums[TN];
                block_sums<TN, 1>(wv, &xv[i], sums);
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] += kDown * sums[j];
            }
            if (wn == 1) {
                store(1 - u, 1 - u);
                load(1 - u, b + 3);
            }
            if (FOLD && (++in_range == blocks_per_split || b + 1 == last)) {
                mend_range(range_begin, b + 1);
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        sum[i][j] += acc[i][j];
                        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                range_begin = b + 1;
                in_range = 0;
            }
        }
    }
    if (!FOLD) mend_range(first, last);
    float* to = out + (FOLD ? 0 : static_cast<size_t>(blockIdx.y) * m * n);
    const bool whole = n % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;   // four values are one store
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = row0 + i * 16;
        if (row >= m) continue;
#pragma unroll
        for (int j = 0; j < (GATED ? TN / 2 : TN); ++j) {
            const int col = col0 + j * 16;
            if (col >= n) continue;
            f32x4 val = FOLD ? sum[FOLD ? i : 0][FOLD ? j : 0] : acc[i][j];
            if constexpr (GATED) {
                const f32x4 up = FOLD ? sum[FOLD ? i : 0][FOLD ? j + TN / 2 : 0] : acc[i][j + TN / 2];
#pragma unroll
                for (int v = 0; v < 4; ++v) val[v] = up[v] * gate_activation(val[v], act);
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (bias && col + v < n) val[v] += bias[col + v];
            }
            float* at = to + static_cast<size_t>(row) * n + col;
            if (whole) {
                *reinterpret_cast<f32x4*>(at) = val;
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (col + v < n) at[v] = val[v];
            }
        }
    }
}

}  // namespace egpt

using namespace egpt;

extern "C" int egpt_gemm_f32(const float* x, const float* w, const float* bias, float* out, int m, int n, int k,
                             int n_splits, void* stream) {
    if (!x || !w || !out || m < 0 || n <= 0 || k <= 0 || n_splits < 1) return EGPT_BAD_ARGUMENT;
    if (k % 4 != 0 || (bias && n_splits != 1)) return EGPT_UNSUPPORTED_SIZE;
    if (m == 0) return EGPT_OK;
    const int total_steps = (k + kStepF - 1) / kStepF;
    const int steps_per_split = (total_steps + n_splits - 1) / n_splits;
    if (n_splits > total_steps || (n_splits - 1) * steps_per_split >= total_steps) return EGPT_BAD_ARGUMENT;   // an empty split
    const long groups = (static_cast<long>(m) + 63) / 64;
    if (groups > 65535 || n_splits > 65535) return EGPT_UNSUPPORTED_SIZE;
    // Two wavefronts to a workgroup instead of four while twice the workgroups still are about one to a CU: the stream of w then
    // comes through more CUs (8 rows, us with two / four: 4.8 / 5.0 for 1,152 x 896 in 7 ranges, 126 workgroups of four; 11.7 / 10.1
    // for 896 x 4,864 in 11, 154).
    const bool two = (n + 63) / 64 * static_cast<long>(n_splits) * groups < 130;
    const unsigned cols = two ? 32 : 64;
    const dim3 grid((n + cols - 1) / cols, static_cast<unsigned>(n_splits), static_cast<unsigned>(groups));
    hipStream_t s = static_cast<hipStream_t>(stream);
#define EGPT_F32(MT_, CH_)                                                                                             \
    do {                                                                                                               \
        if (two) gemm_f32_mfma_kernel<MT_, CH_, 2><<<grid, 128, 0, s>>>(x, w, bias, out, m, n, k, steps_per_split);    \
        else gemm_f32_mfma_kernel<MT_, CH_, 4><<<grid, 256, 0, s>>>(x, w, bias, out, m, n, k, steps_per_split);        \
    } while (0)
    switch (m > 64 ? 4 : (m + 15) / 16) {
        case 1:                                           // (a range of two steps has no use for registers and LDS of four)
            if (steps_per_split <= 2) EGPT_F32(1, 2);
            else EGPT_F32(1, 4);
            break;
        case 2: EGPT_F32(2, 1); break;
        case 3: EGPT_F32(3, 1); break;
        default: EGPT_F32(4, 1); break;
    }
#undef EGPT_F32
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

template <bool GATED>
static int launch_f32_rows(const float* x, const float* w, const float* bias, float* out, int m, int n, int k, int n_splits, int fold,
                           int tile_rows, int act, hipStream_t s) {
    const int total_steps = (k + kStepF - 1) / kStepF;
    const int steps_per_split = (total_steps + n_splits - 1) / n_splits;
    if (n_splits > total_steps || (n_splits - 1) * steps_per_split >= total_steps) return EGPT_BAD_ARGUMENT;   // an empty split
    if (tile_rows != 64 && tile_rows != 128) return EGPT_BAD_ARGUMENT;
    constexpr int cols = GATED ? 64 : 128;
    const long tiles = ((static_cast<long>(m) + tile_rows - 1) / tile_rows) * ((static_cast<long>(n) + cols - 1) / cols);
    if (tiles > 0x7fffffffL || n_splits > 65535) return EGPT_UNSUPPORTED_SIZE;
    const int per = steps_per_split * (kStepF / kBlockF);
    const bool folded = fold && n_splits > 1, tail = k % kBlockF != 0;
    const dim3 grid(static_cast<unsigned>(tiles), folded ? 1u : static_cast<unsigned>(n_splits));
#define EGPT_F32_ROWS(WM_)                                                                                                  \
    do {                                                                                                                    \
        if (folded && tail) gemm_f32_rows_kernel<WM_, true, true, GATED><<<grid, WM_ * 128, 0, s>>>(x, w, bias, out, m, n, k, per, act);   \
        else if (folded) gemm_f32_rows_kernel<WM_, true, false, GATED><<<grid, WM_ * 128, 0, s>>>(x, w, bias, out, m, n, k, per, act);     \
        else if (tail) gemm_f32_rows_kernel<WM_, false, true, GATED><<<grid, WM_ * 128, 0, s>>>(x, w, bias, out, m, n, k, per, act);       \
        else gemm_f32_rows_kernel<WM_, false, false, GATED><<<grid, WM_ * 128, 0, s>>>(x, w, bias, out, m, n, k, per, act);                \
    } while (0)
    if (tile_rows == 128) EGPT_F32_ROWS(4);
    else EGPT_F32_ROWS(2);
#undef EGPT_F32_ROWS
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

extern "C" int egpt_gemm_f32_rows(const float* x, const float* w, const float* bias, float* out, int m, int n, int k,
                                  int n_splits, int fold, int tile_rows, void* stream) {
    if (!x || !w || !out || m < 0 || n <= 0 || k <= 0 || n_splits < 1) return EGPT_BAD_ARGUMENT;
    if (k % 4 != 0 || (bias && n_splits != 1)) return EGPT_UNSUPPORTED_SIZE;
    if (m == 0) return EGPT_OK;
    return launch_f32_rows<false>(x, w, bias, out, m, n, k, n_splits, fold, tile_rows, 0, static_cast<hipStream_t>(stream));
}

extern "C" int egpt_gemm_f32_gated(const float* x, const float* w, float* out, int m, int n, int k, int n_splits, int tile_rows,
                                   int act, void* stream) {
    if (!x || !w || !out || m < 0 || n <= 0 || n > 0x3fffffff || k <= 0 || n_splits < 1 || act < 0 || act > 1) return EGPT_BAD_ARGUMENT;
    if (k % 4 != 0) return EGPT_UNSUPPORTED_SIZE;
    if (m == 0) return EGPT_OK;
    return launch_f32_rows<true>(x, w, nullptr, out, m, n, k, n_splits, 1, tile_rows, act, static_cast<hipStream_t>(stream));
}

extern "C" int egpt_linear(const void* x, const void* w, const void* bias, void* out, int m, int n, int k, int dtype,
                           int out_f32, void* stream) {
    if (!x || !w || !out || m < 0 || n <= 0 || k <= 0) return EGPT_BAD_ARGUMENT;
    if (m == 0) return EGPT_OK;
    if ((static_cast<long>(m) + BM - 1) / BM > 65535) return EGPT_UNSUPPORTED_SIZE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == 0) return launch_tiled<float, float>(x, w, bias, out, m, n, k, s);
    if (dtype == 1) {
        if (out_f32) return launch_tiled<bf16_t, float>(x, w, bias, out, m, n, k, s);
        return launch_tiled<bf16_t, bf16_t>(x, w, bias, out, m, n, k, s);
    }
    return EGPT_BAD_ARGUMENT;
}
