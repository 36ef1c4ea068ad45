// Sampling from float32 logits on the device: argmax, and temperature / top-k / top-p sampling.
//
// The reference samples from probabilities on the host (/root/reference/src/sampler.cpp:39-105):
// p^(1/T) (== softmax(logits / T) after normalisation), keep the k most likely, then the smallest
// set of most likely tokens whose normalised mass reaches top_p, then one uniform draw over the
// kept mass.  Here the kept set is found without sorting, by radix selection on the bit patterns of the
// weights (four passes of eight bits over the row, which stays in cache; masses are added in fixed point so
// that no decision depends on the order of additions), and the draw walks the kept weights in index order.
#include <mutex>

#include "api.h"
#include "common.h"

namespace egpt {

constexpr int kSampleThreads = 1024;

// Calls f(index, value) for every element of p[0..n) once, spread over the workgroup's threads (thread `tid` of
// `n_threads`).  The body reads 16 bytes per thread and keeps eight such loads in flight: a pass over a row is a
// chain of dependent loads otherwise, and its time is their latency, not the row's size.
template <typename F>
__device__ __forceinline__ void for_each_in_row(const float* __restrict__ p, int n, int tid, int n_threads, F f) {
    const int head = min(n, static_cast<int>((4u - ((reinterpret_cast<uintptr_t>(p) >> 2) & 3u)) & 3u));
    for (int j = tid; j < head; j += n_threads) f(j, p[j]);
    const float4* p4 = reinterpret_cast<const float4*>(p + head);
    const int n4 = (n - head) / 4;
    // eight loads issued before the first value is used (the compiler does not do this by itself across calls of f
    // that hold ballots or atomic additions)
    constexpr int kAhead = 8;
    int i = tid;
    for (; i + (kAhead - 1) * n_threads < n4; i += kAhead * n_threads) {
        float4 v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = p4[i + u * n_threads];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int j = head + 4 * (i + u * n_threads);
            f(j, v[u].x);
            f(j + 1, v[u].y);
            f(j + 2, v[u].z);
            f(j + 3, v[u].w);
        }
    }
    for (; i < n4; i += n_threads) {
        const float4 v = p4[i];
        const int j = head + 4 * i;
        f(j, v.x);
        f(j + 1, v.y);
        f(j + 2, v.z);
        f(j + 3, v.w);
    }
    for (int j = head + 4 * n4 + tid; j < n; j += n_threads) f(j, p[j]);
}

// lowest index among equal maxima (/root/reference/src/sampler.cpp:13-20: std::max_element)
__device__ __forceinline__ void argmax_combine(float& v, int& i, float ov, int oi) {
    if (ov > v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}

// The row's best token and its value (every thread); kNoToken and -infinity where there is nothing but NaN.
struct BestToken {
    int index;
    float value;
};
constexpr int kNoToken = 0x7fffffff;
__device__ BestToken block_argmax(const float* __restrict__ row, int vocab, float* s_val, int* s_idx) {
    float best = -INFINITY;
    int best_i = kNoToken;
    for_each_in_row(row, vocab, threadIdx.x, blockDim.x, [&](int j, float v) {
        if (v > best || (v == best && j < best_i)) {
            best = v;
            best_i = j;
        }
    });
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, kWave);
        const int oi = __shfl_xor(best_i, o, kWave);
        argmax_combine(best, best_i, ov, oi);
    }
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) {
        s_val[wave] = best;
        s_idx[wave] = best_i;
    }
    __syncthreads();
    const int n_waves = (blockDim.x + kWave - 1) / kWave;
    best = s_val[0];
    best_i = s_idx[0];
    for (int w = 1; w < n_waves; ++w) argmax_combine(best, best_i, s_val[w], s_idx[w]);
    return {best_i, best};
}

__global__ __launch_bounds__(kSampleThreads) void argmax_kernel(const float* __restrict__ logits,
                                                                int32_t* __restrict__ out, int vocab) {
    __shared__ float s_val[16];
    __shared__ int s_idx[16];
    const int r = blockIdx.x;
    const int best = block_argmax(logits + static_cast<size_t>(r) * vocab, vocab, s_val, s_idx).index;
    if (threadIdx.x == 0) out[r] = best == kNoToken ? 0 : best;
}

// Two stages for wide vocabularies: workgroup (row, c) finds the maximum of its piece of the row, then one
// workgroup per row picks among the pieces (lowest index among equal maxima in both stages).
constexpr int kArgmaxPieces = 32;

// For sampling each wavefront leaves the maximum of its share as well (sub_val [rows][kSubPieces], -infinity where it had no
// token).
constexpr int kSubPieces = kArgmaxPieces * 4;

__global__ __launch_bounds__(256) void argmax_pieces_kernel(const float* __restrict__ logits,
                                                            float* __restrict__ piece_val,
                                                            int32_t* __restrict__ piece_idx, float* __restrict__ sub_val,
                                                            int vocab) {
    __shared__ float s_val[16];
    __shared__ int s_idx[16];
    const int r = blockIdx.x, c = blockIdx.y;
    const int piece = (vocab + kArgmaxPieces - 1) / kArgmaxPieces;
    const int begin = min(vocab, c * piece), n = min(vocab, begin + piece) - begin;
    BestToken best{kNoToken, -INFINITY};
    if (n > 0) best = block_argmax(logits + static_cast<size_t>(r) * vocab + begin, n, s_val, s_idx);
    if (threadIdx.x == 0) {
        piece_val[r * kArgmaxPieces + c] = best.value;
        piece_idx[r * kArgmaxPieces + c] = best.index == kNoToken ? kNoToken : begin + best.index;
    }
    if (sub_val && threadIdx.x < 4) sub_val[r * kSubPieces + c * 4 + threadIdx.x] = n > 0 ? s_val[threadIdx.x] : -INFINITY;
}

// The row's best token out of its pieces' (lowest index among equal maxima; the first of nothing but NaN) and its value, by a whole
// wavefront.
__device__ __forceinline__ BestToken best_of_pieces(const float* __restrict__ piece_val, const int32_t* __restrict__ piece_idx, int r, int lane) {
    float v = lane < kArgmaxPieces ? piece_val[r * kArgmaxPieces + lane] : -INFINITY;
    int i = lane < kArgmaxPieces ? piece_idx[r * kArgmaxPieces + lane] : kNoToken;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(v, o, kWave);
        const int oi = __shfl_xor(i, o, kWave);
        argmax_combine(v, i, ov, oi);
    }
    return {__builtin_amdgcn_readfirstlane(i == kNoToken ? 0 : i), __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)))};
}
__global__ __launch_bounds__(64) void argmax_pick_kernel(const float* __restrict__ piece_val,
                                                         const int32_t* __restrict__ piece_idx,
                                                         int32_t* __restrict__ out) {
    const int best = best_of_pieces(piece_val, piece_idx, blockIdx.x, threadIdx.x).index;
    if (threadIdx.x == 0) out[blockIdx.x] = best;
}

// weight of token j: exp((x_j - max) / T), in [0, 1]
__device__ __forceinline__ float weight_of(float x, float mx, float inv_t) { return expf((x - mx) * inv_t); }

// Fixed-point image of a weight in [0, 1] (40 fractional bits): sums of these are integers, so a sum over the
// row does not depend on the order in which threads add, and neither does any decision taken from it.
__device__ __forceinline__ unsigned long long fixed_of(float w) {
    return static_cast<unsigned long long>(static_cast<double>(w) * 1099511627776.0);
}

// The largest bit pattern tau with count(w >= tau) >= need (non-negative floats order like their bits): radix
// selection, eight bits a level, histogram in LDS.  The weights of a row crowd into a few exponents, so the
// lanes of a wavefront that hit the same bin first agree on one addition (a ballot and a population count).
__device__ uint32_t select_by_count(const float* __restrict__ w, int vocab, unsigned int need, unsigned int* hist,
                                    uint32_t* shared_prefix, unsigned int* shared_need) {
    uint32_t prefix = 0u, mask = 0u;
    const int lane = threadIdx.x % kWave;
    int first_level = 3;
    {
        // The highest digit of a weight's pattern is its exponent (two exponents a bin), and the k-th largest
        // weight is almost always within 2^-15 of the largest (1.0, digit 0x3f): count those eight bins in
        // registers.  If the k-th weight is smaller still, the general histogram below takes over.
        unsigned int c[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
        for_each_in_row(w, vocab, threadIdx.x, blockDim.x, [&](int, float wj) {
            const uint32_t bits = __float_as_uint(wj);
            if (bits >= 0x38000000u) {
                const uint32_t d = 0x3fu - (bits >> 24);
#pragma unroll
                for (int i = 0; i < 8; ++i) c[i] += d == static_cast<uint32_t>(i) ? 1u : 0u;
            }
        });
        for (int i = threadIdx.x; i < 8; i += blockDim.x) hist[i] = 0u;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            unsigned int v = c[i];
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
            if (lane == 0 && v) atomicAdd(&hist[i], v);          // integer sums: order does not matter
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned int cum = 0u;
            int found = -1;
            for (int i = 0; i < 8; ++i) {
                if (cum + hist[i] >= need) {
                    found = i;
                    break;
                }
                cum += hist[i];
            }
            *shared_prefix = found >= 0 ? (0x3fu - found) << 24 : 0xffffffffu;
            *shared_need = found >= 0 ? need - cum : need;
        }
        __syncthreads();
        if (*shared_prefix != 0xffffffffu) {
            prefix = *shared_prefix;
            need = *shared_need;
            mask = 255u << 24;
            first_level = 2;
        }
        __syncthreads();
    }
    for (int level = first_level; level >= 0; --level) {
        const int shift = 8 * level;
        for (int i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0u;
        __syncthreads();
        for_each_in_row(w, vocab, threadIdx.x, blockDim.x, [&](int, float wj) {
            const uint32_t bits = __float_as_uint(wj);
            const uint32_t bin = (bits & mask) == prefix ? (bits >> shift) & 255u : 0xffffffffu;
            unsigned long long todo = __ballot(bin != 0xffffffffu);      // over the lanes that are here
            while (todo) {
                const int leader = __ffsll(static_cast<long long>(todo)) - 1;
                const uint32_t b0 = __shfl(bin, leader, kWave);
                const unsigned long long same = __ballot(bin == b0);
                if (lane == leader) atomicAdd(&hist[b0], static_cast<unsigned int>(__popcll(same)));
                todo &= ~same;
            }
        });
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned int cum = 0u;
            int bin = 255;
            for (; bin > 0; --bin) {
                if (cum + hist[bin] >= need) break;
                cum += hist[bin];
            }
            *shared_prefix = prefix | (static_cast<uint32_t>(bin) << shift);
            *shared_need = need - cum;
        }
        __syncthreads();
        prefix = *shared_prefix;
        need = *shared_need;
        mask |= 255u << shift;
        __syncthreads();
    }
    return prefix;
}

// Among the weights >= lo, the largest bit pattern tau with mass(w >= tau) >= need: the smallest set of most likely tokens whose
// mass reaches need, ties at tau included whole.  In between, mass(w >= lo) >= need and mass(w >= hi) = above < need.  Each pass
// divides [lo, hi): weights that crowd into a few exponents by fifteen pivots, whose masses every thread sums in registers;
// after that by 64 bins in LDS (152,000 weights of a row that top-p alone cuts, four such passes: 540 -> 170 us a row, where
// seven passes of pivots walked it).  Masses are fixed-point integers, whose sums depend on no order.
__device__ uint32_t select_by_mass(const float* __restrict__ w, int vocab, uint32_t lo, uint32_t hi, unsigned long long above,
                                   unsigned long long need, unsigned long long* sums /* [16][15] */, uint32_t* shared_lo,
                                   uint32_t* shared_hi, unsigned long long* shared_above) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, n_waves = blockDim.x / kWave;
    if (lo + 1u < hi && hi == 0x3f800001u && lo < 0x38000000u) {
        // pivots on exponent boundaries near 1.0, where the mass is
        const uint32_t base = 0x37000000u, step = 0x01000000u;       // pivot i = base + (i + 1) * step
        unsigned long long acc[15];
#pragma unroll
        for (int i = 0; i < 15; ++i) acc[i] = 0ull;
        for_each_in_row(w, vocab, threadIdx.x, blockDim.x, [&](int, float wj) {
            const uint32_t bits = __float_as_uint(wj);
            if (bits > base && bits < hi && bits >= lo) {             // only these can lie at or above a pivot
                const unsigned long long f = fixed_of(wj);
#pragma unroll
                for (int i = 0; i < 15; ++i) acc[i] += bits >= base + (i + 1) * step ? f : 0ull;
            }
        });
#pragma unroll
        for (int i = 0; i < 15; ++i) {
            unsigned long long v = acc[i];
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
            if (lane == 0) sums[wave * 15 + i] = v;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t new_lo = lo, new_hi = hi;
            unsigned long long new_above = above;
            for (int i = 0; i < 15; ++i) {
                const uint32_t pivot = base + (i + 1) * step;
                if (pivot >= hi) break;
                if (pivot <= lo) continue;
                unsigned long long mass = above;
                for (int wv = 0; wv < n_waves; ++wv) mass += sums[wv * 15 + i];
                if (mass >= need) {
                    new_lo = pivot;
                } else {
                    new_hi = pivot;
                    new_above = mass;
                    break;
                }
            }
            *shared_lo = new_lo;
            *shared_hi = new_hi;
            *shared_above = new_above;
        }
        __syncthreads();
        lo = *shared_lo;
        hi = *shared_hi;
        above = *shared_above;
        __syncthreads();
    }
    while (lo + 1u < hi) {                           // (every pass leaves at most 1 / 32 of the range, and one pattern in the end)
        const int width = 32 - __clz(static_cast<int>(hi - lo - 1u));
        const int shift = width > 6 ? width - 6 : 0;
        if (threadIdx.x < kWave) sums[threadIdx.x] = 0ull;
        __syncthreads();
        for_each_in_row(w, vocab, threadIdx.x, blockDim.x, [&](int, float wj) {
            const uint32_t bits = __float_as_uint(wj);
            if (bits >= lo && bits < hi) atomicAdd(&sums[(bits - lo) >> shift], fixed_of(wj));
        });
        __syncthreads();
        if (threadIdx.x < kWave) {
            const int bin = kWave - 1 - lane;        // from the greatest weights down
            const unsigned long long mine = sums[bin];
            unsigned long long incl = mine;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const unsigned long long up = __shfl_up(incl, o, kWave);
                if (lane >= o) incl += up;
            }
            const unsigned long long reached = __ballot(above + incl >= need);
            const int holder = reached ? __ffsll(static_cast<long long>(reached)) - 1 : kWave - 1;
            if (lane == holder) {
                *shared_lo = lo + (static_cast<uint32_t>(bin) << shift);
                *shared_hi = min(hi, lo + (static_cast<uint32_t>(bin + 1) << shift));
                *shared_above = above + incl - mine;
            }
        }
        __syncthreads();
        lo = *shared_lo;
        hi = *shared_hi;
        above = *shared_above;
        __syncthreads();
    }
    return lo;
}

// ---- wide vocabularies: the row-wide work spread over many workgroups, the selection on what is left of the row
//
// The selection below walks its row a dozen times with one workgroup, which for 150,000 tokens is 300 us whatever the
// number of rows.  For a wide vocabulary kernels with kSamplePieces workgroups per row come first and leave it a list of
// candidates.
//
// Top-k of at most kSubPieces tokens: the search for the row's maximum leaves the maxima of 128 shares of the row, and the k-th
// largest of those is no larger than the k-th largest token.  One pass lists the tokens that weigh as much (some 30 for a k of
// 20, ties among them), in any order; the last kernel puts them in index order.
//
// All other rows: the weights are counted by exponent, then the tokens at or above the exponent below which none can be kept are
// listed, in index order.  The selection runs on that list: one thread per candidate when they are at most kSampleThreads,
// the row-walking selection otherwise.  A row for which neither cut is asked gets no list: the pieces' masses say in which
// piece the drawn point lies, and that piece alone is walked.  Counted are the weights within 2^-15 of the largest, an exponent
// a bin, which hold the top-p mass of any distribution that is not nearly flat.
//
// 64 rows of 151,936, us: top-k 20, top-p 0.95 at 0.8 52 to 455 (rows whose k-th weight lay below 2^-15 of the largest had all
// their vocabulary for candidates) -> 34; top-k 50 at 0.6 500 -> 40; top-k 200 at 1.0 97 -> 62; top-p alone 541 -> 201; one row of the first
// 30 -> 22.
constexpr int kSamplePieces = 32;
constexpr int kTopBins = 16;            // exponents 127 (weight 1.0) down to 112, one bin each; bin kTopBins: the rest

__device__ __forceinline__ int top_bin_of(uint32_t bits) {           // bits of a weight in [0, 1]; kTopBins: below the bins (and NaN)
    const int e = static_cast<int>(bits >> 23);
    return e >= 128 - kTopBins && e <= 127 ? 127 - e : kTopBins;
}
// The exponential's argument; below kNoTopBin (ln 2^-15 is -10.40) the weight lies in none of the top bins.
__device__ __forceinline__ float exponent_of(float x, float mx, float inv_t) { return (x - mx) * inv_t; }
constexpr float kNoTopBin = -10.5f;
// A row with top-k whose candidates follow from the shares' maxima: nothing of it underflows, and there are k maxima.
constexpr float kLeastExponent = -80.0f;

// The k-th largest of a row's kSubPieces maxima (k <= kSubPieces; 256 threads, `mine` the maximum of thread t < kSubPieces).
__device__ float bound_of_row(float mine, int k, float* s_sub /* [kSubPieces] */, unsigned int* s_bound) {
    const int t = threadIdx.x;
    if (t < kSubPieces) s_sub[t] = mine;
    if (t == 0) *s_bound = 0xffffffffu;
    __syncthreads();
    if (t < kSubPieces) {
        int greater = 0;
#pragma unroll
        for (int i = 0; i < kSubPieces / 4; ++i) {
            const float4 v = reinterpret_cast<const float4*>(s_sub)[i];
            greater += (v.x > mine) + (v.y > mine) + (v.z > mine) + (v.w > mine);
        }
        // the least of those that fewer than k exceed; bits in the order of the numbers
        const unsigned int bits = __float_as_uint(mine), order = bits & 0x80000000u ? ~bits : bits | 0x80000000u;
        if (greater < k) atomicMin(s_bound, order);
    }
    __syncthreads();
    const unsigned int order = *s_bound;
    return __uint_as_float(order & 0x80000000u ? order & 0x7fffffffu : ~order);
}

// The candidates of a piece by the bound of its row, in no order: tight ones (they weigh as much as the bound) from the front of the
// piece's part of the row's list, loose ones (down to the exponent's beginning, if it is one of the top bins': with them the
// list is the one that counting by exponent would leave, and the draw adds up the same numbers in the same places) from its
// back.  `first`: the thread's tokens begin + t, begin + t + 256 ..., kCollectAhead of them, on their way since the kernel began.
constexpr int kCollectAhead = 20;
__device__ void collect_candidates(const float* __restrict__ row, int begin, int n, const float (&first)[kCollectAhead], float mx, float inv_t,
                                   float bound_t, float* __restrict__ ow, int32_t* __restrict__ oi, int* s_n /* [2], zeros */) {
    // (expf may be off by a unit either way: 2^-18 below the bound is below every token that is not)
    const float tight = expf(bound_t) * (1.0f - 3.8147e-6f);
    const uint32_t bits = __float_as_uint(tight);
    const float loose = top_bin_of(bits) < kTopBins ? __uint_as_float(bits & 0x7f800000u) : tight;
    const float far = bound_t - 0.75f;                       // e^-0.75 < 1/2
    auto look = [&](float x, int j) {
        const float t = exponent_of(x, mx, inv_t);
        if (!(t >= far)) return;
        const float w = expf(t);
        if (w < loose) return;
        const int to = w >= tight ? begin + atomicAdd(&s_n[0], 1) : begin + n - 1 - atomicAdd(&s_n[1], 1);
        ow[to] = w;
        oi[to] = begin + j;
    };
#pragma unroll
    for (int i = 0; i < kCollectAhead; ++i)
        if (static_cast<int>(threadIdx.x) + 256 * i < n) look(first[i], threadIdx.x + 256 * i);
    for (int j0 = 256 * kCollectAhead; j0 < n; j0 += 256 * kCollectAhead) {
        float v[kCollectAhead];
#pragma unroll
        for (int i = 0; i < kCollectAhead; ++i) {
            const int j = j0 + threadIdx.x + 256 * i;
            v[i] = j < n ? row[begin + j] : -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < kCollectAhead; ++i)
            if (j0 + static_cast<int>(threadIdx.x) + 256 * i < n) look(v[i], j0 + threadIdx.x + 256 * i);
    }
}

// Rows whose candidates follow from the maxima: their lists.  Others:
// piece_count, piece_mass [rows][kSamplePieces][kTopBins + 1]: per piece of the row, how many weights each bin holds, and, where the
// row's draw asks for it (no top-k), their mass in fixed point
__global__ __launch_bounds__(256, 8) void sample_count_kernel(const float* __restrict__ logits, const float* __restrict__ temperature,
                                                          const int32_t* __restrict__ top_k, const float* __restrict__ piece_val,
                                                          const int32_t* __restrict__ piece_idx, const float* __restrict__ sub_val,
                                                          int32_t* __restrict__ best_out, int32_t* __restrict__ listed,
                                                          int32_t* __restrict__ list_count,
                                                          float* __restrict__ cand_w, int32_t* __restrict__ cand_idx,
                                                          unsigned int* __restrict__ piece_count,
                                                          unsigned long long* __restrict__ piece_mass, int vocab) {
    __shared__ __attribute__((aligned(16))) float s_sub[kSubPieces];
    __shared__ unsigned int s_bound;
    __shared__ int s_n[2];
    __shared__ unsigned int s_count[kTopBins + 1];
    __shared__ unsigned long long s_mass[kTopBins + 1];
    const int r = blockIdx.x, c = blockIdx.y;
    const float temp = temperature[r];
    const int k = top_k[r];
    const bool by_count = k > 0 && k < vocab;
    const float* row = logits + static_cast<size_t>(r) * vocab;
    const int piece = (vocab + kSamplePieces - 1) / kSamplePieces;
    const int begin = min(vocab, c * piece), n = min(vocab, begin + piece) - begin;
    // everything that can be asked for is asked for at once: what follows is a chain of waits otherwise
    const bool may_list = temp > 0.f && by_count && k <= kSubPieces;
    float first[kCollectAhead], sub = 0.f;
    if (may_list) {
#pragma unroll
        for (int i = 0; i < kCollectAhead; ++i) {
            const int j = threadIdx.x + 256 * i;
            first[i] = j < n ? row[begin + j] : -INFINITY;
        }
        if (threadIdx.x < kSubPieces) sub = sub_val[r * kSubPieces + threadIdx.x];
    }
    const BestToken best = best_of_pieces(piece_val, piece_idx, r, threadIdx.x % kWave);
    if (c == 0 && threadIdx.x == 0) best_out[r] = best.index;
    if (!(temp > 0.f)) return;
    const float mx = best.value;
    const float inv_t = 1.0f / fmaxf(temp, 1e-6f);
    if (may_list) {
        if (threadIdx.x < 2) s_n[threadIdx.x] = 0;
        const float bound_t = exponent_of(bound_of_row(sub, k, s_sub, &s_bound), mx, inv_t);
        if (bound_t >= kLeastExponent && fabsf(mx) < INFINITY) {
            collect_candidates(row, begin, n, first, mx, inv_t, bound_t, cand_w + static_cast<size_t>(r) * vocab,
                               cand_idx + static_cast<size_t>(r) * vocab, s_n);
            if (c == 0 && threadIdx.x == 0) listed[r] = 1;
            __syncthreads();
            if (threadIdx.x < 2) list_count[(r * kSamplePieces + c) * 2 + threadIdx.x] = s_n[threadIdx.x];
            return;
        }
    }
    if (c == 0 && threadIdx.x == 0) listed[r] = 0;
    if (threadIdx.x <= kTopBins) {
        s_count[threadIdx.x] = 0u;
        s_mass[threadIdx.x] = 0ull;
    }
    __syncthreads();
    // Nearly every weight lies below the top bins and is summed in registers; the few above go to the bins in LDS
    // (integer additions: the order does not matter).  With top-k a weight that lies below them is not even computed.
    unsigned int low = 0u;
    unsigned long long low_mass = 0ull;
    for_each_in_row(row + begin, n, threadIdx.x, blockDim.x, [&](int, float x) {
        const float t = exponent_of(x, mx, inv_t);
        if (!by_count || !(t < kNoTopBin)) {
            const float w = expf(t);
            const int bin = top_bin_of(__float_as_uint(w));
            if (bin < kTopBins) {
                atomicAdd(&s_count[bin], 1u);
                if (!by_count) atomicAdd(&s_mass[bin], fixed_of(w));
                return;
            }
            low_mass += static_cast<unsigned int>(w * 1099511627776.0f);          // fixed_of: below 2^-15, and 2^40 is exact
        }
        low += t <= 0.f ? 1u : 0u;                           // (a NaN is no candidate)
    });
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        low += __shfl_xor(low, o, kWave);
        low_mass += __shfl_xor(low_mass, o, kWave);
    }
    if (threadIdx.x % kWave == 0 && low) {
        atomicAdd(&s_count[kTopBins], low);
        if (!by_count) atomicAdd(&s_mass[kTopBins], low_mass);
    }
    __syncthreads();
    const size_t base = (static_cast<size_t>(r) * kSamplePieces + c) * (kTopBins + 1);
    if (threadIdx.x <= kTopBins) {
        piece_count[base + threadIdx.x] = s_count[threadIdx.x];
        piece_mass[base + threadIdx.x] = s_mass[threadIdx.x];
    }
}

// What a row's counts say, found by a workgroup of 256 for itself: the last bin whose tokens can be kept (kTopBins: every token can; -1:
// neither cut is asked for, and the draw needs no list), and where each piece's candidates start in the row's list.
struct SamplePlan {
    int last;
    int start, end, total;              // of the workgroup's piece; of the row
    unsigned long long row_mass;        // the mass of the whole row: what top-p without top-k refers to
    int direct_piece;                   // without cuts: the piece that holds the drawn point, and what is left of it there
    unsigned long long direct_target;   // (top-p without top-k: the mass of the bins above `last`, from which its search goes on)
};
struct SamplePlanSpace {
    unsigned int count[kSamplePieces][kTopBins + 1];
    unsigned long long mass[kSamplePieces][kTopBins + 1], bin_mass[kTopBins + 1];
    unsigned int bin_count[kTopBins + 1];
    int last, start[kSamplePieces + 1];
};
__device__ __forceinline__ SamplePlan plan_of_row(int r, int c, int k, float p, float u, const unsigned int* __restrict__ piece_count,
                                                  const unsigned long long* __restrict__ piece_mass, int vocab, SamplePlanSpace& space) {
    SamplePlan plan{kTopBins, 0, 0, 0, 0ull, -1, 0ull};
    const int t = threadIdx.x;
    const bool by_count = k > 0 && k < vocab, by_mass = p > 0.f && p < 1.f;
    const unsigned int* counts = piece_count + static_cast<size_t>(r) * kSamplePieces * (kTopBins + 1);
    const unsigned long long* masses = piece_mass + static_cast<size_t>(r) * kSamplePieces * (kTopBins + 1);
    if (!by_count && !by_mass) {
        // The pieces' masses are known, so the drawn point (in fixed point, of the whole row's mass) names its piece and what is
        // left of it inside that piece; the last kernel walks that piece alone.  (Every wavefront finds the same.)
        const int lane = t % kWave;
        unsigned long long mine = 0ull;
        if (lane < kSamplePieces) {
#pragma unroll
            for (int i = 0; i <= kTopBins; ++i) mine += masses[lane * (kTopBins + 1) + i];
        }
        unsigned long long incl = mine;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const unsigned long long up = __shfl_up(incl, o, kWave);
            if (lane >= o) incl += up;
        }
        const unsigned long long total = __shfl(incl, kSamplePieces - 1, kWave);
        u = fminf(fmaxf(u, 0.f), 0.99999994f);
        unsigned long long target = static_cast<unsigned long long>(static_cast<double>(u) * static_cast<double>(total));
        if (total > 0ull && target >= total) target = total - 1ull;
        const bool here = lane < kSamplePieces && incl > target && incl - mine <= target;   // at most one piece
        const unsigned long long holders = __ballot(here);
        const int piece = holders ? __ffsll(static_cast<long long>(holders)) - 1 : 0;      // (an empty row: piece 0)
        const unsigned long long inside = __shfl(target - (incl - mine), piece, kWave);
        plan.last = -1;
        plan.row_mass = total;
        plan.direct_piece = piece;
        plan.direct_target = holders ? inside : 0ull;
        return plan;
    }
    for (int i = t; i < kSamplePieces * (kTopBins + 1); i += 256) (&space.count[0][0])[i] = counts[i];
    if (!by_count)
        for (int i = t; i < kSamplePieces * (kTopBins + 1); i += 256) (&space.mass[0][0])[i] = masses[i];
    __syncthreads();
    if (t <= kTopBins) {
        unsigned int v = 0u;
#pragma unroll
        for (int i = 0; i < kSamplePieces; ++i) v += space.count[i][t];
        space.bin_count[t] = v;
    } else if (!by_count && t >= kWave && t < kWave + (kTopBins + 1)) {
        unsigned long long v = 0ull;
#pragma unroll
        for (int i = 0; i < kSamplePieces; ++i) v += space.mass[i][t - kWave];
        space.bin_mass[t - kWave] = v;
    }
    __syncthreads();
    if (t == 0) {
        int last = kTopBins;
        if (by_count) {                                      // the k-th largest weight lies in this bin; top-p only removes more
            unsigned int cum = 0u;
            for (int i = 0; i <= kTopBins; ++i) {
                if (cum < static_cast<unsigned int>(k)) last = i;
                cum += space.bin_count[i];
            }
        } else {                                             // the mass p of the whole row is reached within this bin
            unsigned long long total = 0ull, cum = 0ull;
            for (int i = 0; i <= kTopBins; ++i) total += space.bin_mass[i];
            unsigned long long need = static_cast<unsigned long long>(static_cast<double>(p) * static_cast<double>(total));
            if (need == 0ull) need = 1ull;
            unsigned long long over = 0ull;
            for (int i = 0; i <= kTopBins; ++i) {
                if (cum < need) {
                    last = i;
                    over = cum;
                }
                cum += space.bin_mass[i];
            }
            space.bin_mass[0] = total;
            space.bin_mass[1] = over;
        }
        space.last = last;
    }
    __syncthreads();
    plan.last = space.last;
    plan.row_mass = by_count ? 0ull : space.bin_mass[0];
    plan.direct_target = by_count ? 0ull : space.bin_mass[1];
    if (t < kWave) {
        int mine = 0;
        if (t < kSamplePieces) {
#pragma unroll
            for (int i = 0; i <= kTopBins; ++i) mine += i <= plan.last ? static_cast<int>(space.count[t][i]) : 0;
        }
        int incl = mine;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int up = __shfl_up(incl, o, kWave);
            if (t >= o) incl += up;
        }
        if (t <= kSamplePieces) space.start[t] = incl - mine;
    }
    __syncthreads();
    plan.start = space.start[c];
    plan.end = space.start[c + 1];
    plan.total = space.start[kSamplePieces];
    return plan;
}

// the candidates of a piece, in index order: cand_w / cand_idx [rows][vocab]; their number and the plan's other findings per row
__global__ __launch_bounds__(256, 8) void sample_compact_kernel(const float* __restrict__ logits, const float* __restrict__ temperature,
                                                             const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
                                                             const float* __restrict__ uniform, const int32_t* __restrict__ best,
                                                             const unsigned int* __restrict__ piece_count,
                                                             const unsigned long long* __restrict__ piece_mass,
                                                             const int32_t* __restrict__ listed, float* __restrict__ cand_w,
                                                             int32_t* __restrict__ cand_idx, int32_t* __restrict__ cand_count,
                                                             unsigned long long* __restrict__ row_mass,
                                                             int32_t* __restrict__ direct_piece,
                                                             unsigned long long* __restrict__ direct_target,
                                                             int32_t* __restrict__ last_bin, int vocab) {
    __shared__ int s_wave[4];
    __shared__ SamplePlanSpace s_plan;
    const int r = blockIdx.x, c = blockIdx.y;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const float temp = temperature[r];
    if (!(temp > 0.f) || listed[r] != 0) {
        if (c == 0 && threadIdx.x == 0) direct_piece[r] = -1;
        return;
    }
    const float* row = logits + static_cast<size_t>(r) * vocab;
    const float mx = row[best[r]];
    const float inv_t = 1.0f / fmaxf(temp, 1e-6f);
    {
        const int k = top_k[r];
        const float p = top_p[r];
        if (c > 0 && !(k > 0 && k < vocab) && !(p > 0.f && p < 1.f)) return;      // no list is made without cuts
    }
    SamplePlan plan = plan_of_row(r, c, top_k[r], top_p[r], uniform[r], piece_count, piece_mass, vocab, s_plan);
    if (!(fabsf(mx) < INFINITY)) {                           // an infinity or nothing but NaN: the row's best token and no draw
        plan.total = 0;
        plan.last = plan.direct_piece = -1;
    }
    if (c == 0 && threadIdx.x == 0) {
        cand_count[r] = plan.total;
        last_bin[r] = plan.last;
        row_mass[r] = plan.row_mass;
        direct_piece[r] = plan.direct_piece;
        direct_target[r] = plan.direct_target;
    }
    if (plan.last < 0) return;
    const int piece = (vocab + kSamplePieces - 1) / kSamplePieces;
    const int begin = min(vocab, c * piece), end = min(vocab, begin + piece);
    float* ow = cand_w + static_cast<size_t>(r) * vocab;
    int32_t* oi = cand_idx + static_cast<size_t>(r) * vocab;
    int at = plan.start;
    if (plan.end == at) return;
    // a token's weight if it is a candidate.  The top bins go by the weight's bits, its argument only tells most others apart
    const uint32_t cut = static_cast<uint32_t>(127 - min(plan.last, kTopBins - 1)) << 23;
    const float far = plan.last < kTopBins ? -0.6931472f * static_cast<float>(plan.last) - 0.01f : -INFINITY;
    auto weight_of_candidate = [&](float x, float& w) {
        const float t = exponent_of(x, mx, inv_t);
        if (plan.last >= kTopBins) {
            if (t <= 0.f) w = expf(t);
            return t <= 0.f;
        }
        if (t < far) return false;
        w = expf(t);
        return top_bin_of(__float_as_uint(w)) < kTopBins && __float_as_uint(w) >= cut;
    };
    // Every wavefront takes a run of kRun groups of 64 tokens, all loads of a run on their way together; the order of the list is the
    // order of the tokens.
    constexpr int kRun = 20;
    for (int j0 = begin; j0 < end; j0 += 4 * kRun * kWave) {
        float v[kRun];
        const int j = j0 + wave * kRun * kWave + lane;
#pragma unroll
        for (int i = 0; i < kRun; ++i) v[i] = j + i * kWave < end ? row[j + i * kWave] : 0.f;
        unsigned long long masks[kRun];
        int mine = 0;
#pragma unroll
        for (int i = 0; i < kRun; ++i) {
            float w = 0.f;
            const bool keep = j + i * kWave < end && weight_of_candidate(v[i], w);
            v[i] = w;
            masks[i] = __ballot(keep);
            mine += __popcll(masks[i]);
        }
        if (lane == 0) s_wave[wave] = mine;
        __syncthreads();
        int to = at;
        for (int i = 0; i < 4; ++i) {
            to += i < wave ? s_wave[i] : 0;
            at += s_wave[i];
        }
#pragma unroll
        for (int i = 0; i < kRun; ++i) {
            if (masks[i] >> lane & 1ull) {
                const int place = to + __popcll(masks[i] & ((1ull << lane) - 1ull));
                ow[place] = v[i];
                oi[place] = j + i * kWave;
            }
            to += __popcll(masks[i]);
        }
        __syncthreads();
    }
}

// The selection and the draw for a list of at most kSampleThreads weights, one thread each (a list of candidates is
// usually a few dozen tokens, and the passes of the general selection cost their barriers, not their data).
// Token j is among the k most likely iff fewer than k weights are greater than its own, and within the mass `need`
// iff the mass of the greater weights is below it: the same sets as the thresholds of select_by_count and
// select_by_mass (ties whole).  Counts and fixed-point masses are integers, so nothing depends on an order; the
// draw walks the kept weights in index order.  Returns the picked position in the list or -1 (every thread).
__device__ int pick_from_short_list(float wj /* of thread j < n */, int n, bool cut_by_count, unsigned int k, float p,
                                    bool mass_of_row, unsigned long long row_mass, float u, float* s_list /* [kSampleThreads] */,
                                    unsigned long long* s_wave /* [16] */, float* s_piece /* [16] */, int* s_pick /* [2] */) {
    __shared__ __attribute__((aligned(16))) unsigned long long s_fixed[kSampleThreads];
    const int j = threadIdx.x, lane = j % kWave, wave = j / kWave, n_waves = blockDim.x / kWave;
    if (j >= n) wj = 0.f;
    s_fixed[j] = fixed_of(wj);
    s_list[j] = wj;                                   // slots past n hold 0: never greater than a weight
    if (j < 2) s_pick[j] = j == 0 ? 0x7fffffff : -1;
    __syncthreads();
    unsigned int above = 0u;
    unsigned long long mass_above = 0ull;
    const int n4 = (n + 3) / 4;
    for (int i = 0; i < n4; ++i) {                    // every thread reads the same address: a broadcast
        const float4 v = reinterpret_cast<const float4*>(s_list)[i];
        above += (v.x > wj) + (v.y > wj) + (v.z > wj) + (v.w > wj);
        const ulonglong2 a = reinterpret_cast<const ulonglong2*>(s_fixed)[2 * i], b = reinterpret_cast<const ulonglong2*>(s_fixed)[2 * i + 1];
        mass_above += (v.x > wj ? a.x : 0ull) + (v.y > wj ? a.y : 0ull) + (v.z > wj ? b.x : 0ull) + (v.w > wj ? b.y : 0ull);
    }
    bool keep = j < n && (!cut_by_count || above < k);
    if (p > 0.f && p < 1.f) {
        unsigned long long mine = keep ? fixed_of(wj) : 0ull;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) mine += __shfl_xor(mine, o, kWave);
        if (lane == 0) s_wave[wave] = mine;
        __syncthreads();
        unsigned long long kept = 0ull;
        for (int i = 0; i < n_waves; ++i) kept += s_wave[i];
        if (mass_of_row) kept = row_mass;
        unsigned long long need = static_cast<unsigned long long>(static_cast<double>(p) * static_cast<double>(kept));
        if (need == 0ull) need = 1ull;
        keep = keep && mass_above < need;
    }
    // inverse CDF in index order: prefix sums inside the wavefronts, then over them
    const float mine = keep ? wj : 0.f;
    float incl = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const float up = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += up;
    }
    if (lane == kWave - 1) s_piece[wave] = incl;
    __syncthreads();
    float before = 0.f, total = 0.f;
    for (int i = 0; i < n_waves; ++i) {
        before += i < wave ? s_piece[i] : 0.f;
        total += s_piece[i];
    }
    const float target = fminf(fmaxf(u, 0.f), 0.99999994f) * total;
    if (keep && before + incl > target) atomicMin(&s_pick[0], j);
    if (keep) atomicMax(&s_pick[1], j);               // the last kept token catches rounding at the end
    __syncthreads();
    return s_pick[0] != 0x7fffffff ? s_pick[0] : s_pick[1];
}

// The draw inside one piece of a row (tokens [begin, begin + n)) for a row without cuts: `target` is the drawn point
// in the fixed-point mass of the piece.  Every thread takes a run of consecutive tokens, the runs' masses are summed
// up over the workgroup in index order, and the thread whose run holds the point finds the token.  The weights
// are computed as the counting kernel computed them, so the masses are the same integers.  Returns the token or
// -1 (every thread).
__device__ int pick_in_piece(const float* __restrict__ row, int begin, int n, float mx, float inv_t, unsigned long long target,
                             unsigned long long* s_wave /* [16] */, int* s_pick /* [1] */) {
    const int j = threadIdx.x, lane = j % kWave, wave = j / kWave, n_waves = blockDim.x / kWave;
    const int run = (n + static_cast<int>(blockDim.x) - 1) / static_cast<int>(blockDim.x);
    const int r_begin = min(n, j * run), r_end = min(n, r_begin + run);
    unsigned long long mine = 0ull;
    for (int i = r_begin; i < r_end; ++i) mine += fixed_of(weight_of(row[begin + i], mx, inv_t));
    unsigned long long incl = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned long long up = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += up;
    }
    if (lane == kWave - 1) s_wave[wave] = incl;
    if (j == 0) s_pick[0] = -1;
    __syncthreads();
    unsigned long long before = 0ull;
    for (int i = 0; i < wave; ++i) before += s_wave[i];
    const unsigned long long excl = before + incl - mine;
    if (mine > 0ull && excl <= target && target < excl + mine) {
        unsigned long long cum = excl;
        for (int i = r_begin; i < r_end; ++i) {
            cum += fixed_of(weight_of(row[begin + i], mx, inv_t));
            if (cum > target) {
                s_pick[0] = begin + i;
                break;
            }
        }
    }
    __syncthreads();
    return s_pick[0];
}

// The unordered candidates of a row whose list follows from the maxima (n of them, a weight and an index to a thread): those at
// or above the beginning of the k-th weight's exponent, in index order, are
// left in s_list and s_order.  Returns their number (every thread).
__device__ int order_candidates(float wj, int ij, int n, unsigned int k, float* s_list, int* s_order, unsigned int* s_cell /* [2] */) {
    const int j = threadIdx.x;
    if (j < 2) s_cell[j] = j == 0 ? 0xffffffffu : 0u;
    s_list[j] = j < n ? wj : 0.f;
    __syncthreads();
    unsigned int above = 0u;
    const int n4 = (n + 3) / 4;
    for (int i = 0; i < n4; ++i) {
        const float4 v = reinterpret_cast<const float4*>(s_list)[i];
        above += (v.x > wj) + (v.y > wj) + (v.z > wj) + (v.w > wj);
    }
    if (j < n && above < k) atomicMin(&s_cell[0], __float_as_uint(wj));        // the k-th weight is the least of these
    __syncthreads();
    const uint32_t kth = s_cell[0];
    const uint32_t cut = top_bin_of(kth) < kTopBins ? kth & 0x7f800000u : 0u;
    const bool in = j < n && __float_as_uint(wj) >= cut;
    s_order[j] = in ? ij : 0x7fffffff;
    if (in) atomicAdd(&s_cell[1], 1u);
    __syncthreads();
    int rank = 0;
    for (int i = 0; i < n4; ++i) {
        const int4 v = reinterpret_cast<const int4*>(s_order)[i];
        rank += (v.x < ij) + (v.y < ij) + (v.z < ij) + (v.w < ij);
    }
    __syncthreads();
    if (in) {
        s_list[rank] = wj;
        s_order[rank] = ij;
    }
    __syncthreads();
    return static_cast<int>(s_cell[1]);
}

// One workgroup per row.  `weights` is scratch [rows][vocab] float32: the weights are computed once and the
// selection passes read them back (from cache).  With a list of candidates (cand_idx != null) `weights` holds the
// candidates' weights, cand_count[r] their number, and `best` the row's argmax.
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(
    const float* __restrict__ logits, const float* __restrict__ temperature, const int32_t* __restrict__ top_k,
    const float* __restrict__ top_p, const float* __restrict__ uniform, int32_t* __restrict__ out,
    float* __restrict__ weights, int vocab, const int32_t* __restrict__ cand_idx, const int32_t* __restrict__ cand_count,
    const int32_t* __restrict__ listed, const int32_t* __restrict__ list_count, const int32_t* __restrict__ best_in, const unsigned long long* __restrict__ row_mass,
    const int32_t* __restrict__ direct_piece, const unsigned long long* __restrict__ direct_target, const int32_t* __restrict__ last_bin) {
    __shared__ float s_val[16];
    __shared__ int s_idx[16];
    __shared__ unsigned int hist[256];
    __shared__ unsigned long long s_wave[16 * 15];
    __shared__ unsigned int s_need;
    __shared__ uint32_t s_a, s_b;
    __shared__ unsigned long long s_above;
    __shared__ float s_piece[16];
    __shared__ int s_owner;
    __shared__ float s_before;
    __shared__ __attribute__((aligned(16))) float s_list[kSampleThreads];
    __shared__ int s_pick[2];
    __shared__ __attribute__((aligned(16))) int s_order[kSampleThreads];
    const int r = blockIdx.x;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, n_waves = blockDim.x / kWave;
    const float* row = logits + static_cast<size_t>(r) * vocab;
    float* w = weights + static_cast<size_t>(r) * vocab;
    const int32_t* idx_of = cand_idx ? cand_idx + static_cast<size_t>(r) * vocab : nullptr;
    // (a row's few numbers at once: behind the branches that ask for them each would be a wait of its own)
    const float temp = temperature[r], p = top_p[r], u = uniform[r];
    const int k = top_k[r];
    int known_best = 0, is_listed = 0, direct = -1, count = 0, more = 0;
    if (cand_idx) {
        known_best = best_in[r];
        is_listed = listed[r];
        direct = direct_piece[r];
        if (lane < kSamplePieces) {
            count = list_count[(r * kSamplePieces + lane) * 2];
            more = list_count[(r * kSamplePieces + lane) * 2 + 1];
        }
    }
    int best = known_best;
    if (!cand_idx) {
        best = block_argmax(row, vocab, s_val, s_idx).index;
        if (best == kNoToken) best = 0;
    }
    if (!(temp > 0.f)) {  // greedy, as the reference for temperature <= 0 (sampler.cpp:46-49)
        if (threadIdx.x == 0) out[r] = best;
        return;
    }
    const int full_vocab = vocab;
    if (direct >= 0) {                               // no cuts: the drawn point's piece is known, walk it
        const int piece = (vocab + kSamplePieces - 1) / kSamplePieces;
        const int begin = min(vocab, direct * piece), n = min(vocab, begin + piece) - begin;
        const int at = pick_in_piece(row, begin, n, row[best], 1.0f / fmaxf(temp, 1e-6f), direct_target[r], s_wave, s_pick);
        if (threadIdx.x == 0) out[r] = at < 0 ? best : at;
        return;
    }
    const float mx = row[best];
    const float inv_t = 1.0f / fmaxf(temp, 1e-6f);
    const bool unordered = is_listed != 0;
    const int row_piece = (full_vocab + kSamplePieces - 1) / kSamplePieces;
    if (unordered) {
        // the pieces' lists: every wavefront adds up what lies before its two pieces, and brings those together
        static_assert(kSamplePieces == 2 * kSampleThreads / kWave, "two pieces to a wavefront");
        int before = count, before_more = more;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int a = __shfl_up(before, o, kWave), b = __shfl_up(before_more, o, kWave);
            if (lane >= o) {
                before += a;
                before_more += b;
            }
        }
        const int tight = __shfl(before, kWave - 1, kWave), loose = __shfl(before_more, kWave - 1, kWave);
        const bool with_loose = tight + loose <= kSampleThreads;
        if (tight <= kSampleThreads) {
            const int n = with_loose ? tight + loose : tight;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int c = 2 * wave + h, mine = __shfl(count, c, kWave), also = with_loose ? __shfl(more, c, kWave) : 0;
                const int to = __shfl(before, c, kWave) - mine, to_more = tight + __shfl(before_more, c, kWave) - __shfl(more, c, kWave);
                const int begin = min(full_vocab, c * row_piece), end = min(full_vocab, begin + row_piece);
                for (int i = lane; i < mine + also; i += kWave) {
                    const int from = i < mine ? begin + i : end - 1 - (i - mine), at = i < mine ? to + i : to_more + i - mine;
                    s_list[at] = w[from];
                    s_order[at] = idx_of[from];
                }
            }
            __syncthreads();
            const int j = threadIdx.x;
            const float wj = j < n ? s_list[j] : 0.f;
            const int ij = j < n ? s_order[j] : 0x7fffffff;
            __syncthreads();
            vocab = order_candidates(wj, ij, n, static_cast<unsigned int>(k), s_list, s_order, hist);
        } else {
            // more than a thousand equals: the thresholds from the list, brought together in the first piece's place and behind it
            // (every piece's part moves towards the front, one piece after the other), the draw from the row
            int to = 0;
            for (int c = 0; c < kSamplePieces; ++c) {
                const int mine = __shfl(count, c, kWave), begin = min(full_vocab, c * row_piece);
                for (int i0 = 0; i0 < mine; i0 += kSampleThreads) {
                    const int i = i0 + threadIdx.x;
                    const float v = i < mine ? w[begin + i] : 0.f;
                    __syncthreads();
                    if (i < mine) w[to + i] = v;
                    __syncthreads();
                }
                to += mine;
            }
            vocab = tight;
        }
    } else if (cand_idx) {
        vocab = cand_count[r];                       // from here on the row is the list of candidates
    } else {
        for_each_in_row(row, vocab, threadIdx.x, blockDim.x, [&](int j, float x) { w[j] = weight_of(x, mx, inv_t); });
        __syncthreads();   // each thread reads back what others wrote: same workgroup, so a barrier suffices
    }
    const bool k_active = k > 0 && k < full_vocab;
    const unsigned long long mass = cand_idx && !k_active ? row_mass[r] : 0ull;
    if (vocab <= kSampleThreads) {                   // a short row or list: one thread per token
        const float wj = unordered ? s_list[threadIdx.x] : static_cast<int>(threadIdx.x) < vocab ? w[threadIdx.x] : 0.f;
        const int at = pick_from_short_list(wj, vocab, k_active && k < vocab, static_cast<unsigned int>(k), p,
                                            cand_idx && !k_active, mass, u, s_list, s_wave, s_piece, s_pick);
        if (threadIdx.x == 0) out[r] = at < 0 ? best : unordered ? s_order[at] : idx_of ? idx_of[at] : at;
        return;
    }
    // kept set = { j : w_j >= threshold }; the threshold starts at 0 (everything)
    uint32_t threshold = 0u;
    if (k_active && k < vocab)        // (a list of exactly k candidates is the top k)
        threshold = select_by_count(w, vocab, static_cast<unsigned int>(k), hist, &s_a, &s_need);
    if (p > 0.f && p < 1.f) {
        // mass of what top-k kept, in fixed point: per-thread sums, then over the wavefronts in order
        unsigned long long mine = 0ull;
        for_each_in_row(w, vocab, threadIdx.x, blockDim.x, [&](int, float wj) {
            if (__float_as_uint(wj) >= threshold) mine += fixed_of(wj);
        });
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) mine += __shfl_xor(mine, o, kWave);
        if (lane == 0) s_wave[wave] = mine;
        __syncthreads();
        unsigned long long kept = 0ull;
        for (int i = 0; i < n_waves; ++i) kept += s_wave[i];
        __syncthreads();
        // (a list of candidates without top-k holds only the upper part of the row: the mass p refers to the whole row)
        if (cand_idx && !k_active) kept = mass;
        unsigned long long need = static_cast<unsigned long long>(static_cast<double>(p) * static_cast<double>(kept));
        if (need == 0ull) need = 1ull;
        uint32_t top = 0x3f800001u;
        unsigned long long above = 0ull;
        if (cand_idx && !k_active) {                 // the bin that holds it is known
            const int bin = last_bin[r];
            threshold = bin < kTopBins ? static_cast<uint32_t>(127 - bin) << 23 : 0u;
            top = bin == 0 ? 0x3f800001u : static_cast<uint32_t>(128 - min(bin, kTopBins)) << 23;
            above = direct_target[r];
        }
        threshold = select_by_mass(w, vocab, threshold, top, above, need, s_wave, &s_a, &s_b, &s_above);
    }
    // inverse CDF in index order.  Every wavefront owns a contiguous piece of the row; the piece that holds the
    // drawn point is then walked 64 tokens at a time with a prefix sum over the lanes.
    if (unordered) vocab = full_vocab;
    auto weight_or_none = [&](float x) { return x <= mx ? weight_of(x, mx, inv_t) : 0.f; };      // (a NaN is no candidate)
    const int piece = ((vocab + n_waves - 1) / n_waves + kWave - 1) / kWave * kWave;
    const int p_begin = min(vocab, wave * piece), p_end = min(vocab, p_begin + piece);
    float mine = 0.f;
    for_each_in_row((unordered ? row : w) + p_begin, p_end - p_begin, lane, kWave, [&](int, float wj) {
        if (unordered) wj = weight_or_none(wj);
        mine += __float_as_uint(wj) >= threshold ? wj : 0.f;
    });
    mine = wave_sum(mine);
    if (lane == 0) s_piece[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
        for (int i = 0; i < n_waves; ++i) total += s_piece[i];
        const float target = fminf(fmaxf(u, 0.f), 0.99999994f) * total;
        float cum = 0.f;
        int owner = -1;
        float before = 0.f;
        for (int i = 0; i < n_waves; ++i) {
            if (s_piece[i] > 0.f) {
                owner = i;                      // the last piece with mass catches rounding at the end
                before = cum;
                if (cum + s_piece[i] > target) break;
            }
            cum += s_piece[i];
        }
        s_owner = owner;
        s_before = target - before;             // what is left of the target inside the owner's piece
        if (owner < 0) out[r] = best;
    }
    __syncthreads();
    if (wave == s_owner) {
        const float target = s_before;
        float cum = 0.f;
        int pick = -1, last_kept = -1;
        for (int base = p_begin; base < p_end && pick < 0; base += kWave) {
            const int j = base + lane;
            float wj = 0.f;
            if (j < p_end) {
                const float v = unordered ? weight_or_none(row[j]) : w[j];
                wj = __float_as_uint(v) >= threshold ? v : 0.f;
            }
            float incl = wj;                     // inclusive prefix sum over the lanes
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const float up = __shfl_up(incl, o, kWave);
                if (lane >= o) incl += up;
            }
            const unsigned long long kept_mask = __ballot(wj > 0.f);
            const unsigned long long hit = __ballot(wj > 0.f && cum + incl > target);
            if (kept_mask) last_kept = base + 63 - __clzll(static_cast<long long>(kept_mask));
            if (hit) pick = base + __ffsll(static_cast<long long>(hit)) - 1;
            cum += __shfl(incl, kWave - 1, kWave);
        }
        if (lane == 0) {
            const int at = pick >= 0 ? pick : last_kept;
            out[r] = at < 0 ? best : (idx_of && !unordered ? idx_of[at] : at);
        }
    }
}

}  // namespace egpt

using namespace egpt;

// scratch: room for n_rows * 32 floats and n_rows * 32 int32 (used for wide vocabularies), or null.
extern "C" int egpt_argmax(const float* logits, int32_t* out, void* scratch, int n_rows, int vocab, void* stream) {
    if (!logits || !out || n_rows < 0 || vocab <= 0) return EGPT_BAD_ARGUMENT;
    if (n_rows == 0) return EGPT_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (scratch && vocab >= 8192) {
        float* pv = static_cast<float*>(scratch);
        int32_t* pi = reinterpret_cast<int32_t*>(pv + static_cast<size_t>(n_rows) * kArgmaxPieces);
        argmax_pieces_kernel<<<dim3(n_rows, kArgmaxPieces), 256, 0, s>>>(logits, pv, pi, nullptr, vocab);
        EGPT_CHECK_LAUNCH();
        argmax_pick_kernel<<<n_rows, kWave, 0, s>>>(pv, pi, out);
    } else {
        argmax_kernel<<<n_rows, kSampleThreads, 0, s>>>(logits, out, vocab);
    }
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

// ---- the same search without a workspace argument and without any allocation: the pieces live in the library's
// device image.  In host code `argmax_static_scratch` is only a stand-in for the symbol: the memory's address on
// a device comes from hipGetSymbolAddress with that device current, and every GPU has its own copy.
static __device__ __align__(256) unsigned char argmax_static_scratch[EGPT_ARGMAX_STATIC_MAX_ROWS * kArgmaxPieces * 8];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_static_mutex;
void* g_static_ptr[kMaxDevices] = {};

// The buffer's address on the current device, resolved once per device; null on failure.
void* static_scratch_of_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_static_mutex);
    if (!g_static_ptr[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(argmax_static_scratch)) != hipSuccess) return nullptr;
        g_static_ptr[dev] = ptr;
    }
    return g_static_ptr[dev];
}
}  // namespace

extern "C" int egpt_argmax_static_init(void) {
    return static_scratch_of_current_device() ? EGPT_OK : EGPT_STATIC_SCRATCH_UNRESOLVED;
}

extern "C" int egpt_argmax_static(const float* logits, int32_t* out, int n_rows, int vocab, void* stream) {
    if (!logits || !out || n_rows < 0 || vocab <= 0) return EGPT_BAD_ARGUMENT;
    if (n_rows > EGPT_ARGMAX_STATIC_MAX_ROWS) return EGPT_STATIC_SCRATCH_TOO_SMALL;
    if (n_rows == 0) return EGPT_OK;
    void* scratch = static_scratch_of_current_device();
    if (!scratch) return EGPT_STATIC_SCRATCH_UNRESOLVED;
    return egpt_argmax(logits, out, scratch, n_rows, vocab, stream);
}

// weights: scratch for n_rows * vocab floats.
extern "C" int egpt_sample(const float* logits, const float* temperature, const int32_t* top_k, const float* top_p,
                           const float* uniform, int32_t* out, float* weights, int n_rows, int vocab, void* stream) {
    if (!logits || !temperature || !top_k || !top_p || !uniform || !out || !weights || n_rows < 0 || vocab <= 0)
        return EGPT_BAD_ARGUMENT;
    if (n_rows == 0) return EGPT_OK;
    sample_kernel<<<n_rows, kSampleThreads, 0, static_cast<hipStream_t>(stream)>>>(
        logits, temperature, top_k, top_p, uniform, out, weights, vocab, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

// The same for wide vocabularies, in stages (maxima of pieces, counts by exponent, the list of candidates, the selection
// on the list).  workspace: egpt_sample_workspace(n_rows, vocab) bytes of device memory.
static size_t align256(size_t n) { return (n + 255) / 256 * 256; }

extern "C" size_t egpt_sample_workspace(int n_rows, int vocab) {
    const size_t r = static_cast<size_t>(n_rows > 0 ? n_rows : 0), v = static_cast<size_t>(vocab > 0 ? vocab : 0);
    return align256(r * v * 4) * 2                                         // candidates: weights, indices
           + align256(r * kSamplePieces * (kTopBins + 1) * 8)            // masses
           + align256(r * kSamplePieces * (kTopBins + 1) * 4)            // counts
           + align256(r * 4) * 2                                           // number of candidates, best
           + align256(r * 8) * 2 + align256(r * 4)                         // mass of the row; the direct draw's point, piece
           + align256(r * 4) * 2 + align256(r * kSamplePieces * 8) + align256(r * kSubPieces * 4)  // lists by the maxima, the shares' maxima
           + align256(r * kArgmaxPieces * 8);                              // argmax pieces
}

extern "C" int egpt_sample_wide(const float* logits, const float* temperature, const int32_t* top_k, const float* top_p,
                                const float* uniform, int32_t* out, void* workspace, int n_rows, int vocab, void* stream) {
    if (!logits || !temperature || !top_k || !top_p || !uniform || !out || !workspace || n_rows < 0 || vocab <= 0)
        return EGPT_BAD_ARGUMENT;
    if (n_rows == 0) return EGPT_OK;
    if (n_rows > 65535) return EGPT_UNSUPPORTED_SIZE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t r = static_cast<size_t>(n_rows), v = static_cast<size_t>(vocab);
    char* p = static_cast<char*>(workspace);
    float* cand_w = reinterpret_cast<float*>(p);                               p += align256(r * v * 4);
    int32_t* cand_idx = reinterpret_cast<int32_t*>(p);                         p += align256(r * v * 4);
    unsigned long long* piece_mass = reinterpret_cast<unsigned long long*>(p); p += align256(r * kSamplePieces * (kTopBins + 1) * 8);
    unsigned int* piece_count = reinterpret_cast<unsigned int*>(p);            p += align256(r * kSamplePieces * (kTopBins + 1) * 4);
    int32_t* cand_count = reinterpret_cast<int32_t*>(p);                       p += align256(r * 4);
    int32_t* best = reinterpret_cast<int32_t*>(p);                             p += align256(r * 4);
    unsigned long long* row_mass = reinterpret_cast<unsigned long long*>(p);   p += align256(r * 8);
    unsigned long long* direct_target = reinterpret_cast<unsigned long long*>(p); p += align256(r * 8);
    int32_t* direct_piece = reinterpret_cast<int32_t*>(p);                     p += align256(r * 4);
    int32_t* last_bin = reinterpret_cast<int32_t*>(p);                         p += align256(r * 4);
    int32_t* listed = reinterpret_cast<int32_t*>(p);                           p += align256(r * 4);
    int32_t* list_count = reinterpret_cast<int32_t*>(p);                       p += align256(r * kSamplePieces * 8);
    float* sub = reinterpret_cast<float*>(p);                                  p += align256(r * kSubPieces * 4);
    float* pv = reinterpret_cast<float*>(p);
    int32_t* pi = reinterpret_cast<int32_t*>(pv + r * kArgmaxPieces);
    argmax_pieces_kernel<<<dim3(n_rows, kArgmaxPieces), 256, 0, s>>>(logits, pv, pi, sub, vocab);
    EGPT_CHECK_LAUNCH();
    sample_count_kernel<<<dim3(n_rows, kSamplePieces), 256, 0, s>>>(logits, temperature, top_k, pv, pi, sub, best, listed, list_count, cand_w, cand_idx,
                                                                    piece_count, piece_mass, vocab);
    EGPT_CHECK_LAUNCH();
    sample_compact_kernel<<<dim3(n_rows, kSamplePieces), 256, 0, s>>>(logits, temperature, top_k, top_p, uniform, best, piece_count,
                                                                      piece_mass, listed, cand_w, cand_idx, cand_count, row_mass,
                                                                      direct_piece, direct_target, last_bin, vocab);
    EGPT_CHECK_LAUNCH();
    sample_kernel<<<n_rows, kSampleThreads, 0, s>>>(logits, temperature, top_k, top_p, uniform, out, cand_w, vocab, cand_idx,
                                                    cand_count, listed, list_count, best, row_mass, direct_piece, direct_target, last_bin);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}
