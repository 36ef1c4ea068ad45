// Paged attention on the matrix cores (bfloat16), for prompt portions and decoded tokens alike.
//
// A wavefront owns QT tiles of 16 query rows of one request and one key/value head.  A row is a
// (token, query head) pair of the head's group, token-major, so the 7 heads of a decoded token share one
// tile (and every load of its keys), and the rows of a prompt tile have nearly the same causal limit.
// Keys are walked 32 at a time.  The scores are computed transposed,
//     S^T[key, row] = K[key, :] . Q[row, :]        v_mfma_f32_16x16x32_bf16, A = K, B = Q
// so that a lane ends up with the scores of ONE row (its column) for four keys per tile: the row's
// running maximum and sum are per-lane scalars, and the probabilities are, as they lie in registers,
// the B operand of the second product
//     O^T[feature, row] += V^T[feature, key] . P^T[key, row]     A = V^T, B = P^T
// whose A operand is what a page of values looks like in memory (values are stored transposed within
// a page).  No operand passes through LDS.  Softmax statistics and the accumulator are float32
// (as /root/reference/src/cuda/ops/self_attn_detail.cuh:299-383); P is rounded to bfloat16 for the
// second product.  With n_splits > 1 each split of the key range writes an unnormalised partial result
// and its (maximum, sum), which attention_reduce_kernel combines.
#include <type_traits>
#include <utility>

#include "api.h"
#include "common.h"
#include "lds_loads.h"

namespace egpt {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <int HD, int QT>
__global__ __launch_bounds__(64) void attention_mfma_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ q_len, const int32_t* __restrict__ kv_len, int n_seqs, int n_tokens, int nq, int nkv,
    int page_size, float scale, int window, int n_splits) {
    constexpr int KD = HD / 32;  // score MFMAs per key tile (32 features each)
    constexpr int DT = HD / 16;  // output feature tiles
    const int lane = threadIdx.x, lj = lane % 16, lg = lane / 16;
    const int kh = blockIdx.y, split = blockIdx.z;
    const int group_size = nq / nkv;

    // which request, and which group of 16*QT rows of it; within a request the last rows come first: they
    // have the most keys to walk, and the launch is over when the longest wavefront is
    int b, grp;
    auto groups_of = [&](int n) { return (n * group_size + 16 * QT - 1) / (16 * QT); };
    if (!find_block(q_len, n_seqs, blockIdx.x, groups_of, b, grp)) return;
    grp = groups_of(q_len[b]) - 1 - grp;
    const int n = q_len[b], kv = kv_len[b], qs = q_start[b];
    const int rows = n * group_size;
    const int row_base = grp * 16 * QT;
    const int width = (nq + 2 * nkv) * HD;
    const int32_t* table = block_table + static_cast<size_t>(b) * table_width;

    // this lane's row in each tile
    bool valid[QT];
    int tok[QT], head[QT], p_row[QT], lo_row[QT];
    bf16x8 q[QT][KD];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const int r = row_base + t * 16 + lj;
        valid[t] = r < rows;
        const int i = valid[t] ? r / group_size : 0;
        tok[t] = qs + i;
        head[t] = kh * group_size + (valid[t] ? r % group_size : 0);
        p_row[t] = valid[t] ? kv - n + i : -1;
        lo_row[t] = (window > 0 && valid[t]) ? max(0, p_row[t] - window + 1) : 0;
        const bf16_t* qp = qkv + static_cast<size_t>(tok[t]) * width + head[t] * HD + lg * 8;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) {
            uint4 v = valid[t] ? *reinterpret_cast<const uint4*>(qp + kd * 32) : uint4{0u, 0u, 0u, 0u};
            q[t][kd] = __builtin_bit_cast(bf16x8, v);
        }
    }
    const float scale2 = scale * 1.4426950408889634f;   // scores are kept in units of log 2
    // the smallest causal limit and the largest window start among the valid rows of each tile
    int p_min[QT], lo_max[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const int r_first = row_base + t * 16, r_last = min(rows, r_first + 16) - 1;
        const bool any = r_first < rows;
        p_min[t] = any ? kv - n + r_first / group_size : -1;
        const int p_last = any ? kv - n + r_last / group_size : -1;
        lo_max[t] = window > 0 ? max(0, p_last - window + 1) : 0;
    }
    // key blocks (32 keys) this wave needs, and this split's share of them
    const int last_row = min(rows, row_base + 16 * QT) - 1;
    const int p_hi = kv - n + last_row / group_size;
    const int first_pos = kv - n + row_base / group_size;
    const int lo_first = window > 0 ? max(0, first_pos - window + 1) : 0;
    const int kb_begin = lo_first / 32, kb_end = p_hi / 32 + 1;
    const int per_split = (kb_end - kb_begin + n_splits - 1) / n_splits;
    const int my_begin = kb_begin + split * per_split;
    const int my_end = min(kb_end, my_begin + per_split);

    f32x4 o[QT][DT];
    float m_run[QT], l_run[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        m_run[t] = -INFINITY;
        l_run[t] = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) o[t][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // Keys are walked in rounds of kRound blocks of 32; the loads of the next round are in flight while this
    // round computes (a wavefront is alone on its SIMD here, so nothing else hides the latency).
    constexpr int kRound = 2;
    uint4 k_cur[kRound][2][KD], k_nxt[kRound][2][KD];
    uint2 v_cur[kRound][2][DT], v_nxt[kRound][2][DT];
    auto load_round = [&](uint4 (*kk)[2][KD], uint2 (*vv)[2][DT], int kb0) {
        int pages[kRound][2];
        bool live[kRound][2];
#pragma unroll
        for (int i = 0; i < kRound; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const int key0 = (kb0 + i) * 32 + kt * 16;
                // a tile is read only if some row of this wave can see one of its keys: then it lies in a page the
                // request still holds (p_hi < kv; pages wholly behind the window may have been given back)
                live[i][kt] = kb0 + i < my_end && key0 <= p_hi && key0 + 15 >= lo_first;
                pages[i][kt] = table[live[i][kt] ? key0 / page_size : 0];
            }
#pragma unroll
        for (int i = 0; i < kRound; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const int key0 = (kb0 + i) * 32 + kt * 16;
                const bool ok = live[i][kt] && pages[i][kt] >= 0;
                const long page = ok ? pages[i][kt] : 0;
                const int off = ok ? key0 % page_size : 0;
                const bf16_t* kp = k_cache + ((page * nkv + kh) * page_size + off + lj) * HD + lg * 8;
                const bf16_t* vp = v_cache + ((page * nkv + kh) * HD + lj) * static_cast<long>(page_size) + off + lg * 4;
#pragma unroll
                for (int kd = 0; kd < KD; ++kd)
                    kk[i][kt][kd] = ok ? *reinterpret_cast<const uint4*>(kp + kd * 32) : uint4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int d = 0; d < DT; ++d)
                    vv[i][kt][d] = ok ? *reinterpret_cast<const uint2*>(vp + static_cast<long>(d) * 16 * page_size)
                                      : uint2{0u, 0u};
            }
    };

    if (my_begin < my_end) load_round(k_cur, v_cur, my_begin);
    for (int kb0 = my_begin; kb0 < my_end; kb0 += kRound) {
        if (kb0 + kRound < my_end) load_round(k_nxt, v_nxt, kb0 + kRound);
#pragma unroll
        for (int i = 0; i < kRound; ++i) {
            const int kb = kb0 + i;
            if (kb >= my_end) break;
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                // scores in units of log 2: s = (q . k) * scale * log2(e), so that exp is one v_exp_f32
                float s[2][4];
                float mx = -INFINITY;
                // most blocks lie wholly below the diagonal (and inside the window) for every row of the tile:
                // they need no masking
                const bool all_visible = kb * 32 + 31 <= p_min[t] && kb * 32 >= lo_max[t];
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kd = 0; kd < KD; ++kd)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k_cur[i][kt][kd]),
                                                                      q[t][kd], acc, 0, 0, 0);
                    if (all_visible) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            s[kt][v] = acc[v] * scale2;
                            mx = fmaxf(mx, s[kt][v]);
                        }
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int key = kb * 32 + kt * 16 + lg * 4 + v;
                            const bool vis = key <= p_row[t] && key >= lo_row[t];
                            s[kt][v] = vis ? acc[v] * scale2 : -INFINITY;
                            mx = fmaxf(mx, s[kt][v]);
                        }
                    }
                }
                mx = fold_rows(mx, MaxOf());
                const float m_new = fmaxf(m_run[t], mx);
                // a row without any visible key so far keeps maximum -inf; subtracting a finite stand-in makes
                // every exp below 0 without a special case (exp2(-inf) = 0)
                const float m_use = m_new == -INFINITY ? 0.f : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m_run[t] - m_use);
                float sum = 0.f;
                bf16x8 pb;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float pv = __builtin_amdgcn_exp2f(s[kt][v] - m_use);
                        sum += pv;
                        pb[kt * 4 + v] = static_cast<__bf16>(pv);
                    }
                l_run[t] = l_run[t] * alpha + sum;
                m_run[t] = m_new;
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    const uint4 a = uint4{v_cur[i][0][d].x, v_cur[i][0][d].y, v_cur[i][1][d].x, v_cur[i][1][d].y};
                    f32x4 acc = o[t][d];
                    acc[0] *= alpha; acc[1] *= alpha; acc[2] *= alpha; acc[3] *= alpha;
                    o[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), pb, acc, 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kRound; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
                for (int kd = 0; kd < KD; ++kd) k_cur[i][kt][kd] = k_nxt[i][kt][kd];
#pragma unroll
                for (int d = 0; d < DT; ++d) v_cur[i][kt][d] = v_nxt[i][kt][d];
            }
    }

#pragma unroll
    for (int t = 0; t < QT; ++t) {
        float l = l_run[t];
        l = fold_rows(l, AddOf());
        if (!valid[t]) continue;
        const size_t row = static_cast<size_t>(tok[t]) * nq + head[t];
        if (n_splits == 1) {
            const float inv = 1.0f / l;
            bf16_t* op = out + row * HD + lg * 4;
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                uint2 packed;
                packed.x = bf16_pair(o[t][d][0] * inv, o[t][d][1] * inv);
                packed.y = bf16_pair(o[t][d][2] * inv, o[t][d][3] * inv);
                *reinterpret_cast<uint2*>(op + d * 16) = packed;
            }
        } else {
            const size_t prow = static_cast<size_t>(split) * n_tokens * nq + row;
            float* pp = part_o + prow * HD + lg * 4;
#pragma unroll
            for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(pp + d * 16) = o[t][d];
            if (lg == 0) {
                part_ml[prow * 2] = m_run[t] * 0.6931471805599453f;      // back to natural units for the combine
                part_ml[prow * 2 + 1] = l;
            }
        }
    }
}

// Prompt portions.  A workgroup takes RT tiles of 16 rows (of one request and kv head) and walks the keys in
// tiles of 64 * KS, which are staged through LDS and shared by its RT * KS wavefronts; wavefront (rt, ks)
// multiplies row tile rt with the ks-th 64 keys of each tile, and the KS partial results of a row tile are
// combined through LDS at the end.  The next tile's loads are in flight while this one is computed.
// Without the sharing every wavefront reads all of its keys from L2 itself (about 0.5 GB per layer for a
// 2,048-token prompt at these sizes).  A wavefront issues a vector instruction in four cycles, and a prompt
// of a few thousand tokens gives each SIMD only a few wavefronts, so what a tile costs is the vector
// instructions and the waits between them rather than the matrix cores: hence 64 keys per softmax step, the
// accumulator rescaled only when a row's maximum moved, and the split of the keys over wavefronts.
// The arithmetic is that of attention_mfma_kernel.
template <int HD, int RT, int KS>
__global__ __launch_bounds__(64 * RT * KS) void attention_tiled_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_table, int table_width,
    const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len, const int32_t* __restrict__ kv_len,
    int n_seqs, int nq, int nkv, int page_size, int page_shift, float scale, int window, int skip_single) {
    constexpr int KD = HD / 32, DT = HD / 16;
    constexpr int ROWS = 16 * RT;                // rows per workgroup
    constexpr int KT = 64 * KS;                  // keys per LDS tile
    constexpr int KROW = HD + 8, VROW = KT + 8;  // padded rows (bf16 elements)
    constexpr int THREADS = 64 * RT * KS;
    constexpr int CH = HD / (8 * RT);            // 16-byte chunks per thread and tile, of keys and of values
    constexpr int STAGE = KT * KROW + HD * VROW;  // bf16 elements per stage
    constexpr int COMBINE = (KS - 1) * RT * 64 * (DT * 4 + 2) * 2;    // the combination's floats, in bf16 elements
    static_assert(CH >= 1 && HD % (8 * RT) == 0, "a thread takes whole chunks");
    __shared__ __attribute__((aligned(16))) bf16_t smem[(2 * STAGE > COMBINE) ? 2 * STAGE : COMBINE];
    auto ks_at = [&](int stage, int key, int col) -> bf16_t* { return smem + stage * STAGE + key * KROW + col; };
    auto vs_at = [&](int stage, int d, int key) -> bf16_t* { return smem + stage * STAGE + KT * KROW + d * VROW + key; };
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int rt = wave % RT, ksi = wave / RT;
    const int lj = lane % 16, lg = lane / 16;
    const int kh = blockIdx.y;
    const int group_size = nq / nkv;

    int b, grp;
    // (skip_single: requests of one token are the decode kernel's, which spreads their keys over wavefronts)
    auto groups_of = [&](int n) { return (skip_single && n == 1) ? 0 : (n * group_size + ROWS - 1) / ROWS; };
    if (!find_block(q_len, n_seqs, blockIdx.x, groups_of, b, grp)) return;
    grp = groups_of(q_len[b]) - 1 - grp;     // the last rows first: they have the most keys to walk
    const int n = q_len[b], kv = kv_len[b], qs = q_start[b];
    const int rows = n * group_size;
    const int width = (nq + 2 * nkv) * HD;
    const int32_t* table = block_table + static_cast<size_t>(b) * table_width;

    // the workgroup's rows and the keys they need
    const int blk_first = grp * ROWS, blk_last = min(rows, blk_first + ROWS) - 1;
    const int blk_p_hi = kv - n + blk_last / group_size;
    const int blk_first_pos = kv - n + blk_first / group_size;
    const int blk_lo = window > 0 ? max(0, blk_first_pos - window + 1) : 0;
    const int t_begin = blk_lo / KT, t_end = blk_p_hi / KT + 1;

    // this wavefront's tile of 16 rows, this lane's row
    const int row_base = blk_first + rt * 16;
    const int r = row_base + lj;
    const bool valid = r < rows;
    const int i_tok = valid ? r / group_size : 0;
    const int tok = qs + i_tok;
    const int head = kh * group_size + (valid ? r % group_size : 0);
    const int p_row = valid ? kv - n + i_tok : -1;
    const int lo_row = (window > 0 && valid) ? max(0, p_row - window + 1) : 0;
    const bool wave_any = row_base < rows;
    const int w_last = min(rows, row_base + 16) - 1;
    const int w_p_hi = wave_any ? kv - n + w_last / group_size : -1;       // largest causal limit in the tile
    const int w_p_min = wave_any ? kv - n + row_base / group_size : -1;    // smallest
    const int w_lo_first = (window > 0 && wave_any) ? max(0, w_p_min - window + 1) : 0;
    const int w_lo_max = (window > 0 && wave_any) ? max(0, w_p_hi - window + 1) : 0;
    bf16x8 q[KD];
    {
        const bf16_t* qp = qkv + static_cast<size_t>(tok) * width + head * HD + lg * 8;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) {
            const uint4 v = valid ? *reinterpret_cast<const uint4*>(qp + kd * 32) : uint4{0u, 0u, 0u, 0u};
            q[kd] = __builtin_bit_cast(bf16x8, v);
        }
    }
    const float scale2 = scale * 1.4426950408889634f;

    f32x4 o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY;                  // the maximum in units of the raw scores
    // The rows' sums of probabilities are left to the matrix cores: one more tile of "values" whose first feature is
    // all ones (lanes lj == 0 hold it, the other features are zeros) gives sum_key P[key, row] as feature 0 of a
    // 17th output tile, in element 0 of the lanes lg == 0.  (Sixteen additions per step on the vector pipe, which is
    // what this kernel waits for, against two matrix instructions on a pipe that is idle seven eighths of the time.)
    f32x4 o_sum = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<__bf16>(lj == 0 ? 1.0f : 0.0f);

    // The loads of a tile go through three stages, each one iteration ahead of the next, so that no load
    // waits for another inside an iteration: page numbers (tile + 2), keys and values into registers
    // (tile + 1), registers into LDS after the products of this tile.  A thread's chunks of a tile lie in
    // one page (keys: CH chunks of one key; values: eight keys of CH features), so a tile costs it two
    // table entries and two addresses.
    const int page_mask = page_size - 1;             // page sizes here are powers of two
    const int k_row = tid / RT, k_col = (tid % RT) * CH * 8;                 // key within the tile, first feature
    const int v_key = (tid % (KT / 8)) * 8, v_row = tid / (KT / 8);          // first of eight keys, feature (+ 8 RT u)
    uint4 k_regs[CH], v_regs[CH];
    int k_page, v_page;                              // -1: nothing to read (zeros)
    auto lookup = [&](int tile) {
        const int kk = tile * KT + k_row, vk = tile * KT + v_key;
        k_page = (kk <= blk_p_hi && kk >= blk_lo) ? table[kk >> page_shift] : -1;
        v_page = (vk <= blk_p_hi && vk + 7 >= blk_lo) ? table[vk >> page_shift] : -1;
    };
    auto fetch = [&](int tile) {
        const int kk = tile * KT + k_row, vk = tile * KT + v_key;
        if (k_page >= 0) {
            const bf16_t* src = k_cache + ((static_cast<long>(k_page) * nkv + kh) * page_size + (kk & page_mask)) * HD + k_col;
#pragma unroll
            for (int u = 0; u < CH; ++u) k_regs[u] = *reinterpret_cast<const uint4*>(src + u * 8);
        } else {
#pragma unroll
            for (int u = 0; u < CH; ++u) k_regs[u] = uint4{0u, 0u, 0u, 0u};
        }
        if (v_page >= 0) {
            const bf16_t* src = v_cache + ((static_cast<long>(v_page) * nkv + kh) * HD + v_row) * page_size + (vk & page_mask);
#pragma unroll
            for (int u = 0; u < CH; ++u)
                v_regs[u] = *reinterpret_cast<const uint4*>(src + static_cast<long>(u) * (8 * RT) * page_size);
        } else {
#pragma unroll
            for (int u = 0; u < CH; ++u) v_regs[u] = uint4{0u, 0u, 0u, 0u};
        }
    };
    // Where this thread puts its chunks, and where this lane reads its operands, in either stage: the loop below is
    // unrolled over the two stages, so that every LDS access is one of these registers plus an immediate offset.
    bf16_t* const k_put[2] = {ks_at(0, k_row, k_col), ks_at(1, k_row, k_col)};
    bf16_t* const v_put[2] = {vs_at(0, v_row, v_key), vs_at(1, v_row, v_key)};
    const bf16_t* const k_get[2] = {ks_at(0, ksi * 64 + lj, lg * 8), ks_at(1, ksi * 64 + lj, lg * 8)};
    const bf16_t* const v_get[2] = {vs_at(0, lj, ksi * 64 + lg * 4), vs_at(1, lj, ksi * 64 + lg * 4)};
    auto stash = [&](auto stage_c) {
        constexpr int stage = decltype(stage_c)::value;
#pragma unroll
        for (int u = 0; u < CH; ++u) {
            *reinterpret_cast<uint4*>(k_put[stage] + u * 8) = k_regs[u];
            *reinterpret_cast<uint4*>(v_put[stage] + u * 8 * RT * VROW) = v_regs[u];
        }
    };
    auto walk = [&](auto stage_c, int tile) {
        constexpr int stage = decltype(stage_c)::value;
        fetch(tile + 1);           // past the last tile every page number is -1: nothing is read
        lookup(tile + 2);
        const int key0 = tile * KT + ksi * 64;       // this wavefront's 64 keys
        if (wave_any && key0 <= w_p_hi && key0 + 63 >= w_lo_first) {     // else nothing visible to these rows
            // S^T = K Q^T: lane (lj, lg) holds keys kt*16 + lg*4 + v of row lj
            f32x4 acc[4];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                acc[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kd = 0; kd < KD; ++kd) {
                    const uint4 kk = *reinterpret_cast<const uint4*>(k_get[stage] + kt * 16 * KROW + kd * 32);
                    acc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kk), q[kd], acc[kt], 0, 0, 0);
                }
            }
            if (!(key0 + 63 <= w_p_min && key0 >= w_lo_max)) {           // on the diagonal or the window's edge
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int key = key0 + kt * 16 + lg * 4 + v;
                        if (!(key <= p_row && key >= lo_row)) acc[kt][v] = -INFINITY;
                    }
            }
            float mx = fmaxf(fmaxf(acc[0][0], acc[0][1]), fmaxf(acc[0][2], acc[0][3]));
#pragma unroll
            for (int kt = 1; kt < 4; ++kt) mx = fmaxf(mx, fmaxf(fmaxf(acc[kt][0], acc[kt][1]), fmaxf(acc[kt][2], acc[kt][3])));
            mx = fold_rows(mx, MaxOf());
            const float m_new = fmaxf(m_run, mx);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            if (__any(m_new != m_run)) {             // some row's maximum moved: rescale what is accumulated
                const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * scale2);
                o_sum[0] *= alpha;
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    o[d][0] *= alpha; o[d][1] *= alpha; o[d][2] *= alpha; o[d][3] *= alpha;
                }
                m_run = m_new;
            }
            const float shift = -m_use * scale2;
            bf16x8 pb[2];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    pb[kt / 2][(kt % 2) * 4 + v] = static_cast<__bf16>(__builtin_amdgcn_exp2f(fmaf(acc[kt][v], scale2, shift)));
            // O^T += V^T P^T, two products of 32 keys per 16 features, and the tile of ones for the rows' sums
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) o_sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[kb], o_sum, 0, 0, 0);
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const uint2 v0 = *reinterpret_cast<const uint2*>(v_get[stage] + d * 16 * VROW + kb * 32);
                    const uint2 v1 = *reinterpret_cast<const uint2*>(v_get[stage] + d * 16 * VROW + kb * 32 + 16);
                    const uint4 a = uint4{v0.x, v0.y, v1.x, v1.y};
                    o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), pb[kb], o[d], 0, 0, 0);
                }
        }
        stash(std::integral_constant<int, stage ^ 1>{});
        __syncthreads();
    };

    lookup(t_begin);
    fetch(t_begin);
    lookup(t_begin + 1);
    stash(std::integral_constant<int, 0>{});
    __syncthreads();
    for (int tile = t_begin; tile < t_end; tile += 2) {
        walk(std::integral_constant<int, 0>{}, tile);
        if (tile + 1 < t_end) walk(std::integral_constant<int, 1>{}, tile + 1);
    }
    // the row's sum: feature 0 of the tile of ones, which the lane lj of the first quarter holds
    float l = __shfl(o_sum[0], lj, kWave);
    if constexpr (KS > 1) {
        // The wavefronts of one row tile hold partial results over their keys: those with ks > 0 leave
        // theirs in LDS (the tiles are no longer read: the loop ended with a barrier), ks == 0 adds them up.
        constexpr int PER_LANE = DT * 4 + 2;
        float* comb = reinterpret_cast<float*>(smem);
        if (ksi > 0) {
            float* dst = comb + (static_cast<size_t>((ksi - 1) * RT + rt) * PER_LANE) * 64 + lane;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int v = 0; v < 4; ++v) dst[(d * 4 + v) * 64] = o[d][v];
            dst[(DT * 4) * 64] = m_run;
            dst[(DT * 4 + 1) * 64] = l;
        }
        __syncthreads();
        if (ksi > 0) return;
        float m_all = m_run;
#pragma unroll
        for (int j = 0; j < KS - 1; ++j)
            m_all = fmaxf(m_all, comb[(static_cast<size_t>(j * RT + rt) * PER_LANE + DT * 4) * 64 + lane]);
        const float m_ref = m_all == -INFINITY ? 0.f : m_all;
        const float w0 = __builtin_amdgcn_exp2f((m_run - m_ref) * scale2);
        // (written as fused operations so that the rounding doesn't go by what the compiler does with the code around)
#pragma unroll
        for (int j = 0; j < KS - 1; ++j) {
            const float* src = comb + (static_cast<size_t>(j * RT + rt) * PER_LANE) * 64 + lane;
            const float wj = __builtin_amdgcn_exp2f((src[(DT * 4) * 64] - m_ref) * scale2), lj = src[(DT * 4 + 1) * 64];
            l = j == 0 ? fmaf(l, w0, lj * wj) : fmaf(lj, wj, l);
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int v = 0; v < 4; ++v) o[d][v] = fmaf(src[(d * 4 + v) * 64], wj, j == 0 ? o[d][v] * w0 : o[d][v]);
        }
    }
    if (valid) {
        const float inv = 1.0f / l;
        bf16_t* op = out + (static_cast<size_t>(tok) * nq + head) * HD + lg * 4;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            uint2 packed;
            packed.x = bf16_pair(o[d][0] * inv, o[d][1] * inv);
            packed.y = bf16_pair(o[d][2] * inv, o[d][3] * inv);
            *reinterpret_cast<uint2*>(op + d * 16) = packed;
        }
    }
}

// Prompt portions, 32 rows to a wavefront.  The same arithmetic as attention_tiled_kernel with the 32 x 32 x 16 matrix
// instruction: a wavefront takes a block of 32 rows and 64 keys of each tile, S^T[32 keys, 32 rows] = K Q^T leaves a lane
// 16 scores of one row (row = lane % 32), and the probabilities are again the second product's operand as they lie.  Against
// the kernel of 16-row tiles, a score costs half the matrix instructions and half the LDS reads; what is left per score is its
// exponential, a multiply-add, half a maximum and half a conversion.  A workgroup takes RB blocks
// of rows; KS wavefronts per block split each tile of 64 * KS keys and are combined through LDS at the end.  The tiles
// of 64 keys must be whole pages (page sizes 16, 32, 64).
//
// What bounds it: the vector instructions of the softmax.  A block of 32 rows and 64 keys is 143 of them by the counters (an exponential
// takes a wavefront's issue slot for about 8.5 cycles, the others for 4.4: some 800 cycles with the matrix instructions of the SIMD's other
// wavefront between them), against 640 cycles of the matrix cores at head size 64 and 1,152 at 128.  With two wavefronts to a SIMD
// that take matrix and vector instructions in turns a step of both takes 1,000 to 1,300 cycles.  What it was before: one straight line of
// code that alternated matrix and vector instructions, keys and values through registers into LDS (184 vector instructions a
// block by the counters, bank conflicts, every load waited for in front of the iteration's barrier), four wavefronts a CU at head size 128, and a
// block without rows masked in every tile, by which a prompt whose last rows fill their workgroup badly took half as long again.  us a
// layer: 14 heads of 64 on 2, 2,048 / 6,000 / 8,191 tokens 25.9 / 117 / 171 -> 25.1 / 96 / 146; 12 heads of 128 on 2, 1,024 / 2,048 / 5,000
// 25.9 / 47.2 / 136 -> 21.0 / 32.8 / 88.6; 28 on 4, 1,024 / 2,048 / 5,000 29.5 / 72.9 / 289 -> 22.6 / 46.0 / 178.
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;      // (native vectors: arrays of them stay in registers)
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

// max(a, b, c) in one instruction.  (fmaxf quiets signalling NaNs first, which costs an instruction per operand that
// comes from the matrix cores; scores are never NaN here.)
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), in this order
template <int... I, class F>
__device__ __forceinline__ void static_for_each(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_each(std::make_integer_sequence<int, N>{}, f);
}

// LDS of a workgroup: keys, slots 0 and 1, then values, slots 0 to 2; at the end the parts of KS wavefronts (FB * 16 + 2 floats a lane)
template <int HD, int RB, int KS>
constexpr int kRows32Lds = 5 * 64 * KS * HD * 2 > (KS - 1) * RB * 64 * (HD / 2 + 2) * 4 ? 5 * 64 * KS * HD * 2 : (KS - 1) * RB * 64 * (HD / 2 + 2) * 4;

// What a score gets for the distance between its row and its key, by the query head: table [nq][far + 1], float32, added to the scaled
// score; beyond `far` the last entry counts.  In LDS (behind the tiles) a head's entries lie turned round and divided by the scale, so that
// keys that follow each other find theirs one behind the other, with kBiasFront and kBiasBack copies of the last and the first at the
// ends, which rows and keys of a tile that is partly beyond `far` or the diagonal run into.
struct DistanceBias {
    const float* table;
    int far;
    float* lds;
};
constexpr int kBiasFront = 96, kBiasBack = 64;
__host__ __device__ constexpr int bias_row(int far) { return (kBiasFront + far + 1 + kBiasBack + 1) | 1; }     // (odd: the heads' banks differ)

// Rows are rescaled late, when their maximum has grown by 2^8, where the caller says so and where the keys are dealt out, behind so many
// keys.  Against a row's own maximum the largest probability is one, which bfloat16 has exactly; against an older
// one it is rounded like the others, and the result is further from 64 bits: 2-norm of its error at scores of deviation two, late
// and exact, head size 64, 2,048 / 5,000 tokens 0.00185 and 0.00181 / 0.00195 and 0.00182; 512 tokens behind 1,600 keys 0.00216 and 0.00184 (the
// kernel of 16-row tiles 0.00180).  The large steps gain 2 to 6 % by it (us a layer: 14 heads of 64 on 2, 8,191 tokens 168 and 175; 28 of 128
// on 4, 5,000 tokens 195 and 205) and are nearer to 64 bits so than with every row late from the first key on (0.00199, 0.00205); the others,
// which have kernels with exact maxima to compare with, keep them.
constexpr int kLateFrom = 1536;

// Workgroup `index` of a launch (and range `part` of the keys); a token's queries lie `width` values behind those of the one before.
// WIDE: scores of any finite size.  score x scale - maximum x scale as one multiply-add has the rounding of its last operand in it, the
// same factor for a whole row, which divides out as long as it is a number: 2^64 at 2^30.  Beyond (a bias that stands for a mask) the maximum
// is taken off first.
template <int HD, int RB, int KS, bool SPLIT, bool BIAS = false, bool WIDE = BIAS>
__device__ __forceinline__ void rows32_block(
    char* smem, int index, int part, const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_table, int table_width,
    const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len, const int32_t* __restrict__ kv_len,
    int n_seqs, int nq, int nkv, int page_size, int page_shift, float scale, int window, int skip_single,
    float* __restrict__ part_o, float* __restrict__ part_ml, int n_splits, int n_tokens, int width, int late, DistanceBias bias = {}) {
    constexpr int NQ = HD / 16;                  // steps of 16 features of the score product
    constexpr int FB = HD / 32;                  // blocks of 32 output features
    constexpr int ROWS = 32 * RB;
    constexpr int KT = 64 * KS;                  // keys per LDS tile
    constexpr int GROUP = 16 * HD * 2;           // bytes of 16 keys (or of their values)
    constexpr int SLOT = KT * HD * 2;            // bytes of a tile of keys (or of values)
    constexpr int PER_LANE = FB * 16 + 2;        // floats a lane leaves for the combination
    constexpr int LOADS = HD / 32, N_LOADS = 4 * LOADS / RB;     // loads of a group; of a tile's keys (and values) by a wavefront
    constexpr int OWN = N_LOADS > LOADS ? N_LOADS / LOADS : 1;   // groups that they are of
    static_assert(N_LOADS * RB == 4 * LOADS && (N_LOADS % LOADS == 0 || LOADS % N_LOADS == 0), "a tile is whole loads");
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int rb = wave % RB, ksi = wave / RB;
    const int lr = lane % 32, lh = lane / 32;
    // (the kv heads of a block of rows after each other, so that all heads' last rows, which have the most keys, begin first)
    const int kh = index % nkv;
    const int group_size = nq / nkv;

    int b, grp;
    // (skip_single: requests of one token are the decode kernel's, which spreads their keys over wavefronts)
    auto groups_of = [&](int n) { return (skip_single && n == 1) ? 0 : (n * group_size + ROWS - 1) / ROWS; };
    if (!find_block(q_len, n_seqs, index / nkv, groups_of, b, grp)) return;
    grp = groups_of(q_len[b]) - 1 - grp;     // the last rows first: they have the most keys to walk
    const int n = q_len[b], kv = kv_len[b], qs = q_start[b];
    const int rows = n * group_size;
    const int32_t* table = block_table + static_cast<size_t>(b) * table_width;

    // the workgroup's rows and the keys they need
    const int blk_first = grp * ROWS, blk_last = min(rows, blk_first + ROWS) - 1;
    const int blk_p_hi = kv - n + blk_last / group_size;
    const int blk_first_pos = kv - n + blk_first / group_size;
    const int blk_lo = window > 0 ? max(0, blk_first_pos - window + 1) : 0;
    // n_splits > 1: the tiles of keys are dealt over as many workgroups (`part`), each of which leaves its rows'
    // unnormalised result with its maximum and sum in part_o / part_ml for the kernel that combines them
    // (SPLIT is a parameter of the template so that the kernel without it is compiled as if this were not here; a
    // workgroup takes four tiles at least, three at head size 128, where a tile takes twice as long: fewer are not worth sharing)
    constexpr int kLeastTiles = HD == 128 ? 3 : 4;
    const int t_first = blk_lo / KT, t_last = blk_p_hi / KT + 1;
    const int t_per = SPLIT ? max((t_last - t_first + n_splits - 1) / n_splits, kLeastTiles) : t_last - t_first;
    const int t_begin = SPLIT ? t_first + part * t_per : t_first;
    const int t_end = SPLIT ? min(t_last, t_begin + t_per) : t_last;
    [[maybe_unused]] const size_t part_row0 = SPLIT ? static_cast<size_t>(part) * n_tokens * nq : 0;

    // this wavefront's block of 32 rows, this lane's row
    const int row_base = blk_first + rb * 32;
    const int r = row_base + lr;
    const bool valid = r < rows;
    const int i_tok = valid ? r / group_size : 0;
    const int tok = qs + i_tok;
    const int head = kh * group_size + (valid ? r % group_size : 0);
    const int p_row = valid ? kv - n + i_tok : -1;
    const int lo_row = (window > 0 && valid) ? max(0, p_row - window + 1) : 0;
    const bool wave_any = row_base < rows;
    const int w_last = min(rows, row_base + 32) - 1;
    const int w_p_hi = wave_any ? kv - n + w_last / group_size : -1;       // largest causal limit in the block
    const int w_p_min = wave_any ? kv - n + row_base / group_size : -1;    // smallest
    const int w_lo_first = (window > 0 && wave_any) ? max(0, w_p_min - window + 1) : 0;
    const int w_lo_max = (window > 0 && wave_any) ? max(0, w_p_hi - window + 1) : 0;
    bf16x8 q[NQ];
    {
        const bf16_t* qp = qkv + static_cast<size_t>(tok) * width + head * HD + lh * 8;
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            const uint4 v = valid ? *reinterpret_cast<const uint4*>(qp + j * 16) : uint4{0u, 0u, 0u, 0u};
            q[j] = __builtin_bit_cast(bf16x8, v);
        }
    }
    const float scale2 = scale * 1.4426950408889634f;
    if constexpr (SPLIT) {
        if (t_begin >= t_end) {              // no tile of keys is left for this workgroup
            if (valid && ksi == 0 && lh == 0) {
                float* ml = part_ml + (part_row0 + static_cast<size_t>(tok) * nq + head) * 2;
                ml[0] = -INFINITY;
                ml[1] = 0.f;
            }
            return;
        }
    }

    f32x16 o[FB];
#pragma unroll
    for (int f = 0; f < FB; ++f)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[f][e] = 0.f;
    float m_run = -INFINITY;                  // the maximum in units of the raw scores
    // the rows' sums of probabilities come from the matrix cores: a block of "values" whose first feature is all ones
    // (the lanes lane % 32 == 0 hold it) gives them as feature 0 of one more output block, element 0 of the lanes of
    // half 0 (32 additions per step on the vector pipe against four matrix instructions); in SUMS chains
    constexpr int SUMS = HD == 64 ? 2 : 1;
    f32x16 o_sum[SUMS];
#pragma unroll
    for (int c = 0; c < SUMS; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) o_sum[c][e] = 0.f;
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<__bf16>(lr == 0 ? 1.0f : 0.0f);
    f32x16 zero16;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero16[e] = 0.f;

    // A tile is two steps of a wavefront: the matrix instructions (the scores of tile i, the output of tile i - 1), then the vector
    // instructions (the probabilities of tile i).  The two wavefronts of a SIMD take them in turn: wavefronts 4 to 7 are one
    // step behind, so that one of the two is at its matrix instructions while the other is at its vector instructions, and a
    // barrier behind every step keeps them so.
    // With `late` (or SPLIT), behind long contexts the accumulated output is rescaled only when a row's maximum has grown by more than 2^kSlack since
    // the last time: until then the exponentials are taken against the old maximum, so they may reach 2^kSlack instead of 1, which
    // float32 sums and bfloat16 probabilities (the same relative precision at any magnitude) do not mind.
    // Keys and values go from memory straight to LDS, 16 keys (never more than a page's) to a load's base address and a
    // constant of the lane beside it, so that they cost no vector instructions and no registers.  A wavefront that issues a load waits
    // until the memory pipe takes it, some 100 cycles when all issue theirs at once, so they are spread over both steps: the
    // keys of tile i + 1 go out in the first wavefronts' matrix step of tile i (when everybody has read the keys of tile i - 1) and the
    // values of tile i + 1 in the step behind it, with a third slot so that they have two steps and more to arrive as well.
    constexpr float kSlack = 8.0f;
    constexpr bool TURNS = RB * KS == 8;
    const bool second = TURNS && wave >= 4;
    const int page_mask = page_size - 1;             // page sizes here are powers of two
    // A row of a group of keys lies in LDS as pieces of 16 bytes, exchanged by the row's number (piece p of row r in place
    // p ^ (r / 2 & 7)), a feature of a group of values as two pieces, exchanged by the feature's (p ^ (f / 8 & 1)): lanes that
    // read one piece of many rows then hit different banks.  A load puts a lane's 16 bytes at its base + 16 x lane, so the
    // exchange is made in the addresses that lanes load from.
    constexpr int PIECES = HD / 8;                   // of a key's row
    const int load0 = wave * N_LOADS, group0 = load0 / LOADS;    // this wavefront's first load of a tile, and its group
    int k_off[N_LOADS];
#pragma unroll
    for (int i = 0; i < N_LOADS; ++i) {
        const int row = (load0 + i) % LOADS * (64 / PIECES) + lane / PIECES;
        k_off[i] = row * HD * 2 + (((lane % PIECES) ^ (row / 2 & 7)) * 16);
    }
    const int v_piece = (lane % 2) ^ (lane / 16 & 1);        // (feature lane / 2 of a load's 32)
    const int v_off = (lane / 2) * page_size * 2 + v_piece * 16;
    const int v_step = 32 * page_size * 2;
    const size_t page_bytes = static_cast<size_t>(nkv) * page_size * HD * 2, head_bytes = static_cast<size_t>(page_size) * HD * 2;
    const char* const k_head = reinterpret_cast<const char*>(k_cache) + kh * head_bytes;
    const char* const v_head = reinterpret_cast<const char*>(v_cache) + kh * head_bytes;
    // The page numbers of a wavefront's groups of a tile, by scalar loads (constant address space: no other instruction here writes the
    // block table).  The index into it is clamped to the pages that hold the workgroup's keys, so every load reads memory of this
    // request.
    const int idx_lo = blk_lo >> page_shift, idx_hi = blk_p_hi >> page_shift, idx_step = KT >> page_shift;
    const auto* const table_c = reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(table));
    struct Pages {
        int of[OWN];
    };
    auto lookup = [&](int tile) {
        Pages p;
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            const int idx = tile * idx_step + ((group0 + i) * 16 >> page_shift);
            p.of[i] = table_c[min(max(idx, idx_lo), idx_hi)];
        }
        return p;
    };
    auto load_k = [&](const Pages& pages, int i, int slot) {
        const int g = (load0 + i) / LOADS;
        const unsigned page = max(pages.of[i / LOADS], 0);
        load_to_lds(buffer_of(k_head + page * page_bytes, head_bytes), k_off[i], (g * 16 & page_mask) * (HD * 2), smem + slot * SLOT + (load0 + i) * 1024);
    };
    auto load_v = [&](const Pages& pages, int i, int slot) {
        const int g = (load0 + i) / LOADS, u = (load0 + i) % LOADS;
        const unsigned page = max(pages.of[i / LOADS], 0);
        load_to_lds(buffer_of(v_head + page * page_bytes, head_bytes), v_off, (g * 16 & page_mask) * 2 + u * v_step,
                    smem + (2 + slot) * SLOT + (load0 + i) * 1024);
    };
    // Zeros for the values of this tile that no row of the workgroup sees (their probabilities are zeros, but what lies in the
    // page may be no number): every lane those that it loaded.
    auto trim_v = [&](int slot, int tile) {
        if (tile * KT >= blk_lo && tile * KT + KT - 1 <= blk_p_hi) return;
#pragma unroll 1
        for (int i = 0; i < N_LOADS; ++i) {
            const int key = tile * KT + (load0 + i) / LOADS * 16 + v_piece * 8;
            u32x4* at = reinterpret_cast<u32x4*>(smem + (2 + slot) * SLOT + (load0 + i) * 1024 + lane * 16);
            u32x4 v = *at;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (key + e < blk_lo || key + e > blk_p_hi) v[e / 2] &= e % 2 ? 0x0000ffffu : 0xffff0000u;
            *at = v;
        }
    };
    Pages pages, next_pages;                         // of the tile whose loads go out next, and of the one behind it
    int k_slot = 0, v_slot = 0;                      // of the tile that is multiplied
    auto after = [](int v) { return v == 2 ? 0 : v + 1; };
    // behind a tile's second step: the next tile's keys and this one's values are there (the next one's values need not be)
    auto loads_arrived = [&](int tile) {
        arrived<N_LOADS>();
        trim_v(v_slot, tile);
    };
    // Row lr of a block of 32 keys, as the matrix instruction sees it, is the key whose number has bits 2 and 3 of lr exchanged: a
    // lane's scores are then those of keys 16 b + 8 h + v (v in 0..7), the run of eight whose values it supplies to the
    // second product in the order in which a page holds them.
    const int k_lr = (lr & 0x13) | (lr & 4) << 1 | (lr & 8) >> 1;
    int k_get[4];                                    // (in the slot of the next keys to be read; the slots are exchanged by a bit)
#pragma unroll
    for (int j = 0; j < 4; ++j) k_get[j] = (ksi * 64 + k_lr) * (HD * 2) + (((2 * j + lh) ^ (k_lr / 2 & 7)) * 16);
    const int v_lane = 2 * SLOT + ksi * 4 * GROUP + lr * 32 + ((lh ^ (lr / 8 & 1)) * 16);
    int v_get = v_lane + 2 * SLOT;                   // (the slot of the values of the tile before)
    // The matrix instructions of a step, in order: the rows' sums of tile i - 1, which take nothing from LDS, the scores of tile i,
    // the output of tile i - 1.  (Consecutive ones go to different accumulators: one that adds to the result of the one before it
    // would wait for it.)  Operands are read AHEAD instructions ahead.
    constexpr int N_QK = 2 * NQ, N_PV = 4 * FB, N_LDS = N_QK + N_PV, AHEAD = 6;
    f32x16 acc[2];
    bf16x8 pb[4];
    auto matrix_step = [&](auto&& load) {
        u32x4 operand[AHEAD];
        auto read_operand = [&](auto m_c) {
            constexpr int m = decltype(m_c)::value;
            if constexpr (m < N_QK)
                operand[m % AHEAD] = *reinterpret_cast<const u32x4*>(smem + k_get[m / 2 % 4] + m % 2 * 32 * (HD * 2) + m / 8 * 128);
            else if constexpr (m < N_LDS)
                operand[m % AHEAD] = *reinterpret_cast<const u32x4*>(smem + v_get + (m - N_QK) / FB * GROUP + (m - N_QK) % FB * 1024);
        };
        auto sum = [&](int t) {
            o_sum[t % SUMS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pb[t], o_sum[t % SUMS], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        __builtin_amdgcn_s_setprio(1);
        static_for<AHEAD>(read_operand);
        __builtin_amdgcn_sched_barrier(0);
        sum(0);
        if constexpr (SUMS == 2) sum(1), sum(2), sum(3);
        static_for<N_LDS>([&](auto m_c) {
            constexpr int m = decltype(m_c)::value;
            const bf16x8 from_lds = __builtin_bit_cast(bf16x8, operand[m % AHEAD]);
            if constexpr (m < N_QK)
                acc[m % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(from_lds, q[m / 2], m < 2 ? zero16 : acc[m % 2], 0, 0, 0);
            else
                o[(m - N_QK) % FB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(from_lds, pb[(m - N_QK) / FB], o[(m - N_QK) % FB], 0, 0, 0);
            read_operand(std::integral_constant<int, m + AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (SUMS == 1 && m < N_QK && m % 4 == 3 && m / 4 < 3) sum(m / 4 + 1);
            if constexpr (m % (N_LDS / N_LOADS) == 1) {
                load(m / (N_LDS / N_LOADS));
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) k_get[j] ^= SLOT;
        v_get = v_lane + v_slot * SLOT;
    };
    // (Against the row's own maximum the largest probability is one, which bfloat16 has exactly; against an older one it is rounded like
    // the others, at any context: see kLateFrom.)
    const float slack = (SPLIT || late) && blk_p_hi >= kLateFrom ? kSlack / scale2 : 0.f;
    [[maybe_unused]] bool beyond_shift = false;      // WIDE: a row of the wavefront has such a maximum
    float limit = -INFINITY, shift = 0.0f;           // a row's maximum beyond which there is rescaling; what the exponents are shifted by
    const float* const bias_of_row = BIAS ? bias.lds + (valid ? r % group_size : 0) * bias_row(bias.far) + kBiasFront : nullptr;
    auto vector_step = [&](int tile, auto&& load) {
        const int key0 = tile * KT + ksi * 64;
        float beyond = 0.f;                          // what all of a tile's scores get that is `far` or more behind every row
        if constexpr (BIAS) {
            if (w_p_min - (key0 + 63) >= bias.far) {
                beyond = bias_of_row[0];
            } else {
                const float* from = bias_of_row + min(max(bias.far - p_row + key0, -kBiasFront), bias.far + 1) + lh * 8;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[kb][e] += from[kb * 32 + (e / 8) * 16 + e % 8];
            }
        }
        // the diagonal, a window's edge, or nothing at all (a wavefront without rows has nothing to mask: nobody reads its results)
        const int upto = p_row - key0 - lh * 8, from = lo_row - key0 - lh * 8;
        if (wave_any && key0 + 63 > w_p_min) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (kb * 32 + (e / 8) * 16 + e % 8 > upto) acc[kb][e] = -INFINITY;
        }
        if (wave_any && key0 < w_lo_max) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (kb * 32 + (e / 8) * 16 + e % 8 < from) acc[kb][e] = -INFINITY;
        }
        float mx = -INFINITY, mx1 = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
            // (as one piece: between two of them the compiler puts a pause)
            asm("v_max3_f32 %0, %0, %2, %3\n\tv_max3_f32 %1, %1, %6, %7\n\tv_max3_f32 %0, %0, %4, %5\n\tv_max3_f32 %1, %1, %8, %9"
                : "+&v"(mx), "+&v"(mx1)
                : "v"(acc[0][e]), "v"(acc[0][e + 1]), "v"(acc[0][e + 2]), "v"(acc[0][e + 3]), "v"(acc[1][e]), "v"(acc[1][e + 1]),
                  "v"(acc[1][e + 2]), "v"(acc[1][e + 3]));
        }
        mx = max3(mx, mx, mx1);
        const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = max3(__uint_as_float(halves[0]), __uint_as_float(halves[0]), __uint_as_float(halves[1]));
        if constexpr (BIAS) mx += beyond;
        if (__any(mx > limit)) {                     // (-inf is no more than -inf: the first key a row sees counts)
            const float m_new = fmaxf(m_run, mx), m_use = m_new == -INFINITY ? 0.f : m_new;
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * scale2);
            m_run = m_new;
            limit = m_new + slack;
            shift = -m_use * scale2;
            if constexpr (WIDE) beyond_shift = __any(!(fabsf(shift) < 0x1p30f));
#pragma unroll
            for (int c = 0; c < SUMS; ++c) o_sum[c][0] *= alpha;
#pragma unroll
            for (int f = 0; f < FB; ++f)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[f][e] *= alpha;
        }
        float moved = BIAS ? fmaf(beyond, scale2, shift) : shift;
        if constexpr (WIDE) {
            if (beyond_shift) {
                const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[kb][e] = acc[kb][e] + beyond - m_use;
                moved = 0.f;
            }
        }
        // the second product's steps of 16 keys: step t takes elements 8 (t % 2) .. + 7 of block t / 2 from a lane
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int i = (t * N_LOADS + 3) / 4; i < ((t + 1) * N_LOADS + 3) / 4; ++i) {
                load(i);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
                pb[t][e] = static_cast<__bf16>(__builtin_amdgcn_exp2f(fmaf(acc[t / 2][(t % 2) * 8 + e], scale2, moved)));
        }
        // (they are used in the next step: this keeps their computation in this one)
#pragma unroll
        for (int t = 0; t < 4; ++t) asm volatile("" : "+v"(pb[t]));
        __builtin_amdgcn_sched_barrier(0);
    };

#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) pb[t][e] = static_cast<__bf16>(0.0f);
    pages = lookup(t_begin);
#pragma unroll
    for (int i = 0; i < N_LOADS; ++i) load_k(pages, i, 0);
    if constexpr (BIAS) {
        const int row = bias_row(bias.far);
        for (int idx = threadIdx.x; idx < group_size * row; idx += 64 * RB * KS)
        {
            const float of = bias.table[static_cast<size_t>(kh * group_size + idx / row) * (bias.far + 1) +
                                        min(max(bias.far - (idx % row - kBiasFront), 0), bias.far)];
            // (a finite entry stays finite: a row all of whose keys have the lowest number sees them all alike)
            bias.lds[idx] = __builtin_isfinite(of) ? fminf(fmaxf(of / scale, -3.402823466e38f), 3.402823466e38f) : of;
        }
    }
#pragma unroll
    for (int i = 0; i < N_LOADS; ++i) load_v(pages, i, 0);
    pages = lookup(t_begin + 1);
    next_pages = lookup(t_begin + 2);
    // (the first step multiplies this slot of values by probabilities of zero)
#pragma unroll
    for (int i = 0; i < N_LOADS; ++i) *reinterpret_cast<u32x4*>(smem + 4 * SLOT + (wave * N_LOADS + i) * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
    arrived<0>();                                    // (and the queries: nothing else makes the compiler wait for loads in the loop)
    __syncthreads();
    auto keys_of_next = [&](int i) { load_k(pages, i, k_slot ^ 1); };
    auto values_of_next = [&](int i) { load_v(pages, i, after(v_slot)); };
    if (second) {
#pragma unroll
        for (int i = 0; i < N_LOADS; ++i) keys_of_next(i);
        __syncthreads();
#pragma unroll 1
        for (int tile = t_begin; tile < t_end; ++tile) {
            matrix_step(values_of_next);
            loads_arrived(tile);
            __syncthreads();
            k_slot ^= 1;
            v_slot = after(v_slot);
            pages = next_pages;
            next_pages = lookup(tile + 3);
            vector_step(tile, keys_of_next);
            __syncthreads();
        }
    } else {
#pragma unroll 1
        for (int tile = t_begin; tile < t_end; ++tile) {
            matrix_step(keys_of_next);
            __syncthreads();
            vector_step(tile, values_of_next);
            loads_arrived(tile);
            k_slot ^= 1;
            v_slot = after(v_slot);
            pages = next_pages;
            next_pages = lookup(tile + 3);
            __syncthreads();
        }
        if (TURNS) __syncthreads();                  // (as many barriers as the others)
    }
    arrived<0>();                                    // (behind the last tile there were loads that nobody reads)
    // the output product of the last tile
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        o_sum[t % SUMS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pb[t], o_sum[t % SUMS], 0, 0, 0);
#pragma unroll
        for (int f = 0; f < FB; ++f)
            o[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(smem + v_get + t * GROUP + f * 1024)), pb[t], o[f], 0, 0, 0);
    }
    if constexpr (KS > 1) __syncthreads();           // the combination below writes over the tiles
    if constexpr (SUMS == 2) o_sum[0][0] += o_sum[1][0];
    // the row's sum: feature 0 of the block of ones, which lane lr of half 0 holds
    float l = __shfl(o_sum[0][0], lr, kWave);
    [[maybe_unused]] float m_part = m_run;           // the maximum that o and l are in units of
    if constexpr (KS > 1) {
        // The wavefronts of one block of rows hold partial results over their keys: those with ks > 0 leave
        // theirs in LDS (the tiles are no longer read: the loop ended with a barrier), ks == 0 adds them up.
        float* comb = reinterpret_cast<float*>(smem);
        if (ksi > 0) {
            float* dst = comb + (static_cast<size_t>((ksi - 1) * RB + rb) * PER_LANE) * 64 + lane;
#pragma unroll
            for (int f = 0; f < FB; ++f)
#pragma unroll
                for (int e = 0; e < 16; ++e) dst[(f * 16 + e) * 64] = o[f][e];
            dst[(FB * 16) * 64] = m_run;
            dst[(FB * 16 + 1) * 64] = l;
        }
        __syncthreads();
        if (ksi > 0) return;
        float m_all = m_run;
#pragma unroll
        for (int j = 0; j < KS - 1; ++j)
            m_all = fmaxf(m_all, comb[(static_cast<size_t>(j * RB + rb) * PER_LANE + FB * 16) * 64 + lane]);
        if constexpr (SPLIT) m_part = m_all;
        const float m_ref = m_all == -INFINITY ? 0.f : m_all;
        const float w0 = __builtin_amdgcn_exp2f((m_run - m_ref) * scale2);
        // Of the two products of the first sum one is rounded by itself.  Which one isn't a matter of accuracy, but it has to be said: left to
        // the compiler it changed with the way in which the results are packed below, and by it the logits of a model of 28 layers by 0.3 %.
        // (five elements have it the other way round, where that change found them)
        auto other_first = [](int f, int e) { return !SPLIT && f == 0 && e >= 1 && e <= 5; };
#pragma unroll
        for (int j = 0; j < KS - 1; ++j) {
            const float* src = comb + (static_cast<size_t>(j * RB + rb) * PER_LANE) * 64 + lane;
            const float wj = __builtin_amdgcn_exp2f((src[(FB * 16) * 64] - m_ref) * scale2), lj = src[(FB * 16 + 1) * 64];
            l = j == 0 ? fmaf(l, w0, lj * wj) : fmaf(lj, wj, l);
#pragma unroll
            for (int f = 0; f < FB; ++f)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float x = src[(f * 16 + e) * 64];
                    if (j > 0) o[f][e] = fmaf(x, wj, o[f][e]);
                    else if (other_first(f, e)) o[f][e] = fmaf(x, wj, o[f][e] * w0);
                    else o[f][e] = fmaf(o[f][e], w0, x * wj);
                }
        }
    }
    if constexpr (SPLIT) {
        // (element e of block f is feature f * 32 + (e / 4) * 8 + lh * 4 + e % 4: runs of four features; the maximum
        // goes out in units of the exponent's argument, as the combining kernel takes it; -inf: no key seen)
        if (valid) {
            const size_t prow = part_row0 + static_cast<size_t>(tok) * nq + head;
            float* po = part_o + prow * HD + lh * 4;
#pragma unroll
            for (int f = 0; f < FB; ++f)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float4*>(po + f * 32 + g * 8) =
                        float4{o[f][g * 4], o[f][g * 4 + 1], o[f][g * 4 + 2], o[f][g * 4 + 3]};
            if (lh == 0) {
                part_ml[prow * 2] = m_part * scale;
                part_ml[prow * 2 + 1] = l;
            }
        }
        return;
    }
    if (valid) {
        // element e of block f is feature f * 32 + (e / 4) * 8 + lh * 4 + e % 4: runs of four features
        const float inv = 1.0f / l;
        bf16_t* op = out + (static_cast<size_t>(tok) * nq + head) * HD + lh * 4;
#pragma unroll
        for (int f = 0; f < FB; ++f)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                uint2 packed;
                packed.x = bf16_pair(o[f][g * 4] * inv, o[f][g * 4 + 1] * inv);
                packed.y = bf16_pair(o[f][g * 4 + 2] * inv, o[f][g * 4 + 3] * inv);
                *reinterpret_cast<uint2*>(op + f * 32 + g * 8) = packed;
            }
    }
}

template <int HD, int RB, int KS, bool SPLIT>
__global__ __launch_bounds__(64 * RB * KS) void attention_rows32_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_table, int table_width,
    const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len, const int32_t* __restrict__ kv_len,
    int n_seqs, int nq, int nkv, int page_size, int page_shift, float scale, int window, int skip_single,
    float* __restrict__ part_o, float* __restrict__ part_ml, int n_splits, int n_tokens, int late) {
    __shared__ __attribute__((aligned(128))) char smem[kRows32Lds<HD, RB, KS>];
    rows32_block<HD, RB, KS, SPLIT>(smem, blockIdx.x, blockIdx.z, qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len,
                                    n_seqs, nq, nkv, page_size, page_shift, scale, window, skip_single, part_o, part_ml, n_splits, n_tokens,
                                    (nq + 2 * nkv) * HD, late);
}

// The same for queries that lie by themselves, [tokens][nq][HD], with a bias by distance or without one.
template <int HD, int RB, int KS, bool BIAS>
__global__ __launch_bounds__(64 * RB * KS) void attention_heads32_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len,
    const int32_t* __restrict__ kv_len, int n_seqs, int nq, int nkv, int page_size, int page_shift, float scale, int window,
    const float* __restrict__ table, int far) {
    extern __shared__ __attribute__((aligned(128))) char heads_lds[];
    const DistanceBias bias{table, far, reinterpret_cast<float*>(heads_lds + kRows32Lds<HD, RB, KS>)};
    rows32_block<HD, RB, KS, false, BIAS, true>(heads_lds, blockIdx.x, 0, q, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs,
                                          nq, nkv, page_size, page_shift, scale, window, 0, nullptr, nullptr, 1, 0, nq * HD, 0, bias);
}

// Deals the keys of a step's decoded tokens out over `slots` workgroups (per kv head): a request's blocks of 32 keys go to as few
// of them as leave none with more than `per` blocks, `per` being the least for which they all suffice (kLeastPer at least).  One
// launch a step, for all layers.  With the same number of key ranges for every request the longest one sets a layer's
// time: 12 heads of 128 on 2, 40 requests of 128 to 2,048 tokens, a layer 23.5 us -> 18.2; 14 heads of 64 on 2, one request of 8,000
// tokens beside 31 of 500 21.8 -> 15.0.  This kernel takes 4 to 5 us, once a step.
// table [slots][kRangeInts]: request (-1: none), first block, end, tokens in the cache, the token's row, number of parts;
// then [n_seqs][2]: a request's first slot, its number of parts.  n_seqs <= slots <= 256; q_len null: all of one token.
constexpr int kRangeInts = 8, kRangeSlots = 256, kLeastPer = 8, kMostParts = 64;
__global__ __launch_bounds__(kRangeSlots) void decode_ranges_kernel(const int32_t* __restrict__ kv_len, const int32_t* __restrict__ q_start,
                                                                    const int32_t* __restrict__ q_len, int n_seqs, int slots, int window,
                                                                    int32_t* __restrict__ table) {
    __shared__ int s_part[4];
    const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
    auto block_total = [&](int v) {
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
        __syncthreads();
        if (lane == 0) s_part[wave] = v;
        __syncthreads();
        return s_part[0] + s_part[1] + s_part[2] + s_part[3];
    };
    const bool here = t < n_seqs && (q_len == nullptr || q_len[t] == 1);
    const int kv = here ? kv_len[t] : 0, p = kv - 1;
    const int begin = (window > 0 ? max(0, p - window + 1) : 0) / 32, end = here ? p / 32 + 1 : begin;
    const int blocks = max(end - begin, here ? 1 : 0);
    int most = blocks;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, kWave));
    if (lane == 0) s_part[wave] = most;
    __syncthreads();
    most = max(max(s_part[0], s_part[1]), max(s_part[2], s_part[3]));
    __syncthreads();
    int low = max(kLeastPer, (most + kMostParts - 1) / kMostParts), high = max(low, most);
    while (low < high) {
        const int per = (low + high) / 2;
        if (block_total((blocks + per - 1) / per) <= slots) high = per;
        else low = per + 1;
    }
    const int parts = (blocks + low - 1) / low;
    int incl = parts;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int up = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += up;
    }
    __syncthreads();
    if (lane == kWave - 1) s_part[wave] = incl;
    __syncthreads();
    int first = incl - parts, total = 0;
    for (int w = 0; w < 4; ++w) {
        first += w < wave ? s_part[w] : 0;
        total += s_part[w];
    }
    if (t < n_seqs) {
        table[slots * kRangeInts + 2 * t] = first;
        table[slots * kRangeInts + 2 * t + 1] = parts;
    }
    const int per = parts > 0 ? (blocks + parts - 1) / parts : 0;
    for (int i = 0; i < parts; ++i) {
        int32_t* e = table + (first + i) * kRangeInts;
        e[0] = t;
        e[1] = min(end, begin + i * per);
        e[2] = min(end, begin + (i + 1) * per);
        e[3] = kv;
        e[4] = q_start[t];
        e[5] = parts;
    }
    if (t >= total && t < slots) table[t * kRangeInts] = -1;
}

// What the fused variant of the decode kernel computes its queries (and the new token's key and value) from:
// the QKV product as it comes out of the skinny product kernel, before bias, rotation and rounding.
struct FusedQkv {
    const float* prod;        // [in_splits][n_tokens][(nq + 2 nkv) * hd] float32 partial sums
    int in_splits;
    const float* row_ss;      // [ss_splits][n_tokens] sums of squares of the rows (1/rms still to apply), or null
    int ss_splits;
    float inv_hidden, eps;
    const bf16_t* bias;       // [(nq + 2 nkv) * hd] or null
    const float* cos_sin;     // [n_tokens][hd / 2][2]: (cos, sin) of the tokens' rotation angles (egpt_rope_table)
    const int32_t* slots;     // [n_tokens] page * page_size + offset of the token's key and value
    bf16_t* k_cache_w;        // the caches again, writable
    bf16_t* v_cache_w;
};

// Decoded tokens only (one query token per request, its heads of one kv group in one 16-row tile): a
// workgroup of NW wavefronts shares one (request, kv head, key split); each wavefront walks its share of
// the keys, PF blocks of 32 keys per round with all of the round's loads in flight together (the kernel is
// a chain of round trips to memory, not of arithmetic), and the wavefronts' results are combined through
// LDS.  With n_splits > 1 the combined, still unnormalised result goes to part_o / part_ml.
//
// FUSED: the kernel also does what the QKV epilogue kernel does for these tokens, which takes that kernel
// out of the chain of a decode step.  Every workgroup adds up the product's partial sums for its query
// heads, applies the rows' 1/rms, bias and rotation (same operations in the same order as
// qkv_rope_store_kernel, so the same bits) and keeps the queries in LDS.  The workgroup whose key range ends
// with the new token does the same for that token's key and value, writes them to the cache and, because
// its own loads of that cache line may have been issued before, puts them into its operands itself.
//
// RANGED: the keys are dealt out by `decode_ranges_kernel`, every request getting as many workgroups as its context is long;
// grid (slots, kv heads), and a part is kept by its slot.

// What a workgroup reads that is no address: sizes, and what stands for divisions by them.
struct DecodeSizes {
    int table_width, page_size, nkv, n_splits;
    unsigned page_magic, split_magic, wave_magic;                // magic_of(page_size / 16), (n_splits), (n_waves)
    int group, window, n_tokens;                                 // group: query heads of a kv head
    float scale;
    int n_waves;                                                 // of a workgroup (blockDim would be a load by itself)
};

// The order of the loads is what this kernel's time is: everything that depends on no other load goes out at once (the
// context's length, the product's partial sums with what is computed from them), then the page numbers, then the first round of keys
// and values, and only then are the queries made.  Loads are bounded by their buffer's size instead of branches, so that none of
// them ends a batch: a page that is not there is a buffer of no bytes, which reads as zeros; a partial sum past the last one adds
// zero.  (Written with conditions around the loads, the compiler moved the queries' arithmetic in front of the keys' loads and waited
// five times one after the other.)  Instructions count as much: a kernel begins with an empty instruction cache, a jump over code that is
// not needed is a trip for the next line, and 300 instructions take 1 us.  So there are no divisions, code for rare sizes lies behind the
// common path, and a round's keys share one maximum.  14 heads of 64 on 2 behind 2,048 tokens: a step of 24 layers for one request 732 ->
// 693 us, for eight 806 -> 768; by the kernel trace 8.8 -> 7.8 us a layer for one (the fastest 7.0 -> 6.2), of which by timestamps inside the
// loads' issue is 1.5, the trip to the keys 1.2, their products and softmax 1, the wavefronts' combination 0.6.
//
// WIDE: operands that 32 bits of place or loads of two values don't reach (partial sums of 2 GB and more, biases that begin between two of
// 4 bytes, pages of a head's gigabytes): plain loads behind conditions.
template <int HD, int PF, bool FUSED, bool MIXED, bool RANGED, int INF, bool WIDE>
__device__ __forceinline__ void decode_block(
    float* wave_state, int bx, int by, int bz, const int32_t* __restrict__ lengths, const int32_t* __restrict__ block_table,
    const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache, const DecodeSizes& d, const bf16_t* __restrict__ qkv,
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ q_len, const FusedQkv& f) {
    constexpr int KD = HD / 32, DT = HD / 16;
    constexpr int kRow = HD + 2;
    // MIXED: a step that also holds portions of prompts; this kernel takes its requests of one token, parts are kept
    // by request (n_tokens is the number of requests then) and the rest is another kernel's.  (A parameter of the
    // template, so that the kernel of the decode step is compiled as if this were not here.)
    if constexpr (MIXED && !RANGED) {
        if (q_len[bx] != 1) return;
    }
    const int32_t* range = RANGED ? lengths + bx * kRangeInts : nullptr;
    const int b = RANGED ? range[0] : bx, kh = by;
    if constexpr (RANGED) {
        if (b < 0) return;
    }
    // wave_state: [n_waves][16][HD + 2]: O, then maximum, then sum
    const int lane = threadIdx.x % kWave, n_waves = d.n_waves, n_threads = n_waves * kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // known to be the same for the wavefront
    const int lj = lane % 16, lg = lane / 16;
    const int group_size = d.group, nkv = d.nkv, nq = group_size * nkv, page_size = d.page_size;
    const int kv = RANGED ? range[3] : lengths[b];
    __builtin_amdgcn_sched_barrier(0);                // (asked for before anything else)
    const int tok = RANGED ? range[4] : FUSED ? b : q_start[b];
    const int n_splits = RANGED ? range[5] : d.n_splits;
    const int width = (nq + 2 * nkv) * HD;
    const int32_t* table = block_table + static_cast<size_t>(b) * d.table_width;
    // (all arguments that did not come with the wavefront, and the length, in one trip)
    if constexpr (FUSED)
        asm volatile("" ::"s"(f.prod), "s"(f.in_splits), "s"(f.row_ss), "s"(f.ss_splits), "s"(f.bias), "s"(f.cos_sin), "s"(f.slots), "s"(group_size),
                     "s"(d.window), "s"(d.n_tokens), "s"(n_waves), "s"(kv));
    bf16_t* q_lds = reinterpret_cast<bf16_t*>(wave_state + n_waves * 16 * kRow);   // FUSED: [16][HD], then k, v [HD]
    bf16_t* k_lds = q_lds + 16 * HD;
    bf16_t* v_lds = k_lds + HD;

    // ---- FUSED: what the queries, and the new token's key and value, are made of.  An item is two neighbouring pairs
    // (i, i + half), (i + 1, i + 1 + half) of a head; heads past the queries are the key and the value.
    constexpr int half = HD / 2, kItems = half / 2;
    struct Item {
        u32x2 ta[INF], tb[INF];
        uint32_t ba, bb;                         // bias
        u32x4 turn;                              // cos, sin of both pairs
    };
    auto item_col = [&](unsigned it) {
        const int h = it / kItems, i = it % kItems * 2, past = h - group_size;
        const int query = kh * group_size + h, other = nq + kh + past * nkv;
        return (past < 0 ? query : other) * HD + i;
    };
    using place_t = std::conditional_t<WIDE, size_t, int>;
    const place_t stride = static_cast<place_t>(d.n_tokens) * width;      // values of a partial sum
    const buffer_t prod_buf = values_of(f.prod + static_cast<size_t>(tok) * width, WIDE ? 0 : ((f.in_splits - 1) * stride + width) * 4);
    const buffer_t bias_buf = values_of(f.bias, f.bias ? width * 2 : 0);
    const buffer_t turn_buf = values_of(f.cos_sin + static_cast<size_t>(tok) * HD, HD * 4);
    auto parts_load = [&](int col, int j0, u32x2 (&ta)[INF], u32x2 (&tb)[INF]) {
#pragma unroll
        for (int j = 0; j < INF; ++j) {
            if constexpr (WIDE) {
                const float* src = f.prod + static_cast<size_t>(tok) * width + min(j0 + j, f.in_splits - 1) * stride + col;
                const bool there = j0 + j < f.in_splits;
                ta[j] = u32x2{there ? __float_as_uint(src[0]) : 0u, there ? __float_as_uint(src[1]) : 0u};
                tb[j] = u32x2{there ? __float_as_uint(src[half]) : 0u, there ? __float_as_uint(src[half + 1]) : 0u};
                continue;
            }
            const int at = (j0 + j) * stride * 4 + col * 4;              // (behind the last sum: past the buffer's end)
            ta[j] = read8(prod_buf, at);
            tb[j] = read8(prod_buf, at + half * 4);
        }
    };
    auto item_load = [&](unsigned it, Item& r) {
        const int col = item_col(it);
        parts_load(col, 0, r.ta, r.tb);
        if constexpr (WIDE) {
            r.ba = read2(bias_buf, col * 2) | read2(bias_buf, col * 2 + 2) << 16;
            r.bb = read2(bias_buf, col * 2 + half * 2) | read2(bias_buf, col * 2 + half * 2 + 2) << 16;
        } else {
            r.ba = read4(bias_buf, col * 2);
            r.bb = read4(bias_buf, col * 2 + half * 2);
        }
        r.turn = read16(turn_buf, it % kItems * 16);
    };
    [[maybe_unused]] Item first;
    [[maybe_unused]] uint32_t ss_lane = 0;
    [[maybe_unused]] uint32_t slot = 0;
    if constexpr (FUSED) {
        // lane s has the sum of squares of split s
        ss_lane = read4(values_of(f.row_ss, f.row_ss ? f.ss_splits * d.n_tokens * 4 : 0), lane < f.ss_splits ? (lane * d.n_tokens + tok) * 4 : kNowhere);
        // (a wavefront without items goes on: a CU's loads go out one after the other.  The key's and the value's items, which only the
        // last range has, are loaded by every range)
        if (wave * kWave < (group_size + 2) * kItems) item_load(min(static_cast<int>(threadIdx.x), (group_size + 2) * kItems - 1), first);
        int here = tok * 4;
        asm volatile("" : "+v"(here));           // (a lane's value: as the wavefront's it would be waited for at once)
        slot = read4(values_of(f.slots, d.n_tokens * 4), here);
    }
    bf16x8 q[KD];
    const bool valid = lj < group_size;
    if constexpr (!FUSED) {
        const bf16_t* qp = qkv + static_cast<size_t>(tok) * width + (kh * group_size + (valid ? lj : 0)) * HD + lg * 8;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) q[kd] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + kd * 32));
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- the keys of this wavefront
    const int p = kv - 1;
    const int lo = d.window > 0 ? max(0, p - d.window + 1) : 0;
    const int kb_begin = lo >> 5, kb_end = (max(p, 0) >> 5) + 1;
    const int per_split = RANGED ? 0 : divided(kb_end - kb_begin + n_splits - 1, n_splits, d.split_magic);
    const int s_begin = RANGED ? range[1] : kb_begin + bz * per_split, s_end = RANGED ? range[2] : min(kb_end, s_begin + per_split);
    const int per_wave = divided(max(s_end - s_begin, 0) + n_waves - 1, n_waves, d.wave_magic);
    const int w_begin = s_begin + wave * per_wave, w_end = min(s_end, w_begin + per_wave);
    // FUSED: does this workgroup's key range end with the new token?
    const bool writer = FUSED && (RANGED ? s_end == kb_end : s_begin < kb_end && s_begin + per_split >= kb_end);

    // One round of loads: PF blocks of 32 keys and their values for this wavefront, first all page numbers
    // (one wait for all of them), then all key and value loads.
    uint4 kk[PF][2][KD];
    uint2 vv[PF][2][DT];
    const unsigned head_bytes = page_size * (HD * 2), page_bytes = head_bytes * nkv;
    const char* k_head = reinterpret_cast<const char*>(k_cache) + static_cast<size_t>(kh) * head_bytes;
    const char* v_head = reinterpret_cast<const char*>(v_cache) + static_cast<size_t>(kh) * head_bytes;
    const int k_at = lj * (HD * 2) + lg * 16;
    int v_at[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_at[dt] = (dt * 16 + lj) * page_size * 2 + lg * 8;
    auto load_round = [&](int kb0) {
        int pages[PF][2], offs[PF][2];
#pragma unroll
        for (int i = 0; i < PF; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const int key0 = (kb0 + i) * 32 + kt * 16;
                const bool live = kb0 + i < w_end && key0 <= p && key0 + 15 >= lo;
                const int at = divided(key0 >> 4, page_size >> 4, d.page_magic);
                offs[i][kt] = live ? key0 - at * page_size : -1;
                pages[i][kt] = table[live ? at : 0];
            }
        // (all of them asked for before one is waited for)
        if constexpr (PF == 1) asm volatile("" : "+s"(pages[0][0]), "+s"(pages[0][1]));
        if constexpr (PF >= 2) asm volatile("" : "+s"(pages[0][0]), "+s"(pages[0][1]), "+s"(pages[1][0]), "+s"(pages[1][1]));
        if constexpr (PF == 4) asm volatile("" : "+s"(pages[2][0]), "+s"(pages[2][1]), "+s"(pages[3][0]), "+s"(pages[3][1]));
#pragma unroll
        for (int i = 0; i < PF; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const bool ok = offs[i][kt] >= 0 && pages[i][kt] >= 0;
                if constexpr (WIDE) {
                    const size_t row = (static_cast<size_t>(ok ? pages[i][kt] : 0) * nkv + kh) * page_size, o = ok ? offs[i][kt] : 0;
                    const bf16_t* kp = k_cache + (row + o + lj) * HD + lg * 8;
                    const bf16_t* vp = v_cache + row * HD + static_cast<size_t>(lj) * page_size + o + lg * 4;
#pragma unroll
                    for (int kd = 0; kd < KD; ++kd) kk[i][kt][kd] = ok ? *reinterpret_cast<const uint4*>(kp + kd * 32) : uint4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
                        vv[i][kt][dt] = ok ? *reinterpret_cast<const uint2*>(vp + static_cast<size_t>(dt * 16) * page_size) : uint2{0u, 0u};
                    continue;
                }
                const unsigned off = ok ? offs[i][kt] : 0;
                const size_t at = static_cast<size_t>(static_cast<unsigned>(ok ? pages[i][kt] : 0)) * page_bytes;
                const buffer_t kr = values_of(k_head + at + off * (HD * 2), ok ? 16 * HD * 2 : 0);
                const buffer_t vr = values_of(v_head + at + off * 2, ok ? static_cast<size_t>(head_bytes - off * 2) : 0);
#pragma unroll
                for (int kd = 0; kd < KD; ++kd) kk[i][kt][kd] = __builtin_bit_cast(uint4, read16(kr, k_at + kd * 64));
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) vv[i][kt][dt] = __builtin_bit_cast(uint2, read8(vr, v_at[dt]));
            }
    };
    load_round(w_begin);
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (FUSED) {
        float row_scale = 1.f;
        if (f.row_ss) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += __uint_as_float(__builtin_amdgcn_readlane(ss_lane, i));
            if (__builtin_expect(f.ss_splits > 8, 0)) {
                for (int s0 = 8; s0 < min(f.ss_splits, kWave); s0 += 8)
#pragma unroll
                    for (int i = 0; i < 8; ++i) ss += __uint_as_float(__builtin_amdgcn_readlane(ss_lane, s0 + i));
                for (int s0 = kWave; s0 < f.ss_splits; ++s0) ss += f.row_ss[s0 * d.n_tokens + tok];
            }
            row_scale = inv_rms(ss, f.inv_hidden, f.eps);
        }
        auto item_finish = [&](unsigned it, const Item& r) {
            const int h = it / kItems, i = it % kItems * 2;
            float x0[2] = {0.f, 0.f}, x1[2] = {0.f, 0.f};
#pragma unroll
            for (int j = 0; j < INF; ++j)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    x0[e] += __uint_as_float(r.ta[j][e]);
                    x1[e] += __uint_as_float(r.tb[j][e]);
                }
            // more partial sums than one batch of loads: a batch is one trip to memory, not a trip each
            for (int j0 = INF; __builtin_expect(j0 < f.in_splits, 0); j0 += INF) {
                u32x2 ta[INF], tb[INF];
                parts_load(item_col(it), j0, ta, tb);
#pragma unroll
                for (int j = 0; j < INF; ++j)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        x0[e] += __uint_as_float(ta[j][e]);
                        x1[e] += __uint_as_float(tb[j][e]);
                    }
            }
            const uint32_t b0[2] = {r.ba << 16, r.ba & 0xffff0000u}, b1[2] = {r.bb << 16, r.bb & 0xffff0000u};
            bf16_t y0[2], y1[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                x0[e] = scale_then_bias(x0[e], row_scale, __uint_as_float(b0[e]));
                x1[e] = scale_then_bias(x1[e], row_scale, __uint_as_float(b1[e]));
                float r0, r1;                    // queries and the key are rotated, the value is not
                rotate_pair(x0[e], x1[e], __uint_as_float(r.turn[2 * e]), __uint_as_float(r.turn[2 * e + 1]), r0, r1);
                x0[e] = h <= group_size ? r0 : x0[e];
                x1[e] = h <= group_size ? r1 : x1[e];
                y0[e] = from_float<bf16_t>(x0[e]);
                y1[e] = from_float<bf16_t>(x1[e]);
            }
            bf16_t* to = q_lds + (h < group_size ? h : 16 + h - group_size) * HD;      // (the key and the value lie behind 16 queries)
            *reinterpret_cast<uint32_t*>(to + i) = y0[0].bits | static_cast<uint32_t>(y0[1].bits) << 16;
            *reinterpret_cast<uint32_t*>(to + i + half) = y1[0].bits | static_cast<uint32_t>(y1[1].bits) << 16;
            if (__builtin_expect(h < group_size, 1)) return;
            const uint32_t page = slot / static_cast<uint32_t>(page_size), off = slot - page * page_size;
            if (h == group_size) {               // keys: [page][kv head][offset][feature]
                bf16_t* dst = f.k_cache_w + ((static_cast<size_t>(page) * nkv + kh) * page_size + off) * HD + i;
                dst[0] = y0[0];
                dst[1] = y0[1];
                dst[half] = y1[0];
                dst[half + 1] = y1[1];
            } else {                             // values: [page][kv head][feature][offset]
                bf16_t* dst = f.v_cache_w + ((static_cast<size_t>(page) * nkv + kh) * HD + i) * page_size + off;
                dst[0] = y0[0];
                dst[page_size] = y0[1];
                dst[half * static_cast<size_t>(page_size)] = y1[0];
                dst[(half + 1) * static_cast<size_t>(page_size)] = y1[1];
            }
        };
        const int n_items = (group_size + (writer ? 2 : 0)) * kItems;
        if (static_cast<int>(threadIdx.x) < n_items) item_finish(threadIdx.x, first);
        for (int it = threadIdx.x + n_threads; __builtin_expect(it < n_items, 0); it += n_threads) {
            Item r;
            item_load(it, r);
            item_finish(it, r);
        }
        __syncthreads();
        // (a row past the last head holds anything: it is a column of the products that nobody reads)
#pragma unroll
        for (int kd = 0; kd < KD; ++kd)
            q[kd] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(q_lds + lj * HD + kd * 32 + lg * 8));
    }

    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (int kb0 = w_begin; kb0 < w_end; kb0 += PF) {
        if (kb0 > w_begin) load_round(kb0);
        if constexpr (FUSED) {
            // the new token's key and value come from LDS, not from the cache line that was just written
            if (writer && kb0 <= kb_end - 1 && kb_end - 1 < min(w_end, kb0 + PF)) {
                const int i_new = kb_end - 1 - kb0;
#pragma unroll
                for (int i = 0; i < PF; ++i) {
                    if (i != i_new) continue;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        const int key0 = (kb0 + i) * 32 + kt * 16;
                        if (key0 > p || key0 + 15 < p) continue;
                        if (key0 + lj == p) {
#pragma unroll
                            for (int kd = 0; kd < KD; ++kd)
                                kk[i][kt][kd] = *reinterpret_cast<const uint4*>(k_lds + kd * 32 + lg * 8);
                        }
                        const int e = p - (key0 + lg * 4);          // which of this lane's four keys, if any
                        // what is kept of the lane's two words, and where the new value goes
                        const uint32_t kx = e == 0 ? 0xffff0000u : e == 1 ? 0x0000ffffu : 0xffffffffu;
                        const uint32_t ky = e == 2 ? 0xffff0000u : e == 3 ? 0x0000ffffu : 0xffffffffu;
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) {
                            const uint32_t nv = v_lds[dt * 16 + lj].bits, both = nv | nv << 16;
                            vv[i][kt][dt].x = (vv[i][kt][dt].x & kx) | (both & ~kx);
                            vv[i][kt][dt].y = (vv[i][kt][dt].y & ky) | (both & ~ky);
                        }
                    }
                }
            }
        }
        // the scores of all the round's keys, then one maximum, one factor for what was there before and their products (a block
        // past the wavefront's last counts for nothing and is jumped over: computed all the same, behind 100 tokens, where that is every
        // wavefront's second one, it made the kernel 3 to 8 % slower)
        const int last = min(p, w_end * 32 - 1);
        float s[PF][2][4];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < PF; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                if (i > 0 && kb0 + i >= w_end) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) s[i][kt][v] = -INFINITY;
                    continue;
                }
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kd = 0; kd < KD; ++kd)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kk[i][kt][kd]), q[kd], acc,
                                                                  0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int key = (kb0 + i) * 32 + kt * 16 + lg * 4 + v;
                    const bool vis = valid && key <= last && key >= lo;
                    s[i][kt][v] = vis ? acc[v] * d.scale : -INFINITY;
                    mx = fmaxf(mx, s[i][kt][v]);
                }
            }
        mx = fold_rows(mx, MaxOf());
        const float m_new = fmaxf(m_run, mx);
        const bool none = m_new == -INFINITY;
        const float from = none ? 0.f : m_new;             // (no key yet: exp(-infinity - 0) is zero)
        const float alpha = none ? 1.f : __expf(m_run - m_new);
        float sum = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) { o[dt][0] *= alpha; o[dt][1] *= alpha; o[dt][2] *= alpha; o[dt][3] *= alpha; }
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            if (i > 0 && kb0 + i >= w_end) continue;
            bf16x8 pb;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float pv = __expf(s[i][kt][v] - from);
                    sum += pv;
                    pb[kt * 4 + v] = static_cast<__bf16>(pv);
                }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const uint4 av = uint4{vv[i][0][dt].x, vv[i][0][dt].y, vv[i][1][dt].x, vv[i][1][dt].y};
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), pb, o[dt], 0, 0, 0);
            }
        }
        l_run = l_run * alpha + sum;
        m_run = m_new;
    }
    float l = l_run;
    l = fold_rows(l, AddOf());

    // every wavefront leaves its state in LDS; then all threads combine
    float* mine = wave_state + (wave * 16 + lj) * kRow;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 4; ++v) mine[dt * 16 + lg * 4 + v] = o[dt][v];
    if (lg == 0) {
        mine[HD] = m_run;
        mine[HD + 1] = l;
    }
    __syncthreads();
    const size_t row0 = static_cast<size_t>(tok) * nq + kh * group_size;
    // (the states of all wavefronts are read together, of four or eight; past the last one the last again, of which nothing counts: a weight of
    // zero would leave its infinities)
    auto combine = [&](auto most) {
        constexpr int N = decltype(most)::value;
        for (int idx = threadIdx.x; idx < group_size * HD; idx += n_threads) {
            const int r = idx / HD, c = idx % HD;
            float ms[N], ls[N], os[N], mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < N; ++w) {
                const float* st = wave_state + (min(w, n_waves - 1) * 16 + r) * kRow;
                const float m = st[HD];
                ms[w] = w < n_waves ? m : -INFINITY;
                ls[w] = st[HD + 1];
                os[w] = st[c];
                mx = fmaxf(mx, ms[w]);
            }
            if (__builtin_expect(n_waves < N, 0)) {
#pragma unroll
                for (int w = 1; w < N; ++w) {
                    ls[w] = w < n_waves ? ls[w] : 0.f;
                    os[w] = w < n_waves ? os[w] : 0.f;
                }
            }
            float num = 0.f, den = 0.f;
#pragma unroll
            for (int w = 0; w < N; ++w) {
                const float wgt = ms[w] == -INFINITY ? 0.f : __expf(ms[w] - mx);
                num += wgt * os[w];
                den += wgt * ls[w];
            }
            if (n_splits == 1) {
                out[(row0 + r) * HD + c] = from_float<bf16_t>(num / den);
            } else {
                const size_t prow = RANGED ? static_cast<size_t>(bx) * nq + kh * group_size + r
                                           : static_cast<size_t>(bz) * d.n_tokens * nq +
                                                 (MIXED ? static_cast<size_t>(b) * nq + kh * group_size : row0) + r;
                part_o[prow * HD + c] = num;
                if (c == 0) {
                    part_ml[prow * 2] = mx;
                    part_ml[prow * 2 + 1] = den;
                }
            }
        }
    };
    if (__builtin_expect(n_waves > 4, 1)) combine(std::integral_constant<int, 8>());
    else combine(std::integral_constant<int, 4>());
}

// INF: partial sums of the product that are read in one batch (FUSED)
template <int HD, int PF, bool FUSED, bool MIXED = false, bool RANGED = false, int INF = 8, bool WIDE = false>
__global__ __launch_bounds__(512) void attention_decode_kernel(
    // (what the first loads are addressed by: 14 words that arrive with the wavefronts; `lengths` is the table of ranges where
    // there is one)
    const int32_t* __restrict__ lengths, const int32_t* __restrict__ block_table, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int table_width, int page_size, int nkv, int n_splits, unsigned page_magic, unsigned split_magic,
    unsigned wave_magic, int group, int window, int n_tokens, float scale, int n_waves, const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len,
    FusedQkv f) {
    extern __shared__ float wave_state[];
    const DecodeSizes d{table_width, page_size, nkv, n_splits, page_magic, split_magic, wave_magic, group, window, n_tokens, scale, n_waves};
    decode_block<HD, PF, FUSED, MIXED, RANGED, INF, WIDE>(wave_state, blockIdx.x, blockIdx.y, blockIdx.z, lengths, block_table, k_cache, v_cache, d, qkv, out,
                                                    part_o, part_ml, q_start, q_len, f);
}

// Portions of prompts in blocks of 32 RB rows and, behind them in the same launch, the requests of one token dealt out by `ranges`
// (range_slots workgroups for each kv head).  The portions' longest block of rows and the decoded tokens' longest range take about as long as
// each other and neither fills the chip: 512 tokens of a new prompt beside 40 decoded ones behind 128 to 2,048, 12 heads of 128 on 2, are
// 48 workgroups of 20 us and 256 of 13, a layer 32.1 us one launch after the other and 21.9 so.  A CU holds one workgroup of either kind.
template <int HD, int RB, int KS>
__global__ __launch_bounds__(512) void attention_mixed_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_table, int table_width,
    const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len, const int32_t* __restrict__ kv_len,
    int n_seqs, int nq, int nkv, int page_size, int page_shift, float scale, int window, int late, int row_blocks, unsigned page_magic,
    const int32_t* __restrict__ ranges, int range_slots, float* __restrict__ range_o, float* __restrict__ range_ml) {
    static_assert(RB * KS == 8, "eight wavefronts, as the decoded tokens have");
    __shared__ __attribute__((aligned(128))) char smem[kRows32Lds<HD, RB, KS>];
    static_assert(kRows32Lds<HD, RB, KS> >= 8 * 16 * (HD + 2) * 4, "room for what eight wavefronts of decoded tokens leave");
    const int index = blockIdx.x;
    if (index < row_blocks) {
        rows32_block<HD, RB, KS, false>(smem, index, 0, qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs, nq, nkv,
                                      page_size, page_shift, scale, window, 1, nullptr, nullptr, 1, 0, (nq + 2 * nkv) * HD, late);
    } else {
        const int i = index - row_blocks;
        const DecodeSizes d{table_width, page_size, nkv, 1, page_magic, 0, (1u << 28) + 1, nq / nkv, window, n_seqs, scale, 8};
        decode_block<HD, 2, false, true, true, 8, false>(reinterpret_cast<float*>(smem), i % range_slots, i / range_slots, 0, ranges, block_table, k_cache, v_cache,
                                                  d, qkv, out, range_o, range_ml, q_start, q_len, FusedQkv{});
    }
}

// out[row, :] = sum_s exp(m_s - M) o_s / sum_s exp(m_s - M) l_s over the splits; one wavefront per row, R features of it a lane (R * 64
// of them or fewer).  Lane s takes split s's (maximum, sum) so that the weights of up to 64 splits are known after one round of loads;
// the first eight splits' partial outputs are asked for together with them (a part of a split without visible keys may hold anything:
// it is read and then dropped), the others eight at a time.  Against four features a lane whatever the head size and shuffles through LDS, the same
// step with this kernel alone exchanged, us: 14 heads of 64 on 2, 24 layers, 64 users behind 130 to 2,048 tokens 1,161 -> 1,141, 32 behind 2,048
// 1,024 -> 1,004; 12 of 128 on 2, 28 layers, 32 behind 1,500 to 2,000 1,837 -> 1,800, 40 beside a portion of 512 3,490 -> 3,467.  (A kernel trace has
// the same 4.9 us for both, the trips to memory behind attention's writes; the fastest 2.6 -> 1.5.)
template <int R>
__global__ __launch_bounds__(64) void attention_reduce_kernel(const float* __restrict__ part_o,
                                                              const float* __restrict__ part_ml,
                                                              const int32_t* __restrict__ q_start,
                                                              const int32_t* __restrict__ q_len,
                                                              const int32_t* __restrict__ dealt, int n_rows, int hd, int n_splits, int nq,
                                                              bf16_t* __restrict__ out) {
    const int row = blockIdx.x, lane = threadIdx.x;
    // q_start given: the parts are kept by request, of which only those of one token have any, and the result goes
    // to that token's row
    int out_row = row;
    if (q_start != nullptr) {
        const int seq = row / nq;
        if (dealt == nullptr && q_len[seq] != 1) return;
        out_row = q_start[seq] * nq + row % nq;
    }
    // dealt given: the parts lie by slot, and a request with a single one has its result already
    int first_part = row, between = n_rows;
    if (dealt != nullptr) {
        const int seq = row / nq;
        n_splits = dealt[2 * seq + 1];
        if (n_splits <= 1) return;
        first_part = dealt[2 * seq] * nq + row % nq;
        between = nq;
    }
    const float* from = part_o + static_cast<size_t>(first_part) * hd;
    const size_t step = static_cast<size_t>(between) * hd;
    int at[R];                                           // (a lane past the head's last feature reads that one again)
#pragma unroll
    for (int r = 0; r < R; ++r) at[r] = min(lane + r * kWave, hd - 1);
    float v[8][R];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r) v[i][r] = from[min(i, n_splits - 1) * step + at[r]];
    const size_t mine = (static_cast<size_t>(min(lane, n_splits - 1)) * between + first_part) * 2;
    const float m_read = part_ml[mine], l = part_ml[mine + 1];
    const float m = lane < n_splits ? m_read : -INFINITY;
    const float m_max = wave_max(m);
    const float wgt = m == -INFINITY ? 0.f : __expf(m - m_max);    // a split without visible keys weighs nothing
    const float inv = 1.0f / wave_sum(m == -INFINITY ? 0.f : wgt * l);
    float acc[R] = {};
    auto add = [&](int s0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wgt), s0 + i));
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] += w * (w != 0.f ? v[i][r] : 0.f);
        }
    };
    add(0);
    for (int s0 = 8; s0 < n_splits; s0 += 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) v[i][r] = from[min(s0 + i, n_splits - 1) * step + at[r]];
        add(s0);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (lane + r * kWave < hd) out[static_cast<size_t>(out_row) * hd + lane + r * kWave] = from_float<bf16_t>(acc[r] * inv);
}
static void launch_reduce(const float* part_o, const float* part_ml, const int32_t* q_start, const int32_t* q_len, const int32_t* dealt, int n_rows,
                          int hd, int n_splits, int nq, void* out, hipStream_t s) {
    auto launch = [&](auto kernel) {
        kernel<<<n_rows, 64, 0, s>>>(part_o, part_ml, q_start, q_len, dealt, n_rows, hd, n_splits, nq, static_cast<bf16_t*>(out));
    };
    if (hd <= 64) launch(attention_reduce_kernel<1>);
    else if (hd <= 128) launch(attention_reduce_kernel<2>);
    else launch(attention_reduce_kernel<4>);
}

template <int HD, int QT>
static int launch_mfma(const void* qkv, void* out, float* part_o, float* part_ml, const void* k_cache,
                       const void* v_cache, const int32_t* block_table, int table_width, const int32_t* q_start,
                       const int32_t* q_len, const int32_t* kv_len, int n_seqs, int n_tokens, int nq, int nkv,
                       int page_size, float scale, int window, int n_splits, int combine, hipStream_t s) {
    const int group = nq / nkv;
    const long groups = (static_cast<long>(n_tokens) * group) / (16 * QT) + n_seqs;   // upper bound
    dim3 grid(static_cast<unsigned>(groups), nkv, n_splits);
    attention_mfma_kernel<HD, QT><<<grid, 64, 0, s>>>(
        static_cast<const bf16_t*>(qkv), static_cast<bf16_t*>(out), part_o, part_ml,
        static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache), block_table, table_width, q_start,
        q_len, kv_len, n_seqs, n_tokens, nq, nkv, page_size, scale, window, n_splits);
    EGPT_CHECK_LAUNCH();
    if (n_splits > 1 && combine) {
        launch_reduce(part_o, part_ml, nullptr, nullptr, nullptr, n_tokens * nq, HD, n_splits, 1, out, s);
        EGPT_CHECK_LAUNCH();
    }
    return EGPT_OK;
}

constexpr int kDecodeLdsMost = 96 * 1024;       // bytes of LDS a workgroup of the decode kernel may ask for

template <auto Kernel>
static bool raise_lds() {
    static bool raised = false;
    if (!raised)
        raised = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kDecodeLdsMost) == hipSuccess;
    return raised;
}

// PF: key blocks per round of loads of a wavefront.  More of them in flight is fewer round trips but more
// registers; when there are so many workgroups that they must share CUs, fewer registers are worth more.
template <int HD, int PF>
static int launch_decode(const void* qkv, void* out, float* part_o, float* part_ml, const void* k_cache,
                         const void* v_cache, const int32_t* block_table, int table_width, const int32_t* q_start,
                         const int32_t* kv_len, int n_seqs, int n_tokens, int nq, int nkv, int page_size, float scale,
                         int window, int n_splits, int n_waves, int combine, const FusedQkv* fused,
                         const int32_t* q_len, const int32_t* ranges, int slots, hipStream_t s) {
    dim3 grid(n_seqs, nkv, n_splits);
    if (ranges) grid = dim3(slots, nkv);
    size_t lds = static_cast<size_t>(n_waves) * 16 * (HD + 2) * sizeof(float);
    if (fused) lds += 18 * HD * sizeof(bf16_t);          // 16 query heads, the new key and value
    if (lds > kDecodeLdsMost) return EGPT_UNSUPPORTED_SIZE;
    const FusedQkv fq = fused ? *fused : FusedQkv{};
    // (up to 16 partial sums behind the last one are asked for by their place, which has to be past the buffer's end and not around it)
    const bool wide = 2.0 * page_size * HD * nkv > 4294967295.0 || 2.0 * page_size * HD > 2147483647.0 ||
                      (fused && ((fq.in_splits + 32.0) * n_tokens * (nq + 2 * nkv) * HD * 4 > 2147483647.0 || (reinterpret_cast<uintptr_t>(fq.bias) & 3) != 0));
    auto launch = [&](auto kernel, bool (*raise)(), const int32_t* lengths, const void* q, const int32_t* counts, int splits) {
        // (eight wavefronts at head size 128: more than a kernel may take without being asked; once per instance)
        if (lds > 64 * 1024 && !raise()) return EGPT_UNSUPPORTED_SIZE;
        kernel<<<grid, n_waves * kWave, lds, s>>>(lengths, block_table, static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache),
                                                  table_width, page_size, nkv, splits, magic_of(page_size / 16), magic_of(splits), magic_of(n_waves), nq / nkv,
                                                  window, n_tokens, scale, n_waves, static_cast<const bf16_t*>(q), static_cast<bf16_t*>(out), part_o, part_ml, q_start, counts, fq);
        return EGPT_OK;
    };
    int e;
#define EGPT_DECODE(...) attention_decode_kernel<HD, __VA_ARGS__>, raise_lds<attention_decode_kernel<HD, __VA_ARGS__>>
    if (wide) {
        if (ranges && fused) e = launch(EGPT_DECODE(2, true, false, true, 8, true), ranges, nullptr, nullptr, 1);
        else if (ranges) e = launch(EGPT_DECODE(2, false, true, true, 8, true), ranges, qkv, q_len, 1);
        else if (fused) e = launch(EGPT_DECODE(2, true, false, false, 8, true), kv_len, nullptr, nullptr, n_splits);
        else if (q_len) e = launch(EGPT_DECODE(2, false, true, false, 8, true), kv_len, qkv, q_len, n_splits);
        else e = launch(EGPT_DECODE(2, false, false, false, 8, true), kv_len, qkv, nullptr, n_splits);
    } else if (ranges && fused) e = fused->in_splits > 8 ? launch(EGPT_DECODE(2, true, false, true, 16), ranges, nullptr, nullptr, 1)
                                                  : launch(EGPT_DECODE(2, true, false, true, 8), ranges, nullptr, nullptr, 1);
    else if (ranges) e = launch(EGPT_DECODE(2, false, true, true), ranges, qkv, q_len, 1);
    else if (fused) e = fused->in_splits > 8 ? launch(EGPT_DECODE(PF, true, false, false, 16), kv_len, nullptr, nullptr, n_splits)
                                             : launch(EGPT_DECODE(PF, true, false, false, 8), kv_len, nullptr, nullptr, n_splits);
    else if (q_len) e = launch(EGPT_DECODE(PF, false, true), kv_len, qkv, q_len, n_splits);
    else e = launch(EGPT_DECODE(PF, false), kv_len, qkv, nullptr, n_splits);
#undef EGPT_DECODE
    if (e != EGPT_OK) return e;
    EGPT_CHECK_LAUNCH();
    if (ranges) {
        launch_reduce(part_o, part_ml, q_start, q_len, ranges + slots * kRangeInts, n_tokens * nq, HD, 1, nq, out, s);
        EGPT_CHECK_LAUNCH();
    } else if (n_splits > 1 && combine) {
        launch_reduce(part_o, part_ml, q_len ? q_start : nullptr, q_len, nullptr, n_tokens * nq, HD, n_splits, nq, out, s);
        EGPT_CHECK_LAUNCH();
    }
    return EGPT_OK;
}

static int dispatch_decode(const void* qkv, void* out, float* part_o, float* part_ml, const void* k_cache,
                           const void* v_cache, const int32_t* block_table, int table_width, const int32_t* q_start,
                           const int32_t* kv_len, int n_seqs, int nq, int nkv, int hd, int page_size, float scale,
                           int window, int n_splits, int n_waves, int combine, int lean, const FusedQkv* fused,
                           const int32_t* q_len, const int32_t* ranges, int slots, hipStream_t s) {
    // lean: the variant with half the loads in flight and fewer registers, 2: with a block of keys a round (the caller's choice, see the wrapper)
#define EGPT_LAUNCH_DECODE(HD_, PF_)                                                                                \
    launch_decode<HD_, PF_>(qkv, out, part_o, part_ml, k_cache, v_cache, block_table, table_width, q_start, kv_len, \
                            n_seqs, n_seqs, nq, nkv, page_size, scale, window, n_splits, n_waves, combine, fused,   \
                            q_len, ranges, slots, s)
    if (ranges && (slots < n_seqs || slots > kRangeSlots || !part_o || !part_ml)) return EGPT_BAD_ARGUMENT;
    if (hd == 64) return lean == 2 ? EGPT_LAUNCH_DECODE(64, 1) : lean ? EGPT_LAUNCH_DECODE(64, 2) : EGPT_LAUNCH_DECODE(64, 4);
    return lean ? EGPT_LAUNCH_DECODE(128, 1) : EGPT_LAUNCH_DECODE(128, 2);
#undef EGPT_LAUNCH_DECODE
}

}  // namespace egpt

using namespace egpt;

// Prompt portions (and mixed batches) with keys and values shared through LDS by the wavefronts of a
// workgroup.  Same operands and meaning as egpt_paged_attention_mfma with n_splits == 1; page sizes that are
// powers of two.  `shape` = 10 * (tiles of 16 rows per workgroup) + (wavefronts that split a tile's keys).
template <int HD, int RT, int KS>
static void launch_tiled(const void* qkv, void* out, const void* k_cache, const void* v_cache,
                         const int32_t* block_table, int table_width, const int32_t* q_start, const int32_t* q_len,
                         const int32_t* kv_len, int n_seqs, int n_tokens, int nq, int nkv, int page_size,
                         int page_shift, float scale, int window, int skip_single, hipStream_t s) {
    const long groups = (static_cast<long>(n_tokens) * (nq / nkv)) / (16 * RT) + n_seqs;   // upper bound
    dim3 grid(static_cast<unsigned>(groups), nkv);
    attention_tiled_kernel<HD, RT, KS><<<grid, 64 * RT * KS, 0, s>>>(
        static_cast<const bf16_t*>(qkv), static_cast<bf16_t*>(out), static_cast<const bf16_t*>(k_cache),
        static_cast<const bf16_t*>(v_cache), block_table, table_width, q_start, q_len, kv_len, n_seqs, nq, nkv,
        page_size, page_shift, scale, window, skip_single);
}

template <int HD, int RB, int KS>
static void launch_rows32(const void* qkv, void* out, const void* k_cache, const void* v_cache,
                          const int32_t* block_table, int table_width, const int32_t* q_start, const int32_t* q_len,
                          const int32_t* kv_len, int n_seqs, int n_tokens, int nq, int nkv, int page_size,
                          int page_shift, float scale, int window, int skip_single, float* part_o, float* part_ml,
                          int n_splits, int late, hipStream_t s) {
    const long groups = (static_cast<long>(n_tokens) * (nq / nkv)) / (32 * RB) + n_seqs;   // upper bound
    dim3 grid(static_cast<unsigned>(groups * nkv), 1, n_splits);
#define EGPT_ROWS32_ARGS                                                                                           \
    static_cast<const bf16_t*>(qkv), static_cast<bf16_t*>(out), static_cast<const bf16_t*>(k_cache),               \
        static_cast<const bf16_t*>(v_cache), block_table, table_width, q_start, q_len, kv_len, n_seqs, nq, nkv,    \
        page_size, page_shift, scale, window, skip_single, part_o, part_ml, n_splits, n_tokens, late
    if (n_splits > 1) attention_rows32_kernel<HD, RB, KS, true><<<grid, 64 * RB * KS, 0, s>>>(EGPT_ROWS32_ARGS);
    else attention_rows32_kernel<HD, RB, KS, false><<<grid, 64 * RB * KS, 0, s>>>(EGPT_ROWS32_ARGS);
#undef EGPT_ROWS32_ARGS
    // (the rows of requests that were left out have no parts: what is combined for them is written over by the
    // kernel that takes them, which runs behind this one)
    if (n_splits > 1)
        launch_reduce(part_o, part_ml, nullptr, nullptr, nullptr, n_tokens * nq, HD, n_splits, 1, out, s);
}

template <int HD, int RB, int KS>
static int launch_mixed(const void* qkv, void* out, const void* k_cache, const void* v_cache, const int32_t* block_table, int table_width,
                        const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len, int n_seqs, int n_tokens, int nq, int nkv,
                        int page_size, int page_shift, float scale, int window, int late, const int32_t* ranges, int slots, float* range_o,
                        float* range_ml, hipStream_t s) {
    const long blocks = ((static_cast<long>(n_tokens) * (nq / nkv)) / (32 * RB) + n_seqs) * nkv;          // upper bound
    const long grid = blocks + static_cast<long>(slots) * nkv;
    if (grid > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    attention_mixed_kernel<HD, RB, KS><<<static_cast<unsigned>(grid), 512, 0, s>>>(
        static_cast<const bf16_t*>(qkv), static_cast<bf16_t*>(out), static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache),
        block_table, table_width, q_start, q_len, kv_len, n_seqs, nq, nkv, page_size, page_shift, scale, window, late, static_cast<int>(blocks),
        magic_of(page_size / 16), ranges, slots, range_o, range_ml);
    EGPT_CHECK_LAUNCH();
    launch_reduce(range_o, range_ml, q_start, q_len, ranges + slots * kRangeInts, n_seqs * nq, HD, 1, nq, out, s);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

static int paged_attention_tiled(const void* qkv, void* out, const void* k_cache, const void* v_cache,
                                          const int32_t* block_table, int table_width, const int32_t* q_start,
                                          const int32_t* q_len, const int32_t* kv_len, int n_seqs, int n_tokens,
                                          int nq, int nkv, int hd, int page_size, float scale, int window,
                                          int shape, int key_splits, float* part_o, float* part_ml,
                                          int single_splits, int single_waves, int single_lean, const int32_t* ranges, int slots,
                                          float* range_o, float* range_ml, void* stream) {
    if (!qkv || !out || !k_cache || !v_cache || !block_table || !q_start || !q_len || !kv_len)
        return EGPT_BAD_ARGUMENT;
    if (n_seqs <= 0 || n_tokens < 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || table_width <= 0 || window < 0)
        return EGPT_BAD_ARGUMENT;
    if ((hd != 64 && hd != 128) || page_size < 16 || (page_size & (page_size - 1)) != 0 || nkv > 65535)
        return EGPT_UNSUPPORTED_SIZE;
    const int late = shape >= 1000;
    shape -= late * 1000;
    if (late && shape < 100) return EGPT_BAD_ARGUMENT;
    const int skip_single = single_waves != 0;
    if (skip_single) {
        if (single_waves < 0 || single_splits < 1 || (single_splits > 1 && (!part_o || !part_ml)))
            return EGPT_BAD_ARGUMENT;
        if (nq / nkv > 16 || single_splits > 64 || single_waves > 8) return EGPT_UNSUPPORTED_SIZE;
    }
    if (shape >= 100 && page_size > 64) return EGPT_UNSUPPORTED_SIZE;     // its tiles of 64 keys are whole pages
    if (key_splits < 1 || (key_splits > 1 && (!part_o || !part_ml))) return EGPT_BAD_ARGUMENT;
    if (key_splits > 64 || (key_splits > 1 && shape < 100)) return EGPT_UNSUPPORTED_SIZE;
    if (n_tokens == 0) return EGPT_OK;
    int page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (ranges && key_splits == 1 && (shape == 142 || (shape == 124 && hd == 64))) {
        if (slots < n_seqs || slots > kRangeSlots) return EGPT_BAD_ARGUMENT;
        return (shape == 124 ? launch_mixed<64, 2, 4> : hd == 64 ? launch_mixed<64, 4, 2> : launch_mixed<128, 4, 2>)(
            qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs, n_tokens, nq, nkv, page_size, page_shift, scale,
            window, late, ranges, slots, range_o, range_ml, s);
    }
#define EGPT_TILED(HD_, RT_, KS_)                                                                                  \
    launch_tiled<HD_, RT_, KS_>(qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len,      \
                                n_seqs, n_tokens, nq, nkv, page_size, page_shift, scale, window, skip_single, s)
#define EGPT_ROWS32(HD_, RB_, KS_)                                                                                 \
    launch_rows32<HD_, RB_, KS_>(qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len,     \
                                 n_seqs, n_tokens, nq, nkv, page_size, page_shift, scale, window, skip_single,     \
                                 part_o, part_ml, key_splits, late, s)
    // shape = 10 * row tiles + key splits of a workgroup; 100 + 10 * blocks of 32 rows + key splits: the kernel of
    // 32-row blocks
    if (hd == 64) {
        switch (shape) {
            case 121: EGPT_ROWS32(64, 2, 1); break;
            case 122: EGPT_ROWS32(64, 2, 2); break;
            case 124: EGPT_ROWS32(64, 2, 4); break;
            case 141: EGPT_ROWS32(64, 4, 1); break;
            case 142: EGPT_ROWS32(64, 4, 2); break;
            case 181: EGPT_ROWS32(64, 8, 1); break;
            case 41: EGPT_TILED(64, 4, 1); break;
            case 42: EGPT_TILED(64, 4, 2); break;
            case 44: EGPT_TILED(64, 4, 4); break;
            case 22: EGPT_TILED(64, 2, 2); break;
            case 24: EGPT_TILED(64, 2, 4); break;
            default: return EGPT_BAD_ARGUMENT;
        }
    } else {
        switch (shape) {
            case 121: EGPT_ROWS32(128, 2, 1); break;
            case 122: EGPT_ROWS32(128, 2, 2); break;
            case 141: EGPT_ROWS32(128, 4, 1); break;
            case 142: EGPT_ROWS32(128, 4, 2); break;
            case 181: EGPT_ROWS32(128, 8, 1); break;
            case 41: EGPT_TILED(128, 4, 1); break;
            case 42: EGPT_TILED(128, 4, 2); break;
            case 22: EGPT_TILED(128, 2, 2); break;
            default: return EGPT_BAD_ARGUMENT;
        }
    }
#undef EGPT_TILED
#undef EGPT_ROWS32
    EGPT_CHECK_LAUNCH();
    if (skip_single)
        return dispatch_decode(qkv, out, ranges ? range_o : part_o, ranges ? range_ml : part_ml, k_cache, v_cache, block_table, table_width,
                               q_start, kv_len, n_seqs, nq, nkv, hd, page_size, scale, window, single_splits, single_waves, 1,
                               single_lean, nullptr, q_len, ranges, slots, s);
    return EGPT_OK;
}

constexpr int kLdsMost = 160 * 1024;
template <int HD, int RB, int KS, bool BIAS>
static int launch_heads32(const void* q, void* out, const void* k_cache, const void* v_cache, const int32_t* block_table, int table_width,
                          const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len, int n_seqs, int n_tokens, int nq, int nkv,
                          int page_size, int page_shift, float scale, int window, const float* table, int far, hipStream_t s) {
    const long blocks = ((static_cast<long>(n_tokens) * (nq / nkv)) / (32 * RB) + n_seqs) * nkv;          // upper bound
    const long lds = kRows32Lds<HD, RB, KS> + (BIAS ? static_cast<long>(nq / nkv) * bias_row(far) * 4 : 0);
    if (lds > kLdsMost || blocks > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    static bool raised = false;                      // (more than 64 KB: asked for once per instance)
    if (!raised) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_heads32_kernel<HD, RB, KS, BIAS>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                kLdsMost) != hipSuccess)
            return EGPT_UNSUPPORTED_SIZE;
        raised = true;
    }
    attention_heads32_kernel<HD, RB, KS, BIAS><<<static_cast<unsigned>(blocks), 64 * RB * KS, static_cast<size_t>(lds), s>>>(
        static_cast<const bf16_t*>(q), static_cast<bf16_t*>(out), static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache),
        block_table, table_width, q_start, q_len, kv_len, n_seqs, nq, nkv, page_size, page_shift, scale, window, table, far);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

extern "C" int egpt_heads_attention(const void* q, void* out, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                    int table_width, const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len, int n_seqs,
                                    int n_tokens, int nq, int nkv, int hd, int page_size, float scale, int window, const float* dist_bias,
                                    int dist_far, int row_blocks, void* stream) {
    if (!q || !out || !k_cache || !v_cache || !block_table || !q_start || !q_len || !kv_len) return EGPT_BAD_ARGUMENT;
    if (n_seqs <= 0 || n_tokens < 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || table_width <= 0 || window < 0 || !(scale > 0.f) || dist_far < 0 ||
        (row_blocks != 4 && row_blocks != 8))
        return EGPT_BAD_ARGUMENT;
    if ((hd != 64 && hd != 128) || page_size < 16 || page_size > 64 || (page_size & (page_size - 1)) != 0 || dist_far > 16384) return EGPT_UNSUPPORTED_SIZE;
    if (n_tokens == 0) return EGPT_OK;
    int page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define EGPT_HEADS32(HD_, RB_, KS_)                                                                                                    \
    (dist_bias ? launch_heads32<HD_, RB_, KS_, true> : launch_heads32<HD_, RB_, KS_, false>)(                                          \
        q, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs, n_tokens, nq, nkv, page_size, page_shift,  \
        scale, window, dist_bias, dist_far, s)
    if (hd == 64) return row_blocks == 4 ? EGPT_HEADS32(64, 4, 2) : EGPT_HEADS32(64, 8, 1);
    // (with a bias two slots of 128 keys and three of their values leave no room for its table)
    return row_blocks == 4 && !dist_bias ? EGPT_HEADS32(128, 4, 2) : EGPT_HEADS32(128, 8, 1);
#undef EGPT_HEADS32
}

extern "C" int egpt_paged_attention_tiled(const void* qkv, void* out, const void* k_cache, const void* v_cache,
                                          const int32_t* block_table, int table_width, const int32_t* q_start,
                                          const int32_t* q_len, const int32_t* kv_len, int n_seqs, int n_tokens,
                                          int nq, int nkv, int hd, int page_size, float scale, int window,
                                          int shape, int key_splits, float* part_o, float* part_ml,
                                          int single_splits, int single_waves, int single_lean, void* stream) {
    return paged_attention_tiled(qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs, n_tokens, nq, nkv,
                                 hd, page_size, scale, window, shape, key_splits, part_o, part_ml, single_splits, single_waves,
                                 single_lean, nullptr, 0, nullptr, nullptr, stream);
}

// The same with the requests of one token dealt out by `ranges` (egpt_decode_ranges) over `slots` workgroups of eight wavefronts
// per kv head; range_o [slots][nq][hd] and range_ml [slots][nq][2] take their parts.
extern "C" int egpt_paged_attention_mixed(const void* qkv, void* out, const void* k_cache, const void* v_cache,
                                          const int32_t* block_table, int table_width, const int32_t* q_start,
                                          const int32_t* q_len, const int32_t* kv_len, int n_seqs, int n_tokens,
                                          int nq, int nkv, int hd, int page_size, float scale, int window,
                                          int shape, int key_splits, float* part_o, float* part_ml,
                                          const int32_t* ranges, int slots, float* range_o, float* range_ml, void* stream) {
    if (!ranges || !range_o || !range_ml || slots < n_seqs) return EGPT_BAD_ARGUMENT;
    if (slots > kRangeSlots) return EGPT_UNSUPPORTED_SIZE;
    return paged_attention_tiled(qkv, out, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs, n_tokens, nq, nkv,
                                 hd, page_size, scale, window, shape, key_splits, part_o, part_ml, 1, 8, 1, ranges, slots, range_o,
                                 range_ml, stream);
}

// One decoded token per request (n_tokens == n_seqs, q_len all 1), nq / nkv <= 16: workgroups of n_waves
// wavefronts (1..8) per (request, kv head, key split).  Same operands and meaning as egpt_paged_attention_mfma.
extern "C" int egpt_paged_attention_decode(const void* qkv, void* out, float* part_o, float* part_ml,
                                           const void* k_cache, const void* v_cache, const int32_t* block_table,
                                           int table_width, const int32_t* q_start, const int32_t* kv_len, int n_seqs,
                                           int nq, int nkv, int hd, int page_size, float scale, int window,
                                           int n_splits, int n_waves, int combine, int lean, void* stream) {
    if (!qkv || !out || !k_cache || !v_cache || !block_table || !q_start || !kv_len) return EGPT_BAD_ARGUMENT;
    if (n_seqs <= 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || table_width <= 0 || window < 0 || n_splits < 1 ||
        (n_splits > 1 && (!part_o || !part_ml)))
        return EGPT_BAD_ARGUMENT;
    if ((hd != 64 && hd != 128) || page_size < 16 || page_size % 16 != 0 || nq / nkv > 16 || nkv > 65535 || n_splits > 64 ||
        n_waves < 1 || n_waves > 8)
        return EGPT_UNSUPPORTED_SIZE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dispatch_decode(qkv, out, part_o, part_ml, k_cache, v_cache, block_table, table_width, q_start, kv_len,
                           n_seqs, nq, nkv, hd, page_size, scale, window, n_splits, n_waves, combine, lean, nullptr, nullptr, nullptr, 0, s);
}

// The same with the QKV epilogue folded in: the queries, and the new token's key and value, are computed from
// the float32 QKV product (partial sums qkv_prod [in_splits][n_seqs][(nq + 2 nkv) * hd], the rows' sums of
// squares row_ss [ss_splits][n_seqs] or null, bias or null), rotated over the whole head by the angles whose
// cosines and sines are in cos_sin [n_seqs][hd / 2][2] (egpt_rope_table), and the key and value are stored at
// slots[t] of the caches.  Token t belongs to request t.
static int attention_decode_fused(const float* qkv_prod, int in_splits, const float* row_ss, int ss_splits,
                                           int hidden, float eps, const void* bias, const float* cos_sin,
                                           const int32_t* slots, void* out, float* part_o,
                                           float* part_ml, void* k_cache, void* v_cache, const int32_t* block_table,
                                           int table_width, const int32_t* q_start, const int32_t* kv_len, int n_seqs,
                                           int nq, int nkv, int hd, int page_size, float scale, int window,
                                           int n_splits, int n_waves, int combine, int lean, const int32_t* ranges,
                                           int range_slots, void* stream) {
    if (!qkv_prod || in_splits < 1 || !cos_sin || !slots || !out || !k_cache || !v_cache ||
        !block_table || !q_start || !kv_len || (row_ss && (ss_splits < 1 || hidden < 1)))
        return EGPT_BAD_ARGUMENT;
    if (n_seqs <= 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || table_width <= 0 || window < 0 || n_splits < 1 ||
        (n_splits > 1 && (!part_o || !part_ml)))
        return EGPT_BAD_ARGUMENT;
    if ((hd != 64 && hd != 128) || page_size < 16 || page_size % 16 != 0 || nq / nkv > 16 || nkv > 65535 || n_splits > 64 ||
        n_waves < 1 || n_waves > 8)
        return EGPT_UNSUPPORTED_SIZE;
    FusedQkv f = {};
    f.prod = qkv_prod; f.in_splits = in_splits;
    f.row_ss = row_ss; f.ss_splits = row_ss ? ss_splits : 0;
    f.inv_hidden = row_ss ? 1.0f / static_cast<float>(hidden) : 0.f;
    f.eps = eps;
    f.bias = static_cast<const bf16_t*>(bias);
    f.cos_sin = cos_sin; f.slots = slots;
    f.k_cache_w = static_cast<bf16_t*>(k_cache); f.v_cache_w = static_cast<bf16_t*>(v_cache);
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dispatch_decode(nullptr, out, part_o, part_ml, k_cache, v_cache, block_table, table_width, q_start, kv_len,
                           n_seqs, nq, nkv, hd, page_size, scale, window, n_splits, n_waves, combine, lean, &f, nullptr, ranges, range_slots, s);
}

extern "C" int egpt_attention_decode_fused(const float* qkv_prod, int in_splits, const float* row_ss, int ss_splits,
                                           int hidden, float eps, const void* bias, const float* cos_sin,
                                           const int32_t* slots, void* out, float* part_o,
                                           float* part_ml, void* k_cache, void* v_cache, const int32_t* block_table,
                                           int table_width, const int32_t* q_start, const int32_t* kv_len, int n_seqs,
                                           int nq, int nkv, int hd, int page_size, float scale, int window,
                                           int n_splits, int n_waves, int combine, int lean, void* stream) {
    return attention_decode_fused(qkv_prod, in_splits, row_ss, ss_splits, hidden, eps, bias, cos_sin, slots, out, part_o, part_ml, k_cache,
                                  v_cache, block_table, table_width, q_start, kv_len, n_seqs, nq, nkv, hd, page_size, scale, window,
                                  n_splits, n_waves, combine, lean, nullptr, 0, stream);
}

// The same with the keys dealt out by `ranges` (egpt_decode_ranges) over range_slots workgroups of eight wavefronts per kv head;
// part_o [range_slots][nq][hd] and part_ml [range_slots][nq][2] take their parts, which are combined into out.
extern "C" int egpt_attention_decode_ranged(const float* qkv_prod, int in_splits, const float* row_ss, int ss_splits,
                                            int hidden, float eps, const void* bias, const float* cos_sin,
                                            const int32_t* slots, void* out, float* part_o,
                                            float* part_ml, void* k_cache, void* v_cache, const int32_t* block_table,
                                            int table_width, const int32_t* q_start, const int32_t* kv_len, int n_seqs,
                                            int nq, int nkv, int hd, int page_size, float scale, int window,
                                            const int32_t* ranges, int range_slots, void* stream) {
    if (!ranges || !part_o || !part_ml || range_slots < n_seqs) return EGPT_BAD_ARGUMENT;
    if (range_slots > kRangeSlots) return EGPT_UNSUPPORTED_SIZE;
    return attention_decode_fused(qkv_prod, in_splits, row_ss, ss_splits, hidden, eps, bias, cos_sin, slots, out, part_o, part_ml, k_cache,
                                  v_cache, block_table, table_width, q_start, kv_len, n_seqs, nq, nkv, hd, page_size, scale, window,
                                  1, 8, 1, 1, ranges, range_slots, stream);
}

// bfloat16 only; head size 64 or 128; page size a multiple of 16.  rows_per_wave: 16 (decoded tokens) or 32.
// part_o [n_splits][n_tokens][nq][hd] and part_ml [n_splits][n_tokens][nq][2] float32 are needed when n_splits > 1;
// with combine == 0 they are left for the caller to combine (the output projection does it while it stages x).
extern "C" int egpt_paged_attention_mfma(const void* qkv, void* out, float* part_o, float* part_ml, const void* k_cache,
                                         const void* v_cache, const int32_t* block_table, int table_width,
                                         const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len,
                                         int n_seqs, int n_tokens, int nq, int nkv, int hd, int page_size, float scale,
                                         int window, int n_splits, int rows_per_wave, int combine, void* stream) {
    if (!qkv || !out || !k_cache || !v_cache || !block_table || !q_start || !q_len || !kv_len)
        return EGPT_BAD_ARGUMENT;
    if (n_seqs <= 0 || n_tokens < 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || table_width <= 0 || window < 0 ||
        n_splits < 1 || (n_splits > 1 && (!part_o || !part_ml)))
        return EGPT_BAD_ARGUMENT;
    if ((hd != 64 && hd != 128) || page_size < 16 || page_size % 16 != 0 || nkv > 65535 || n_splits > 64 ||
        (rows_per_wave != 16 && rows_per_wave != 32))
        return EGPT_UNSUPPORTED_SIZE;
    if (n_tokens == 0) return EGPT_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define EGPT_ATTN_ARGS                                                                                              \
    qkv, out, part_o, part_ml, k_cache, v_cache, block_table, table_width, q_start, q_len, kv_len, n_seqs, n_tokens, \
        nq, nkv, page_size, scale, window, n_splits, combine, s
    if (hd == 64) return rows_per_wave == 16 ? launch_mfma<64, 1>(EGPT_ATTN_ARGS) : launch_mfma<64, 2>(EGPT_ATTN_ARGS);
    return rows_per_wave == 16 ? launch_mfma<128, 1>(EGPT_ATTN_ARGS) : launch_mfma<128, 2>(EGPT_ATTN_ARGS);
#undef EGPT_ATTN_ARGS
}

// The table by which the decode kernels above deal out the keys (see decode_ranges_kernel): slots * 8 + n_seqs * 2 numbers.
extern "C" int egpt_decode_ranges(const int32_t* kv_len, const int32_t* q_start, const int32_t* q_len, int n_seqs, int slots, int window,
                                  int32_t* table, void* stream) {
    if (!kv_len || !q_start || !table || n_seqs <= 0 || slots < n_seqs || window < 0) return EGPT_BAD_ARGUMENT;
    if (slots > kRangeSlots) return EGPT_UNSUPPORTED_SIZE;
    decode_ranges_kernel<<<1, kRangeSlots, 0, static_cast<hipStream_t>(stream)>>>(kv_len, q_start, q_len, n_seqs, slots, window, table);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

// Combines the parts that egpt_paged_attention_mfma left with combine == 0: out [n_rows][hd] bfloat16.
extern "C" int egpt_attention_combine(const float* part_o, const float* part_ml, void* out, int n_rows, int hd,
                                      int n_splits, void* stream) {
    if (!part_o || !part_ml || !out || n_rows < 0 || hd <= 0 || n_splits < 1) return EGPT_BAD_ARGUMENT;
    if (n_splits > 64 || hd > 256) return EGPT_UNSUPPORTED_SIZE;
    if (n_rows == 0) return EGPT_OK;
    launch_reduce(part_o, part_ml, nullptr, nullptr, nullptr, n_rows, hd, n_splits, 1, out, static_cast<hipStream_t>(stream));
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}
