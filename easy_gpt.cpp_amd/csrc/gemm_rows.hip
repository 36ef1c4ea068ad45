// out[m, n] = sum_k x[m, k] * w[n, k] in bfloat16 for many rows of x (more than 16): tiles staged through LDS by loads that
// go there directly, v_mfma_f32_16x16x32_bf16, float32 accumulation.  The result leaves as bfloat16, as float32 partial
// sums of a split k range, or activated: w = [gate; up] and out = act(x gate^T) * (x up^T), both factors still in float32.
//
// A workgroup owns BM rows of x and BN rows of w (columns of the result) and walks k in steps of 64.  A step of an operand
// lies in LDS as rows of 128 bytes whose eight pieces of 16 bytes are exchanged by the row's number (piece p of row r stands
// in place p ^ (r & 7)): the lanes that read one piece of many rows hit different banks (no conflicts in the counters).  A
// load puts a lane's 16 bytes at the wavefront's base + 16 x lane, so the exchange is made in the addresses that lanes load from.
// A step is computed in two halves of 32 values of k.  Between them stands the one barrier of the step, with the second
// half's operands in registers already; behind it the next loads go out and the next step's first half is read under the
// second half's products.
//
// Tiles of few rows and columns keep five or six steps of both operands on their way where there are few of them: a step of 64 x 64
// takes 0.17 us so and 0.32 with two and three, which is the L2's latency (600 x 896 x 4,864 in one range 30.4 us -> 19.1).
// With 17 to 64 rows the deep rings are what streams the weights: one workgroup to a CU, at 64 rows 1,536 x 8,960 and the norm behind it in
// 14.7 us (20.4 by the weight-streaming kernel of gemm_skinny.hip, which holds one step of w in registers), 152,064 x 3,584 in 217,
// 5.0 TB/s; `_few_plan` in kernels/hip.py chooses the shape.
// A workgroup stays for several tiles: as many are launched as the CUs hold, and the loads of a workgroup's next tile go out under
// the last steps of the one before, so that a tile's first products do not wait for memory and the result leaves meanwhile.
//
// What bounds it: alone, the loop runs at 1.9 PFLOP/s on zeros and 1.6 on random numbers (the card then lowers its clock): 2,640
// cycles a step of 256 x 256, where the products take 2,048, and so do the LDS's reads and writes together.  Beside its steps
// a tile of 256 x 256 takes 10,000 cycles when it is activated (47,000 in all at 14 steps of k): 128 exponentials and
// reciprocals a lane, each of four issues, and the instructions around them, two wavefronts to a SIMD.  What it was before: a
// workgroup per tile, expf and the division in full, all rows of x before the next columns (us, weights from memory): 2,048 rows
// x 9,728 x 896 gated 53.3 -> 41.2, 8,191 x 9,728 x 896 172 -> 127, 8,191 x 17,920 x 1,536 444 -> 351, 2,048 x 37,888 x 3,584 461 -> 416;
// 8,191 x 896 x 896 23.1 -> 18.2.  Of that the strips of eight tiles of rows (`item_of`) are the 8,191 x 17,920 x 1,536's 442 -> 361: an
// XCD's 32 workgroups otherwise read 32 tiles of x for one of w.  Four wavefronts of 128 x 128 (fewer LDS reads): the registers do
// not suffice, 3,300 cycles a step.
// The weights come from memory, and all workgroups that share a tile of w ask for it at the same time, so nobody finds it in
// the L2 and everybody waits for memory's latency: two steps of w and one of x are on their way (160 KB of LDS).  Deeper rings in
// steps of 32 values (64-byte pieces of rows) gained nothing, 32x32x16 products are 7 % slower on random numbers.
// `_own_rows`, `_own_short` and `_own_gate` in kernels/hip.py draw the lines to the library, with both sides' times.
#include <type_traits>

#include "api.h"
#include "common.h"
#include "lds_loads.h"

namespace egpt {

typedef __attribute__((ext_vector_type(8))) __bf16 r_bf16x8;
typedef __attribute__((ext_vector_type(4))) float r_f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 r_bf16x4;
typedef __attribute__((ext_vector_type(2))) unsigned r_u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned r_u32x4;

constexpr int kLdsOfCu = 160 * 1024;
constexpr int kStrip = 8;                      // tiles of rows that are walked together, column by column
constexpr int kRowsStep = 64;                  // values of k per step: 128 bytes a row

// gate_activation of four values.  A wavefront issues a vector instruction in four cycles and holds 64 gates a lane, so what an
// activation takes is seen in the kernel: expf and the division with their cases spelled out are some 45 instructions a value
// (5 us of a tile of 256 x 256), these 15.  The exponential's argument is split as expf splits it, into a whole power of two, which
// an addition leaves in the low bits of a float32, and the rest with log2(e) in two parts; a reciprocal is made good by the
// division's remainder.  No case of either arises while |exponent| < 87; beyond it the general form.  Errors in units of the last
// place, this and gate_activation: z from -80 to -20 0.355 and 0.353 on average, 1.86 and 1.86 at most, -20 to -6 0.373 and 0.370, 2.72 and
// 2.72, -1 to 0 0.412 and 0.411, 2.01 and 2.01, 0 to 6 alike.  (Two instructions fewer, with the exponential of the whole argument and its rounding
// error put back by a factor: 1.68 and 0.60 in the first two ranges, 5.8 at most.)
template <int ACT>
__device__ __forceinline__ r_f32x4 gate4(r_f32x4 z) {
    r_f32x4 v;
    float most = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float y = gate_exponent(z[e], ACT);
        most = fmaxf(most, fabsf(y));
        constexpr float kWhole = 12583039.0f;                // 1.5 * 2^23 + 127: the sum's low bits are the power's exponent
        const float whole = fmaf(y, -1.442695041f, kWhole);
        const float rest = fmaf(y, -1.925962989e-8f, fmaf(y, -1.442695041f, kWhole - whole));
        const float d = fmaf(__builtin_amdgcn_exp2f(rest), __uint_as_float(__float_as_uint(whole) << 23), 1.0f);
        const float r = __builtin_amdgcn_rcpf(d), q = z[e] * r;
        v[e] = fmaf(fmaf(-q, d, z[e]), r, q);
    }
    if (!(most < 87.f)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gate_activation(z[e], ACT);
    }
    return v;
}

enum RowsOut { kRowsBf16 = 0, kRowsF32 = 1, kRowsGated = 2, kRowsRelu2 = 3, kRowsRotated = 4 };

// kRowsRotated: w makes queries, keys and values, whole heads of 2 `half` columns each, and what a tile ends with is what
// qkv_rope_store_rows_kernel does with such a product, operation for operation: bias, the rotation of queries and keys, keys and values
// into their pages.  `n` counts pairs (i, i + half) of a head's columns; a wavefront holds both of a pair as it holds gate and up.
struct RotatedOut {
    const bf16_t* bias;            // [2 n] or null
    const float* cos_sin;          // [rows of x][half][2]
    const int32_t* slots;          // [rows of x] page * page_size + offset
    bf16_t* k_cache;
    bf16_t* v_cache;
    int nq, nkv, half, page_size;
};

// Products of rows grouped by expert (moe.hip makes the table of tiles): tile i has rows tiles[3 i + 2 ..] of one expert, the
// numbers of tiles[1 + 3 i ..] being the expert, the tile's first grouped row and its rows; w is [experts][rows of w][k].
struct Groups {
    const int32_t* tiles;          // null: one matrix for all rows
    const int32_t* row_token;      // the row of x that a grouped row reads (null: the grouped row itself)
    int x_rows;                    // rows of x
};

template <int BM, int BN, int WM, int WN, int XB, int WB, int OUT, bool GROUPED>
__global__ __launch_bounds__(WM * WN * 64, BM * BN / (WM * WN) > 8192 ? 1 : 2) void gemm_rows_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k, int splits,
    int steps_per_split, int act, Groups groups, RotatedOut rot) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = WM * WN;
    constexpr int TM = BM / WM / 16, TN = BN / WN / 16;        // 16 x 16 tiles of a wavefront
    constexpr int XL = BM / 8 / NW, WL = BN / 8 / NW;          // loads of a wavefront per step: eight rows each
    static_assert(XL * 8 * NW == BM && WL * 8 * NW == BN, "a step is whole loads");
    constexpr int kXBytes = BM * 128, kWBytes = BN * 128;
    __shared__ __attribute__((aligned(128))) char xs[XB * kXBytes];
    __shared__ __attribute__((aligned(128))) char ws[WB * kWBytes];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int li = lane % 16, lg = lane / 16;
    const int wm = wave / WN, wn = wave % WN;

    // Workgroups are handed to the eight dies in turn: a die gets a contiguous range of items, rows of x fastest, so that
    // its L2 holds the few rows of w and x that its tiles share.  A workgroup takes items blockIdx.x, blockIdx.x +
    // gridDim.x ... (a grid of several items to a workgroup is a multiple of eight).
    constexpr int BC = OUT == kRowsGated || OUT == kRowsRotated ? BN / 2 : BN;         // columns of the result (or pairs) in a tile
    const int mt = GROUPED ? groups.tiles[0] : (m + BM - 1) / BM, nt = (n + BC - 1) / BC;
    const int tiles = mt * nt, items = tiles * splits;
    if (GROUPED && static_cast<int>(blockIdx.x) >= items) return;      // (the grid is sized for the most tiles that the rows can make)
    const int total = k / kRowsStep;
    const size_t row_bytes = static_cast<size_t>(k) * 2;
    const bool gather = GROUPED && groups.row_token != nullptr;
    struct Item {
        int m0, n0, rows, split, begin, end;               // first row, first column, rows, range of k: its number, its steps
        r_i32x4 x, w;                                      // operands from the tile's first row on (nothing beyond its last)
    };
    auto item_of = [&](int index) {
        Item it;
        if (index >= items) {                              // none: loads from it touch no memory
            it.m0 = it.n0 = it.rows = it.split = it.begin = it.end = 0;
            it.x = buffer_of(x, 0);
            it.w = buffer_of(w, 0);
            return it;
        }
        const int q = items / 8, r = items % 8, d = index % 8;
        const int item = d * q + (d < r ? d : r) + index / 8;
        const bf16_t* from = w;
        if (GROUPED) {
            // all columns of a tile of rows after each other: an expert's matrix stays in the die's L2 for its tiles
            const int32_t* entry = groups.tiles + 1 + 3 * (item / nt);
            it.m0 = entry[1];
            it.n0 = item % nt * BC;
            it.rows = entry[2];
            it.split = 0;
            from += static_cast<size_t>(entry[0]) * (OUT == kRowsGated ? 2 * n : n) * k;
        } else {
            it.split = splits == 1 ? 0 : item / tiles;
            const int tile = item - it.split * tiles;
            if (mt == 1) {                                 // (a division is 25 instructions, in front of everything)
                it.m0 = 0;
                it.n0 = tile * BC;
            } else {
                const int strips = (mt + kStrip - 1) / kStrip, per_strip = (mt + strips - 1) / strips;
                const int strip = tile / (per_strip * nt), top = strip * per_strip;
                const int high = min(per_strip, mt - top), at = tile - top * nt, column = at / high;
                it.m0 = (top + at - column * high) * BM;
                it.n0 = column * BC;
            }
            it.rows = min(m - it.m0, BM);
        }
        it.begin = it.split * steps_per_split;
        it.end = min(total, it.begin + steps_per_split);
        it.x = gather ? buffer_of(x, groups.x_rows * row_bytes) : buffer_of(x + static_cast<size_t>(it.m0) * k, it.rows * row_bytes);
        const int w0 = OUT == kRowsRotated ? it.n0 / rot.half * 2 * rot.half + it.n0 % rot.half : it.n0;      // (a tile is whole heads or a part of one)
        it.w = buffer_of(from + static_cast<size_t>(w0) * k,
                         (OUT == kRowsGated || OUT == kRowsRotated ? 2 * n - w0 : min(n - it.n0, BN)) * row_bytes);
        return it;
    };
    int index = blockIdx.x;
    Item now = item_of(index);

    // ---- loads: a lane's byte offsets from the tile's first rows, the same for every tile (what lies beyond an operand's
    // last row reads as zero; gate columns beyond the last are up columns, and nobody stores them)
    const int piece = (lane % 8) ^ (lane / 8);
    int xo[XL], wo[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        int g = (wave * XL + i) * 8 + lane / 8;
        if (gather) g = groups.row_token[now.m0 + min(g, now.rows - 1)];
        xo[i] = g * static_cast<int>(row_bytes) + piece * 16;
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int r = (wave * WL + i) * 8 + lane / 8;
        int g = r;
        if (OUT == kRowsGated) {
            // a wavefront's columns: the first half of them gates, the second half the up columns of the same numbers
            constexpr int C = BN / WN;
            g = r / C * (C / 2) + r % (C / 2) + (r % C >= C / 2 ? n : 0);
        }
        if (OUT == kRowsRotated) {
            // and so are the first and the second columns of pairs
            constexpr int C = BN / WN;
            const int pair = r / C * (C / 2) + r % (C / 2);
            g = pair / rot.half * 2 * rot.half + pair % rot.half + (r % C >= C / 2 ? rot.half : 0);
        }
        wo[i] = g * static_cast<int>(row_bytes) + piece * 16;
    }
    // where the next step's loads of an operand come from: `left` steps of an item from byte `at` of its rows on, `by` further
    // each (an item that is none stays where it is)
    struct Source {
        r_i32x4 rows;
        int at, by, left;
    };
    auto source_x = [&](const Item& it) { return Source{it.x, it.begin * (kRowsStep * 2), it.rows > 0 ? kRowsStep * 2 : 0, it.rows > 0 ? it.end - it.begin : 1 << 30}; };
    auto source_w = [&](const Item& it) { return Source{it.w, it.begin * (kRowsStep * 2), it.rows > 0 ? kRowsStep * 2 : 0, it.rows > 0 ? it.end - it.begin : 1 << 30}; };
    auto load_x = [&](int buffer, Source& from) {
#pragma unroll
        for (int i = 0; i < XL; ++i) load_to_lds(from.rows, xo[i], from.at, xs + buffer * kXBytes + (wave * XL + i) * 1024);
        from.at += from.by;
        --from.left;
    };
    // at most this many loads behind those of the step that is waited for: step s asks for x of step s + XB, then for w of s + WB
    constexpr int kBehind = XB < WB ? WL + (XB - 2) * (XL + WL) : (WB - 2) * (XL + WL);
    static_assert(XB >= 2 && XB <= WB, "the order of a step's loads");
    auto load_w = [&](int buffer, Source& from) {
#pragma unroll
        for (int i = 0; i < WL; ++i) load_to_lds(from.rows, wo[i], from.at, ws + buffer * kWBytes + (wave * WL + i) * 1024);
        from.at += from.by;
        --from.left;
    };
    // ---- operands of a half step
    const int xa = (wm * (BM / WM) + li) * 128, wa = (wn * (BN / WN) + li) * 128;
    const int place[2] = {((0 + lg) ^ (li & 7)) * 16, ((4 + lg) ^ (li & 7)) * 16};
    r_bf16x8 xf[2][TM], wf[2][TN];
    auto read = [&](int xb, int wb, int h) {
        const char* xfrom = xs + xb * kXBytes + xa + place[h];
        const char* wfrom = ws + wb * kWBytes + wa + place[h];
#pragma unroll
        for (int j = 0; j < TN; ++j) wf[h][j] = *reinterpret_cast<const r_bf16x8*>(wfrom + j * 2048);
#pragma unroll
        for (int i = 0; i < TM; ++i) xf[h][i] = *reinterpret_cast<const r_bf16x8*>(xfrom + i * 2048);
    };
    r_f32x4 acc[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = r_f32x4{0.f, 0.f, 0.f, 0.f};
    };
    auto multiply = [&](int h) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][j], xf[h][i], acc[i][j], 0, 0, 0);
        constexpr int per = TM * TN / (TM + TN) > 0 ? TM * TN / (TM + TN) : 1;
#pragma unroll
        for (int i = 0; i < TM + TN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, per, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // ---- the result: a lane holds columns 4 lg .. 4 lg + 3 of row li of every 16 x 16 tile (n is a multiple of four).  Rounded
    // results of two neighbouring tiles change places between lanes, so that a lane stores 16 bytes and four of them 64 bytes
    // of a row (8,191 x 896 x 896: 21.0 us with 8 bytes a lane, 18.2 so).  Every
    // wavefront makes at least kStores stores whatever the tile's edges are (those beyond an edge go nowhere), so that the
    // first wait of the next item can count them.
    constexpr int TC = OUT == kRowsGated ? TN / 2 : TN;
    constexpr bool kPairs = OUT != kRowsF32 && TC % 2 == 0;
    constexpr int kStores = kPairs ? TM * TC / 2 : TM * TC;
    constexpr int kOutBytes = OUT == kRowsF32 ? 4 : 2;
    auto store_as = [&](auto activation) {
        constexpr int ACT = decltype(activation)::value;
        char* from = static_cast<char*>(out) + (static_cast<size_t>(now.split) * m + now.m0) * n * kOutBytes;
        const auto to = __builtin_amdgcn_make_buffer_rsrc(from, 0, now.rows * n * kOutBytes, 0x00020000);
        const int col0 = now.n0 + wn * (BC / WN);
        auto value = [&](int i, int j) {
            r_f32x4 v = acc[i][j];
            if constexpr (OUT == kRowsGated) v = gate4<ACT>(v) * acc[i][j + TN / 2];
            if constexpr (OUT == kRowsRelu2) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = fmaxf(v[e], 0.f) * fmaxf(v[e], 0.f);
            }
            return v;
        };
        auto rounded = [&](int i, int j) { return __builtin_bit_cast(r_u32x2, __builtin_convertvector(value(i, j), r_bf16x4)); };
        if (kPairs && n % 8 == 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int at = (wm * (BM / WM) + i * 16 + li) * n;
#pragma unroll
                for (int j = 0; j < TC / 2 * 2; j += 2) {
                    const r_u32x2 a = rounded(i, j), b = rounded(i, j + 1);
                    const r_u32x2 p = __builtin_bit_cast(r_u32x2, __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false));
                    const r_u32x2 q = __builtin_bit_cast(r_u32x2, __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false));
                    const int col = col0 + (j + lg % 2) * 16 + lg / 2 * 8;
                    __builtin_amdgcn_raw_buffer_store_b128(r_u32x4{p[0], q[0], p[1], q[1]}, to, col < n ? (at + col) * 2 : 0x7ffffff0, 0, 0);
                }
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int at = (wm * (BM / WM) + i * 16 + li) * n;
#pragma unroll
            for (int j = 0; j < TC; ++j) {
                const int col = col0 + j * 16 + lg * 4, offset = col < n ? (at + col) * kOutBytes : 0x7ffffff0;
                if constexpr (OUT == kRowsF32) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(r_u32x4, value(i, j)), to, offset, 0, 0);
                else __builtin_amdgcn_raw_buffer_store_b64(rounded(i, j), to, offset, 0, 0);
            }
        }
    };
    [[maybe_unused]] auto store_rotated = [&]() {
        const int width = 2 * n;
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) {
            const int pair = now.n0 + wn * (BC / WN) + j * 16 + lg * 4;               // the first of this lane's four
            if (pair >= n) continue;
            const int head = pair / rot.half, at = pair % rot.half, col = head * 2 * rot.half + at;
            const bool is_v = head >= rot.nq + rot.nkv;
            r_f32x4 ba{0.f, 0.f, 0.f, 0.f}, bb = ba;
            if (rot.bias) {
                ba = __builtin_convertvector(*reinterpret_cast<const r_bf16x4*>(rot.bias + col), r_f32x4);
                bb = __builtin_convertvector(*reinterpret_cast<const r_bf16x4*>(rot.bias + col + rot.half), r_f32x4);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int r = wm * (BM / WM) + i * 16 + li;
                if (r >= now.rows) continue;
                const size_t t = static_cast<size_t>(now.m0) + r;
                r_f32x4 a = acc[i][j], b = acc[i][j + TN / 2];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[e] = scale_then_bias(a[e], 1.f, ba[e]);
                    b[e] = scale_then_bias(b[e], 1.f, bb[e]);
                }
                if (!is_v) {
                    const r_f32x4* cs = reinterpret_cast<const r_f32x4*>(rot.cos_sin + (t * rot.half + at) * 2);
                    const r_f32x4 c0 = cs[0], c1 = cs[1];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float ra, rb;
                        rotate_pair(a[e], b[e], e < 2 ? c0[2 * e] : c1[2 * e - 4], e < 2 ? c0[2 * e + 1] : c1[2 * e - 3], ra, rb);
                        a[e] = ra;
                        b[e] = rb;
                    }
                }
                const r_bf16x4 ya = __builtin_convertvector(a, r_bf16x4), yb = __builtin_convertvector(b, r_bf16x4);
                if (head < rot.nq) {
                    bf16_t* to = static_cast<bf16_t*>(out) + t * width + col;
                    *reinterpret_cast<r_bf16x4*>(to) = ya;
                    *reinterpret_cast<r_bf16x4*>(to + rot.half) = yb;
                    continue;
                }
                const int slot = rot.slots[t];
                if (slot < 0) continue;
                const size_t page = slot / rot.page_size, off = slot % rot.page_size, kh = is_v ? head - rot.nq - rot.nkv : head - rot.nq;
                if (!is_v) {             // keys: [page][kv head][offset][feature]
                    bf16_t* to = rot.k_cache + ((page * rot.nkv + kh) * rot.page_size + off) * (2 * rot.half) + at;
                    *reinterpret_cast<r_bf16x4*>(to) = ya;
                    *reinterpret_cast<r_bf16x4*>(to + rot.half) = yb;
                } else {                 // values: [page][kv head][feature][offset]
                    bf16_t* to = rot.v_cache + ((page * rot.nkv + kh) * (2 * rot.half) + at) * rot.page_size + off;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        *reinterpret_cast<__bf16*>(to + static_cast<size_t>(e) * rot.page_size) = ya[e];
                        *reinterpret_cast<__bf16*>(to + static_cast<size_t>(e + rot.half) * rot.page_size) = yb[e];
                    }
                }
            }
        }
    };
    auto store = [&]() {
        if constexpr (OUT == kRowsRotated) {
            store_rotated();
            return;
        }
        if (OUT == kRowsGated && act != kGateSilu) store_as(std::integral_constant<int, kGateGeluTanh>());
        else store_as(std::integral_constant<int, kGateSilu>());
    };
    Source fx = source_x(now), fw = source_w(now);
    const Item none = item_of(items);
    // (the order in which the loop would have asked)
#pragma unroll
    for (int i = -WB; i < 0; ++i) {
        if (i + XB >= 0) {
            if (fx.left == 0) fx = source_x(none);
            load_x(i + XB, fx);
        }
        if (fw.left == 0) fw = source_w(none);
        load_w(i + WB, fw);
    }
    // (where there is a next item, this one has WB steps at least)
    Item next = item_of(index + gridDim.x);
    clear();
    arrived<kBehind + XL + WL>();
    __syncthreads();
    read(0, 0, 0);
    // xb, wb: the buffers of the step
    int xb = 0, wb = 0, left = now.end - now.begin;
    auto step = [&]() {
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        load_x(xb, fx);
        load_w(wb, fw);
        xb = XB == 2 ? xb ^ 1 : xb + 1 == XB ? 0 : xb + 1;
        wb = wb + 1 == WB ? 0 : wb + 1;
        read(xb, wb, 0);
        multiply(1);
        --left;
    };
    bool stored = false;
#pragma unroll 1
    for (;;) {
        // an item's first step and its last WB ones, under which the loads of the workgroup's next item begin
        read(xb, wb, 1);
        multiply(0);
        if (stored) arrived<(kBehind + kStores < 63 ? kBehind + kStores : 63)>();
        else arrived<kBehind>();
        stored = false;
        if (fx.left == 0) fx = source_x(next);
        if (fw.left == 0) fw = source_w(next);
        step();
        // those between, a line of their own without branches (a branch in every step: 1.4 us a step of 256 x 256 against 1.2)
#pragma unroll 1
        while (left > WB) {
            read(xb, wb, 1);
            multiply(0);
            arrived<kBehind>();
            step();
        }
        if (left > 0) continue;
        store();
        if (next.rows == 0) break;
        clear();
        stored = OUT != kRowsRotated;                     // (which makes as many stores as its rows ask for)
        index += gridDim.x;
        now = next;
        next = item_of(index + gridDim.x);
        left = now.end - now.begin;
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);                      // (nothing is on its way to LDS when the workgroup ends)
#endif
}

template <int BM, int BN, int WM, int WN, int XB, int WB>
int launch_rows(const void* x, const void* w, void* out, int m, int n, int k, int splits, int per, int kind, int act, hipStream_t s) {
    const long mt = (m + BM - 1) / BM, nt = kind == kRowsGated ? (n + BN / 2 - 1) / (BN / 2) : (n + BN - 1) / BN;
    if (mt * nt * splits > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    // as many workgroups as the CUs hold, each taking its items in turn, where every item has the WB steps that are on
    // their way when it begins; else a workgroup per item
    constexpr int kHeld = kLdsOfCu / ((XB * BM + WB * BN) * 128);
    const int last_steps = k / kRowsStep - (splits - 1) * per;
    const long held = per >= WB && last_steps >= WB ? 256L * kHeld : mt * nt * splits;
    const dim3 grid(static_cast<unsigned>(mt * nt * splits < held ? mt * nt * splits : held));
    const auto* xp = static_cast<const bf16_t*>(x);
    const auto* wp = static_cast<const bf16_t*>(w);
    const Groups none{nullptr, nullptr, 0};
    if (kind == kRowsGated) gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsGated, false><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, m, n, k, splits, per, act, none, {});
    else if (kind == kRowsF32) gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsF32, false><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, m, n, k, splits, per, act, none, {});
    else gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsBf16, false><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, m, n, k, splits, per, act, none, {});
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

template <int BM, int BN, int WM, int WN, int XB, int WB>
int launch_rotated(const void* x, const void* w, void* out, int m, int pairs, int k, const RotatedOut& rot, hipStream_t s) {
    constexpr int BC = BN / 2;
    if (BC % rot.half != 0 && rot.half % BC != 0) return EGPT_UNSUPPORTED_SIZE;
    const long items = static_cast<long>((m + BM - 1) / BM) * ((pairs + BC - 1) / BC);
    if (items > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    constexpr int kHeld = kLdsOfCu / ((XB * BM + WB * BN) * 128);
    const int steps = k / kRowsStep;
    const long held = steps >= WB ? 256L * kHeld : items;
    gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsRotated, false><<<static_cast<unsigned>(items < held ? items : held), WM * WN * 64, 0, s>>>(
        static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), out, m, pairs, k, 1, steps, 0, Groups{nullptr, nullptr, 0}, rot);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

template <int BM, int BN, int WM, int WN, int XB, int WB>
int launch_groups(const void* x, const void* w, void* out, const Groups& g, long tiles, int n, int k, int kind, int act, hipStream_t s) {
    const long nt = kind == kRowsGated ? (n + BN / 2 - 1) / (BN / 2) : (n + BN - 1) / BN;
    if (tiles * nt > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    const unsigned grid = static_cast<unsigned>(tiles * nt);
    const auto* xp = static_cast<const bf16_t*>(x);
    const auto* wp = static_cast<const bf16_t*>(w);
    const int per = k / kRowsStep;
    if (kind == kRowsGated) gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsGated, true><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, 0, n, k, 1, per, act, g, {});
    else if (kind == kRowsF32) gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsF32, true><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, 0, n, k, 1, per, act, g, {});
    else gemm_rows_kernel<BM, BN, WM, WN, XB, WB, kRowsRelu2, true><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, 0, n, k, 1, per, act, g, {});
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

}  // namespace egpt

using namespace egpt;

extern "C" int egpt_gemm_rows(const void* x, const void* w, void* out, int m, int n, int k, int splits, int kind, int act,
                              int shape, void* stream) {
    if (!x || !w || !out || m < 0 || n <= 0 || k <= 0 || splits < 1 || kind < 0 || kind > kRowsGated || act < 0 || act > 1) return EGPT_BAD_ARGUMENT;
    if (k % kRowsStep != 0 || n % 4 != 0 || (splits != 1 && kind != kRowsF32)) return EGPT_UNSUPPORTED_SIZE;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16) return EGPT_UNSUPPORTED_SIZE;
    // a lane's byte offsets from its tile's first row are 32-bit numbers, in the operands and in the result
    if (static_cast<long long>(k) * 2 * (kind != kRowsGated ? 256 : n > 256 ? 2LL * n : n + 256LL) > 0x7fffffffLL || n > 0x1fffff) return EGPT_UNSUPPORTED_SIZE;
    if (m == 0) return EGPT_OK;
    const int total = k / kRowsStep, per = (total + splits - 1) / splits;
    if (splits > total || (splits - 1) * per >= total) return EGPT_BAD_ARGUMENT;      // an empty range
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the tiles that `_rows_shapes` in kernels/hip.py chooses from
    switch (shape) {
        case 0: return launch_rows<256, 256, 2, 4, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 1: return launch_rows<192, 256, 2, 4, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 2: return launch_rows<128, 256, 2, 4, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 3: return launch_rows<128, 128, 2, 2, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 4: return launch_rows<64, 64, 2, 2, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 5: return launch_rows<64, 64, 2, 2, 5, 5>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 6: return launch_rows<64, 128, 2, 2, 6, 6>(x, w, out, m, n, k, splits, per, kind, act, s);
        default: return EGPT_BAD_ARGUMENT;
    }
}

extern "C" int egpt_gemm_rows_rotated(const void* x, const void* w, const void* bias, const float* cos_sin, const int32_t* slots, void* out,
                                      void* k_cache, void* v_cache, int m, int k, int nq, int nkv, int hd, int page_size, int shape,
                                      void* stream) {
    if (!x || !w || !cos_sin || !slots || !out || !k_cache || !v_cache || m < 0 || k <= 0 || nq <= 0 || nkv <= 0 || hd <= 0 || page_size <= 0) return EGPT_BAD_ARGUMENT;
    const long long width = (static_cast<long long>(nq) + 2LL * nkv) * hd;
    // (heads of 32 to 256 columns: a tile is whole heads or a power of two of a head's pairs)
    if (k % kRowsStep != 0 || hd < 32 || hd > 256 || (hd & (hd - 1)) != 0 || width > 0x1fffff) return EGPT_UNSUPPORTED_SIZE;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(bias) |
         reinterpret_cast<uintptr_t>(cos_sin) | reinterpret_cast<uintptr_t>(k_cache)) % 16)
        return EGPT_UNSUPPORTED_SIZE;
    // a lane's byte offsets from its tile's first row are 32-bit numbers
    if (static_cast<long long>(k) * 2 * 512 > 0x7fffffffLL || width * k * 2 > 0x7fffffffLL) return EGPT_UNSUPPORTED_SIZE;
    if (m == 0) return EGPT_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const RotatedOut rot{static_cast<const bf16_t*>(bias), cos_sin, slots, static_cast<bf16_t*>(k_cache), static_cast<bf16_t*>(v_cache), nq, nkv, hd / 2, page_size};
    const int pairs = static_cast<int>(width / 2);
    switch (shape) {
        case 0: return launch_rotated<256, 256, 2, 4, 2, 3>(x, w, out, m, pairs, k, rot, s);
        case 1: return launch_rotated<192, 256, 2, 4, 2, 3>(x, w, out, m, pairs, k, rot, s);
        case 2: return launch_rotated<128, 256, 2, 4, 2, 3>(x, w, out, m, pairs, k, rot, s);
        case 3: return launch_rotated<128, 128, 2, 2, 2, 3>(x, w, out, m, pairs, k, rot, s);
        case 4: return launch_rotated<64, 64, 2, 2, 2, 3>(x, w, out, m, pairs, k, rot, s);
        case 5: return launch_rotated<64, 64, 2, 2, 5, 5>(x, w, out, m, pairs, k, rot, s);
        case 6: return launch_rotated<64, 128, 2, 2, 6, 6>(x, w, out, m, pairs, k, rot, s);
        default: return EGPT_BAD_ARGUMENT;
    }
}

extern "C" int egpt_moe_rows(const void* x, const void* w, const int32_t* row_token, const int32_t* tiles, void* out, int n_rows,
                             int x_rows, int n, int k, int experts, int tile_rows, int kind, int act, void* stream) {
    if (!x || !w || !tiles || !out || n_rows < 0 || x_rows < 0 || n <= 0 || k <= 0 || experts <= 0 || (!row_token && x_rows != n_rows) ||
        kind < kRowsF32 || kind > kRowsRelu2 || act < 0 || act > 1)
        return EGPT_BAD_ARGUMENT;
    if (k % kRowsStep != 0 || n % 4 != 0) return EGPT_UNSUPPORTED_SIZE;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16) return EGPT_UNSUPPORTED_SIZE;
    // byte offsets within x (gathered rows) and within an expert's matrix are 32-bit numbers
    if (static_cast<long long>(k) * 2 * (x_rows > 128 ? x_rows : 128) > 0x7fffffffLL || static_cast<long long>(k) * 2 * (n > 128 ? 2LL * n : n + 128LL) > 0x7fffffffLL || n > 0x3fffff) return EGPT_UNSUPPORTED_SIZE;
    if (n_rows == 0) return EGPT_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Groups g{tiles, row_token, x_rows};
    const long most = tile_rows > 0 ? n_rows / tile_rows + experts + 1 : 0;
    switch (tile_rows) {
        case 64: return launch_groups<64, 64, 2, 2, 2, 3>(x, w, out, g, most, n, k, kind, act, s);
        case 128: return launch_groups<128, 128, 2, 2, 2, 3>(x, w, out, g, most, n, k, kind, act, s);
        default: return EGPT_BAD_ARGUMENT;
    }
}
