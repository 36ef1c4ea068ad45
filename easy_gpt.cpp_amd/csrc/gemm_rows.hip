// out[m, n] = sum_k x[m, k] * w[n, k] in bfloat16 for many rows of x (more than 64): tiles staged through LDS by loads that
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
// What bounds it: alone, the loop runs at 1.9 PFLOP/s on zeros and 1.6 on random numbers (the card then lowers its clock).
// The weights come from memory, and all workgroups that share a tile of w ask for it at the same time, so nobody finds it in
// the L2 and everybody waits for memory's latency: with one step of both operands on its way, 2,048 x 37,888 x 3,584 took
// 486 us; with two of w and one of x (160 KB of LDS) 461, and on zeros 470 against 393.  Deeper rings in steps of 32 values
// (64-byte pieces of rows) gained nothing: 509.  32x32x16 products: the same on zeros, 7 % slower on random numbers.  The
// order of tiles: a die gets neighbouring tiles of one range of k (2,048 x 3,584 x 18,944 in two ranges: 247 -> 238 us).
// Against the library's first choice (us, weights from memory; gated ones with its activation kernel, others with the norm that
// reads the result): 2,048 rows x 18,944 gated x 3,584 456 against 547, 8,191 x 8,960 gated x 1,536 436 against 446; 2,048 x 3,584 x
// 18,944 238 against 382, 552 x 1,536 x 8,960 33 against 43, 552 x 896 x 896 11.0 against 12.6; but 8,191 x 18,944 gated x 3,584
// 1,871 against 1,818 and 2,048 x 2,048 x 1,536 30 against 28.  `_own_rows` and `_own_gate` in kernels/hip.py draw the lines.
#include "api.h"
#include "common.h"

namespace egpt {

typedef __attribute__((ext_vector_type(8))) __bf16 r_bf16x8;
typedef __attribute__((ext_vector_type(4))) float r_f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned short r_u16x4;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kRowsStep = 64;                  // values of k per step: 128 bytes a row

// At most N of this wavefront's loads into LDS are still on their way, and its LDS reads are done; then all wavefronts meet.
// (The loads are written in assembly and have no result in registers; __syncthreads() alone does not wait for them.)
template <int N>
__device__ __forceinline__ void landed() {
    __builtin_amdgcn_s_waitcnt((N & 15) | 0x0f70 | (N >> 4) << 14);
    __syncthreads();
}

typedef __attribute__((ext_vector_type(4))) int r_i32x4;

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"        // (m0 is a reserved register; nothing else here uses it)
// 16 bytes a lane from `resource` at byte `offset` + `at` to LDS: `lds` (the same for the whole wavefront) + 16 x lane.
__device__ __forceinline__ void load_to_lds(r_i32x4 resource, int offset, int at, char* lds) {
    const unsigned to = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_void*)lds));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(offset), "s"(resource), "s"(at)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ r_i32x4 buffer_of(const void* p, size_t bytes) {
    const uint64_t at = reinterpret_cast<uint64_t>(p);
    return r_i32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(at)), __builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32) & 0xffff),
                   __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
}

enum RowsOut { kRowsBf16 = 0, kRowsF32 = 1, kRowsGated = 2, kRowsRelu2 = 3 };

// Products of rows grouped by expert (moe.hip makes the table of tiles): tile i has rows tiles[3 i + 2 ..] of one expert, the
// numbers of tiles[1 + 3 i ..] being the expert, the tile's first grouped row and its rows; w is [experts][rows of w][k].
struct Groups {
    const int32_t* tiles;          // null: one matrix for all rows
    const int32_t* row_token;      // the row of x that a grouped row reads (null: the grouped row itself)
    int x_rows;                    // rows of x
};

template <int BM, int BN, int WM, int WN, int WB, int OUT, bool GROUPED>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_rows_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k, int splits,
    int steps_per_split, int act, Groups groups) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = WM * WN;
    constexpr int TM = BM / WM / 16, TN = BN / WN / 16;        // 16 x 16 tiles of a wavefront
    constexpr int XL = BM / 8 / NW, WL = BN / 8 / NW;          // loads of a wavefront per step: eight rows each
    static_assert(XL * 8 * NW == BM && WL * 8 * NW == BN, "a step is whole loads");
    constexpr int kXBytes = BM * 128, kWBytes = BN * 128;
    __shared__ __attribute__((aligned(128))) char xs[2 * kXBytes];
    __shared__ __attribute__((aligned(128))) char ws[WB * kWBytes];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int li = lane % 16, lg = lane / 16;
    const int wm = wave / WN, wn = wave % WN;

    // workgroups are handed to the eight dies in turn: a die gets a contiguous range of tiles, rows of x fastest, so that
    // its L2 holds the few rows of w and x that its tiles share
    constexpr int BC = OUT == kRowsGated ? BN / 2 : BN;         // columns of the result in a tile
    const int mt = GROUPED ? groups.tiles[0] : (m + BM - 1) / BM, nt = (n + BC - 1) / BC;
    const int tiles = mt * nt, items = tiles * splits;
    int item = blockIdx.x;
    if (GROUPED && item >= items) return;                      // (the grid is sized for the most tiles that the rows can make)
    {
        const int q = items / 8, r = items % 8, d = item % 8, i = item / 8;
        item = d * q + (d < r ? d : r) + i;
    }
    const int tile = item % tiles, split = item / tiles;
    int m0 = tile % mt * BM, n0 = tile / mt * BC, rows = min(m - m0, BM);
    if (GROUPED) {
        // all columns of a tile of rows after each other: an expert's matrix stays in the die's L2 for its tiles
        const int32_t* entry = groups.tiles + 1 + 3 * (item / nt);
        m0 = entry[1];
        n0 = item % nt * BC;
        rows = entry[2];
        w += static_cast<size_t>(entry[0]) * (OUT == kRowsGated ? 2 * n : n) * k;
    }
    const int total = k / kRowsStep;
    const int s_begin = split * steps_per_split, s_end = min(total, s_begin + steps_per_split);

    // ---- loads: a lane's byte offsets from the tile's first rows (rows beyond the last repeat the last)
    const int piece = (lane % 8) ^ (lane / 8);
    const size_t row_bytes = static_cast<size_t>(k) * 2;
    const bool gather = GROUPED && groups.row_token != nullptr;
    const r_i32x4 xr = gather ? buffer_of(x, groups.x_rows * row_bytes) : buffer_of(x + static_cast<size_t>(m0) * k, rows * row_bytes);
    const r_i32x4 wr = buffer_of(w + static_cast<size_t>(n0) * k, (OUT == kRowsGated ? 2 * n - n0 : min(n - n0, BN)) * row_bytes);
    int xo[XL], wo[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int r = (wave * XL + i) * 8 + lane / 8;
        int g = min(r, rows - 1);
        if (gather) g = groups.row_token[m0 + g];
        xo[i] = g * static_cast<int>(row_bytes) + piece * 16;
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int r = (wave * WL + i) * 8 + lane / 8;
        int g = min(r, n - n0 - 1);
        if (OUT == kRowsGated) {
            // a wavefront's columns: the first half of them gates, the second half the up columns of the same numbers
            constexpr int C = BN / WN;
            const int col = r / C * (C / 2) + r % (C / 2);
            g = min(col, n - n0 - 1) + (r % C >= C / 2 ? n : 0);
        }
        wo[i] = g * static_cast<int>(row_bytes) + piece * 16;
    }
    const int last = s_end - 1;                              // (beyond the last step the last one again, which nobody reads)
    auto load_x = [&](int buffer, int step) {
        const int at = min(step, last) * (kRowsStep * 2);
#pragma unroll
        for (int i = 0; i < XL; ++i) load_to_lds(xr, xo[i], at, xs + buffer * kXBytes + (wave * XL + i) * 1024);
    };
    auto load_w = [&](int buffer, int step) {
        const int at = min(step, last) * (kRowsStep * 2);
#pragma unroll
        for (int i = 0; i < WL; ++i) load_to_lds(wr, wo[i], at, ws + buffer * kWBytes + (wave * WL + i) * 1024);
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
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = r_f32x4{0.f, 0.f, 0.f, 0.f};
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
    load_x(0, s_begin);
    load_w(0, s_begin);
    load_x(1, s_begin + 1);
#pragma unroll
    for (int i = 1; i < WB; ++i) load_w(i, s_begin + i);
    landed<0>();
    read(0, 0, 0);
    int xb = 0, wb = 0;
#pragma unroll 1
    for (int s = s_begin; s < s_end; ++s) {
        const int xn = xb ^ 1, wnext = wb + 1 == WB ? 0 : wb + 1;
        read(xb, wb, 1);
        multiply(0);
        landed<(WB - 2) * WL>();
        __builtin_amdgcn_sched_barrier(0);
        load_x(xb, s + 2);
        load_w(wb, s + WB);
        read(xn, wnext, 0);
        multiply(1);
        xb = xn;
        wb = wnext;
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);                      // (nothing is on its way to LDS when the workgroup ends)
    // ---- a lane holds columns 4 lg .. 4 lg + 3 of row li of every 16 x 16 tile (n is a multiple of four)
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int at = wm * (BM / WM) + i * 16 + li, row = m0 + at;
        if (at >= rows) continue;
        if constexpr (OUT == kRowsGated) {
#pragma unroll
            for (int j = 0; j < TN / 2; ++j) {
                const int col = n0 + wn * (BN / WN / 2) + j * 16 + lg * 4;
                bf16_t* o = static_cast<bf16_t*>(out) + static_cast<size_t>(row) * n + col;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gate_activation(acc[i][j][e], act) * acc[i][j + TN / 2][e];
                if (col < n)
                    *reinterpret_cast<r_u16x4*>(o) = r_u16x4{f32_to_bf16_bits(v[0]), f32_to_bf16_bits(v[1]), f32_to_bf16_bits(v[2]), f32_to_bf16_bits(v[3])};
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = n0 + wn * (BN / WN) + j * 16 + lg * 4;
                if constexpr (OUT == kRowsF32) {
                    float* o = static_cast<float*>(out) + (static_cast<size_t>(split) * m + row) * n + col;
                    if (col < n) *reinterpret_cast<r_f32x4*>(o) = acc[i][j];
                } else {
                    bf16_t* o = static_cast<bf16_t*>(out) + static_cast<size_t>(row) * n + col;
                    r_f32x4 v = acc[i][j];
                    if constexpr (OUT == kRowsRelu2)
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = fmaxf(v[e], 0.f) * fmaxf(v[e], 0.f);
                    if (col < n)
                        *reinterpret_cast<r_u16x4*>(o) = r_u16x4{f32_to_bf16_bits(v[0]), f32_to_bf16_bits(v[1]), f32_to_bf16_bits(v[2]), f32_to_bf16_bits(v[3])};
                }
            }
        }
    }
#endif
}

template <int BM, int BN, int WM, int WN, int WB>
int launch_rows(const void* x, const void* w, void* out, int m, int n, int k, int splits, int per, int kind, int act, hipStream_t s) {
    const long mt = (m + BM - 1) / BM, nt = kind == kRowsGated ? (n + BN / 2 - 1) / (BN / 2) : (n + BN - 1) / BN;
    if (mt * nt * splits > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    const dim3 grid(static_cast<unsigned>(mt * nt * splits));
    const auto* xp = static_cast<const bf16_t*>(x);
    const auto* wp = static_cast<const bf16_t*>(w);
    const Groups none{nullptr, nullptr, 0};
    if (kind == kRowsGated) gemm_rows_kernel<BM, BN, WM, WN, WB, kRowsGated, false><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, m, n, k, splits, per, act, none);
    else if (kind == kRowsF32) gemm_rows_kernel<BM, BN, WM, WN, WB, kRowsF32, false><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, m, n, k, splits, per, act, none);
    else gemm_rows_kernel<BM, BN, WM, WN, WB, kRowsBf16, false><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, m, n, k, splits, per, act, none);
    EGPT_CHECK_LAUNCH();
    return EGPT_OK;
}

template <int BM, int BN, int WM, int WN, int WB>
int launch_groups(const void* x, const void* w, void* out, const Groups& g, long tiles, int n, int k, int kind, int act, hipStream_t s) {
    const long nt = kind == kRowsGated ? (n + BN / 2 - 1) / (BN / 2) : (n + BN - 1) / BN;
    if (tiles * nt > 0x7fffffffL) return EGPT_UNSUPPORTED_SIZE;
    const unsigned grid = static_cast<unsigned>(tiles * nt);
    const auto* xp = static_cast<const bf16_t*>(x);
    const auto* wp = static_cast<const bf16_t*>(w);
    const int per = k / kRowsStep;
    if (kind == kRowsGated) gemm_rows_kernel<BM, BN, WM, WN, WB, kRowsGated, true><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, 0, n, k, 1, per, act, g);
    else if (kind == kRowsF32) gemm_rows_kernel<BM, BN, WM, WN, WB, kRowsF32, true><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, 0, n, k, 1, per, act, g);
    else gemm_rows_kernel<BM, BN, WM, WN, WB, kRowsRelu2, true><<<grid, WM * WN * 64, 0, s>>>(xp, wp, out, 0, n, k, 1, per, act, g);
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
    // a lane's byte offsets from its tile's first row are 32-bit numbers
    if (static_cast<long long>(k) * 2 * (kind == kRowsGated ? 2LL * n : 256) > 0x7fffffffLL) return EGPT_UNSUPPORTED_SIZE;
    if (m == 0) return EGPT_OK;
    const int total = k / kRowsStep, per = (total + splits - 1) / splits;
    if (splits > total || (splits - 1) * per >= total) return EGPT_BAD_ARGUMENT;      // an empty range
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the tiles that `_rows_shapes` in kernels/hip.py chooses from
    switch (shape) {
        case 0: return launch_rows<256, 256, 2, 4, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 1: return launch_rows<192, 256, 2, 4, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 2: return launch_rows<128, 256, 2, 4, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 3: return launch_rows<128, 128, 2, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
        case 4: return launch_rows<64, 64, 2, 2, 3>(x, w, out, m, n, k, splits, per, kind, act, s);
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
    if (static_cast<long long>(k) * 2 * x_rows > 0x7fffffffLL || static_cast<long long>(k) * 2 * 2 * n > 0x7fffffffLL) return EGPT_UNSUPPORTED_SIZE;
    if (n_rows == 0) return EGPT_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Groups g{tiles, row_token, x_rows};
    const long most = tile_rows > 0 ? n_rows / tile_rows + experts + 1 : 0;
    switch (tile_rows) {
        case 64: return launch_groups<64, 64, 2, 2, 3>(x, w, out, g, most, n, k, kind, act, s);
        case 128: return launch_groups<128, 128, 2, 2, 3>(x, w, out, g, most, n, k, kind, act, s);
        default: return EGPT_BAD_ARGUMENT;
    }
}
