// Shared device helpers for the gfx950 kernels: element types, conversions, reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace egpt {

constexpr int kWave = 64;  // CDNA wavefront width

// bfloat16 as raw bits; arithmetic is always done in float.
struct bf16_t {
    uint16_t bits;
};

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16_t v) { return __uint_as_float(static_cast<uint32_t>(v.bits) << 16); }

// round to nearest even; NaN stays NaN
// (v_cvt_pk_bf16_f32: one instruction for two values in the place of some fourteen; the same bits as rounding half to even on the
// integer, NaN made quiet: tests/test_gpu_rounding.py has every upper half with lower halves around the tie, subnormals among them)
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }
__device__ __forceinline__ uint32_t bf16_pair(float low, float high) {
    typedef __attribute__((ext_vector_type(2))) float two;
    typedef __attribute__((ext_vector_type(2))) __bf16 two_bf16;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((two{low, high}), two_bf16));
}

template <typename T>
__device__ __forceinline__ T from_float(float v);
template <>
__device__ __forceinline__ float from_float<float>(float v) { return v; }
template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float v) { return bf16_t{f32_to_bf16_bits(v)}; }

// The QKV epilogue's arithmetic, spelled out operation by operation: several kernels do it (one by one, four
// pairs at a time, inside the decode attention) and must leave the same bits, which they would not if the
// compiler were free to contract each one's multiplications and additions in its own way.
__device__ __forceinline__ float scale_then_bias(float x, float scale, float bias) { return __fmaf_rn(x, scale, bias); }
__device__ __forceinline__ float inv_rms(float ss, float inv_hidden, float eps) {
    return 1.0f / sqrtf(__fmaf_rn(ss, inv_hidden, eps));
}
__device__ __forceinline__ void rotate_pair(float a, float b, float c, float s, float& ra, float& rb) {
    ra = __fmaf_rn(a, c, -__fmul_rn(b, s));
    rb = __fmaf_rn(a, s, __fmul_rn(b, c));
}

// The activation of a gated feed-forward's gate: 0 silu, z / (1 + exp(-z)); 1 the tanh form of gelu,
// z / 2 (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3))), which is z / (1 + exp(-2 sqrt(2 / pi) (z + 0.044715 z^3))).
constexpr int kGateSilu = 0, kGateGeluTanh = 1;
constexpr int kUngatedRelu2 = 2;         // no gate: the square of relu (where a product can begin with either)
__device__ __forceinline__ float gate_exponent(float z, int act) {
    return act == kGateSilu ? z : 1.5957691216057308f * fmaf(0.044715f * z * z, z, z);
}
__device__ __forceinline__ float gate_activation(float z, int act) { return z / (1.0f + expf(-gate_exponent(z, act))); }

// The residual stream of steps of few tokens in 64-bit fixed point (units of 2^-32).  Several workgroups that split
// a product's k range add their partial results straight into it with integer atomics: integer addition does not
// care for the order, so the sum is the same bits whatever the scheduling, and the kernels that read the stream
// read one small tensor instead of every workgroup's partial sums.  A float32 value times 2^32 is an integer for
// every magnitude of 2^-8 and above and is rounded to one below (an absolute error of at most 2^-33, whatever the
// other values of the stream are); the stream holds magnitudes below 2^31.  What does not fit is not hidden as
// a small number: a magnitude of 2^31 or more, an infinity or a NaN enters as the largest magnitude of its sign
// (NaN: the negative one), which the norm behind it turns into a row of zeros and one entry of +-sqrt(width) - a
// step of more than 16 rows, and the float32 path, keep such values in float32 and show them as they are.
typedef long long fixed_t;
constexpr float kFixedOne = 4294967296.0f;
constexpr float kFixedLimit = 2147483648.0f;          // 2^31
__device__ __forceinline__ fixed_t to_fixed(float v) {
    if (!(fabsf(v) < kFixedLimit)) return v > 0.f ? 0x7fffffffffffffffLL : -0x7fffffffffffffffLL - 1;
    return __float2ll_rn(v * kFixedOne);
}
__device__ __forceinline__ float fixed_to_float(fixed_t v) { return __ll2float_rn(v) * (1.0f / kFixedOne); }
__device__ __forceinline__ void fixed_add(fixed_t* p, float v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(p), static_cast<unsigned long long>(to_fixed(v)));
}
// what a residual stream of either kind is read and written as
__device__ __forceinline__ float residual_load(const float* p) { return *p; }
__device__ __forceinline__ float residual_load(const fixed_t* p) { return fixed_to_float(*p); }
__device__ __forceinline__ void residual_store(float* p, float v) { *p = v; }
__device__ __forceinline__ void residual_store(fixed_t* p, float v) { *p = to_fixed(v); }

// The output of a product arrives either as one tensor of the activation type, or as float32 partial
// sums [n_splits][rows][cols] of a split-k product, which are added here in split order.
template <typename T>
struct ProductView {
    const T* whole;          // used when n_splits == 0
    const float* partial;    // used when n_splits > 0
    int n_splits;
    size_t split_stride;     // rows * cols
    __device__ __forceinline__ bool present() const { return whole != nullptr || partial != nullptr; }
    __device__ __forceinline__ float at(size_t idx) const {
        if (n_splits == 0) return to_float(whole[idx]);
        if (n_splits == 1) return partial[idx];          // a product written out in float32: one load, not a round of sixteen
        // up to sixteen loads in flight at a time (a chain of dependent kernels pays for round trips, not
        // bytes); the order of the additions is fixed
        float v = 0.f;
        for (int s0 = 0; s0 < n_splits; s0 += 16) {
            float t[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) t[i] = s0 + i < n_splits ? partial[(s0 + i) * split_stride + idx] : 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) v += t[i];
        }
        return v;
    }
};

// N values of a product.  All their loads are on their way together, of up to 16 / N partial sums at a time: N calls of at()
// are N round trips one after the other, since what form the product has is found out anew in each.  (2,535 rows of 896
// values, us: a norm over one float32 array and the residual stream 15.5 with at(), 11.5 with this; a gated norm of seven
// heads of 128 from four partial sums 25.0 and 13.3.)  The order of the additions is that of at().  A thread whose place lies
// behind the end names any other.
template <int N, typename T>
__device__ __forceinline__ void read_values(const ProductView<T>& p, const size_t (&at)[N], float (&v)[N]) {
    if (p.n_splits == 0) {
        T raw[N];
#pragma unroll
        for (int i = 0; i < N; ++i) raw[i] = p.whole[at[i]];
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = to_float(raw[i]);
        return;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = p.partial[at[i]];
    constexpr int U = N < 16 ? 16 / N : 1;
    for (int s0 = 1; s0 < p.n_splits; s0 += U) {
        float t[U][N];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u < p.n_splits) {
#pragma unroll
                for (int i = 0; i < N; ++i) t[u][i] = p.partial[(s0 + u) * p.split_stride + at[i]];
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u < p.n_splits) {
#pragma unroll
                for (int i = 0; i < N; ++i) v[i] += t[u][i];
            }
    }
}

// Four neighbouring values: kernels whose time is their instructions read and write a row by quads, with one index and one test for
// four values.  A quad begins on a multiple of four values of an operand that itself begins on 16 bytes (`quads`, on the host).
__device__ __forceinline__ void read_quad(const float* p, float (&v)[4]) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void read_quad(const bf16_t* p, float (&v)[4]) {
    const uint2 a = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
    v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
}
__device__ __forceinline__ void write_quad(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = float4{v[0], v[1], v[2], v[3]}; }
__device__ __forceinline__ void write_quad(bf16_t* p, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(p) = uint2{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3])};
}
// (and pairs and single values by the same names)
__device__ __forceinline__ void read_quad(const float* p, float (&v)[2]) {
    const float2 a = *reinterpret_cast<const float2*>(p);
    v[0] = a.x; v[1] = a.y;
}
__device__ __forceinline__ void read_quad(const bf16_t* p, float (&v)[2]) {
    const uint32_t a = *reinterpret_cast<const uint32_t*>(p);
    v[0] = __uint_as_float(a << 16); v[1] = __uint_as_float(a & 0xffff0000u);
}
template <typename T>
__device__ __forceinline__ void read_quad(const T* p, float (&v)[1]) { v[0] = to_float(p[0]); }
__device__ __forceinline__ void write_quad(float* p, const float (&v)[2]) { *reinterpret_cast<float2*>(p) = float2{v[0], v[1]}; }
__device__ __forceinline__ void write_quad(bf16_t* p, const float (&v)[2]) { *reinterpret_cast<uint32_t*>(p) = bf16_pair(v[0], v[1]); }
template <typename T>
__device__ __forceinline__ void write_quad(T* p, const float (&v)[1]) { p[0] = from_float<T>(v[0]); }
// of a product, partial sums added in the order of at(), the loads of up to three of them on their way together (and none in vain: one
// sum after the first is read once, not three times)
template <int N, int E>
__device__ __forceinline__ void add_quads(const float* p, size_t stride, float (&v)[E]) {
    float t[N][E];
#pragma unroll
    for (int u = 0; u < N; ++u) read_quad(p + u * stride, t[u]);
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] += t[u][e];
}
template <typename T, int E>
__device__ __forceinline__ void read_quad(const ProductView<T>& p, size_t at, float (&v)[E]) {
    if (p.n_splits == 0) return read_quad(p.whole + at, v);
    const float* from = p.partial + at;
    read_quad(from, v);
    if (p.n_splits == 1) return;
    from += p.split_stride;
    int left = p.n_splits - 1;
    for (; left >= 3; left -= 3, from += 3 * p.split_stride) add_quads<3>(from, p.split_stride, v);
    if (left == 2) add_quads<2>(from, p.split_stride, v);
    if (left == 1) add_quads<1>(from, p.split_stride, v);
}
// Whether all of these begin on 16 bytes (null does).
template <typename... P>
static inline bool quads(const P*... p) { return ((reinterpret_cast<uintptr_t>(p) | ...) & 15) == 0; }
// Threads for a row of so many quads, a quad each.
static inline int quad_threads(int values) { return (values / 4 + kWave - 1) / kWave * kWave; }

// floor(x / d) for x and d < 2^27, as a product: no more than one too many, which is put right (a division is 30 instructions, and
// a kernel like this one is as long as its chain of them).
static unsigned magic_of(int d) { return static_cast<unsigned>((1ULL << 32) / (2 * static_cast<unsigned>(d)) + 1); }
__device__ __forceinline__ int divided(int x, int d, unsigned magic) {
    const int q = static_cast<int>(__umulhi(2 * static_cast<unsigned>(x), magic));
    return q - (q * d > x ? 1 : 0);
}

// A product whose x operand was (h * norm weight) still lacks each row's factor 1 / sqrt(sum_s ss[s][row] / hidden + eps):
// the sums of squares arrive beside it (null: the product is complete).
struct RowFactor {
    const float* ss;
    int splits, n_rows, hidden;
    float eps;
    __device__ __forceinline__ float of(int row) const {
        if (ss == nullptr) return 1.0f;
        float total = 0.f;
        for (int s = 0; s < splits; ++s) total += ss[static_cast<size_t>(s) * n_rows + row];
        return inv_rms(total, 1.0f / static_cast<float>(hidden), eps);
    }
};

// Reductions over a wavefront's lanes in registers: rotations and exchanges of rows of 16 lanes (DPP, v_permlane*_swap) are vector
// instructions, where a shuffle goes through LDS and its result is waited for.  (Decode steps of the 0.5B sizes, us: 64 users 1,359
// with shuffles and 1,336 so; one user's within what two runs differ by.)  The pairs that are added up, and so the bits, are those of shuffles with
// lanes 32, 16, 8, 4, 2, 1 apart (or 1, 2, 4, 8): behind a step the values repeat at its distance, so that a rotation by the next one
// reaches the partner's value.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
struct AddOf {
    __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct MaxOf {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
template <class Op>
__device__ __forceinline__ float fold_32_apart(float v, Op op) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <class Op>
__device__ __forceinline__ float fold_16_apart(float v, Op op) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <class Op>
__device__ __forceinline__ float fold_wave(float v, Op op) {
    v = fold_16_apart(fold_32_apart(v, op), op);
    v = op(v, dpp_move<0x128>(v));                        // row_ror:8, 4, 2, 1
    v = op(v, dpp_move<0x124>(v));
    v = op(v, dpp_move<0x122>(v));
    return op(v, dpp_move<0x121>(v));
}
// over the 16 lanes of a row, with lanes 1, 2, 4, 8 apart
template <class Op>
__device__ __forceinline__ float fold_row(float v, Op op) {
    v = op(v, dpp_move<0xb1>(v));                         // quad_perm 1 0 3 2, 2 3 0 1, row_half_mirror, row_mirror
    v = op(v, dpp_move<0x4e>(v));
    v = op(v, dpp_move<0x141>(v));
    return op(v, dpp_move<0x140>(v));
}
// over the four lanes with the same place in their rows, with lanes 16, 32 apart
template <class Op>
__device__ __forceinline__ float fold_rows(float v, Op op) { return fold_32_apart(fold_16_apart(v, op), op); }
__device__ __forceinline__ float wave_sum(float v) { return fold_wave(v, AddOf()); }
__device__ __forceinline__ float wave_max(float v) { return fold_wave(v, MaxOf()); }

// Which request's rows a workgroup has: the requests' blocks of rows lie one after the other, request s has blocks_of(q_len[s]) of
// them.  False: block `index` is nobody's.  64 requests at a time, by a sum over the lanes; one after the other they are a chain of
// loads (40 decoded tokens in front of the one portion of a step of the 1.5B sizes: 4,031 us a step, 3,933 so), which is only as good for a few.
template <class F>
__device__ __forceinline__ bool find_block(const int32_t* __restrict__ q_len, int n_seqs, int index, F blocks_of, int& seq, int& block) {
    if (n_seqs <= 4) {
        for (seq = 0, block = index; seq < n_seqs; ++seq) {
            const int n = blocks_of(q_len[seq]);
            if (block < n) return true;
            block -= n;
        }
        return false;
    }
    const int lane = threadIdx.x % kWave;
    for (int s0 = 0; s0 < n_seqs; s0 += kWave) {
        const int n = s0 + lane < n_seqs ? blocks_of(q_len[s0 + lane]) : 0;
        int upto = n;
        upto += __builtin_amdgcn_update_dpp(0, upto, 0x111, 0xf, 0xf, true);          // row_shr:1, 2, 4, 8: the sum within a row
        upto += __builtin_amdgcn_update_dpp(0, upto, 0x112, 0xf, 0xf, true);
        upto += __builtin_amdgcn_update_dpp(0, upto, 0x114, 0xf, 0xf, true);
        upto += __builtin_amdgcn_update_dpp(0, upto, 0x118, 0xf, 0xf, true);
        upto += __builtin_amdgcn_update_dpp(0, upto, 0x142, 0xa, 0xf, false);         // row_bcast:15 and 31: the rows before it
        upto += __builtin_amdgcn_update_dpp(0, upto, 0x143, 0xc, 0xf, false);
        const unsigned long long behind = __ballot(upto > index);
        if (behind != 0) {
            const int at = __builtin_ctzll(behind);
            seq = s0 + at;
            block = index - (__builtin_amdgcn_readlane(upto, at) - __builtin_amdgcn_readlane(n, at));
            return true;
        }
        index -= __builtin_amdgcn_readlane(upto, kWave - 1);
    }
    return false;
}

// Sum over a block of up to 1024 threads; every thread gets the result.  `scratch` holds >= 16 floats.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int n_waves = (blockDim.x + kWave - 1) / kWave;
    v = wave_sum(v);
    __syncthreads();  // scratch may still be read from an earlier call
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < n_waves; ++w) total += scratch[w];
    return total;
}
// The same of N values at once by `waves` wavefronts, 16 at most, with scratch of its own that nothing else uses: one wait.
template <int N>
__device__ __forceinline__ void block_totals(float (&v)[N], float (*scratch)[16], int waves) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[i] = wave_sum(v[i]);
        if (lane == 0) scratch[i][wave] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float part = scratch[i][lane % 16];
        v[i] = fold_row(lane % 16 < waves ? part : 0.f, AddOf());
    }
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int n_waves = (blockDim.x + kWave - 1) / kWave;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float m = scratch[0];
    for (int w = 1; w < n_waves; ++w) m = fmaxf(m, scratch[w]);
    return m;
}

}  // namespace egpt

// Error codes returned by every entry point (0 = launched).
#define EGPT_OK 0
#define EGPT_BAD_ARGUMENT 1
#define EGPT_UNSUPPORTED_SIZE 2
#define EGPT_LAUNCH_FAILED 3
#define EGPT_STATIC_SCRATCH_TOO_SMALL 4
#define EGPT_STATIC_SCRATCH_UNRESOLVED 5

#define EGPT_CHECK_LAUNCH()                                   \
    do {                                                      \
        hipError_t e_ = hipGetLastError();                    \
        if (e_ != hipSuccess) return EGPT_LAUNCH_FAILED;      \
    } while (0)
