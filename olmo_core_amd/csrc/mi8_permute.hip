// Token permutation for mixture-of-experts layers: the row copies that bracket the expert GEMMs.
//
//   gather          out[i]       = x[indices[i] / top_k] * w[indices[i]]            (rows sorted by expert)
//   scatter         out[t]       = sum_j round(x[inv[t*top_k + j]] * w[t*top_k + j]) (back to token order)
//   scatter_wgrad   out[indices[i]] = dot(x[i], grad[indices[i] / top_k])            (gradient of the weights)
//
// and their capacity-limited ("binned") forms, where expert e owns `capacity` rows and keeps at most that many
// of its tokens.  All of it is HBM-bound row traffic: one wave per row, 16-byte accesses, products in fp32 with
// one rounding to the element type.  The scatter never materialises the [tokens, top_k, hidden] intermediate of
// a copy-then-sum formulation: a small kernel inverts the permutation (inv[indices[i]] = i) and every output row
// is then reduced in registers, term by term in slot order.
//
// An index outside [0, tokens * top_k) is skipped (treated as a dropped token) rather than followed.
#include "mi8_common.h"

namespace mi8 {
namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / 64;
constexpr int64_t kMaxBlocks = 256 * 8;

// ---- element types --------------------------------------------------------------------------------------
template <int DT>
struct El;
template <>
struct El<MI8_BF16> {
    using T = uint16_t;
    __device__ static __forceinline__ float to_f32(T v) { return bits_to_f32((uint32_t)v << 16); }
    __device__ static __forceinline__ T from_f32(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
};
template <>
struct El<MI8_F16> {
    using T = uint16_t;
    __device__ static __forceinline__ float to_f32(T v) { return (float)__builtin_bit_cast(_Float16, v); }
    __device__ static __forceinline__ T from_f32(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
};
template <>
struct El<MI8_F32> {
    using T = uint32_t;
    __device__ static __forceinline__ float to_f32(T v) { return bits_to_f32(v); }
    __device__ static __forceinline__ T from_f32(float f) { return f32_to_bits(f); }
};
template <>
struct El<MI8_RAW8> {  // opaque bytes (fp8 rows): copied, never scaled
    using T = uint8_t;
    __device__ static __forceinline__ float to_f32(T v) { return (float)v; }
    __device__ static __forceinline__ T from_f32(float f) { return (T)f; }
};

__device__ __forceinline__ float load_weight(const void* w, int w_dtype, int64_t i)
{
    if (w_dtype == MI8_F32) return reinterpret_cast<const float*>(w)[i];
    const uint16_t v = reinterpret_cast<const uint16_t*>(w)[i];
    return w_dtype == MI8_BF16 ? El<MI8_BF16>::to_f32(v) : El<MI8_F16>::to_f32(v);
}

// A 16-byte chunk as N elements of type T
template <typename T>
union Chunk {
    uint4 raw;
    T e[16 / sizeof(T)];
};

// ---- one row: dst = round(src * w) (src == nullptr: zeros).  `vec`: rows are 16-byte aligned multiples of 16.
template <int DT, bool SCALE>
__device__ __forceinline__ void copy_row(const void* src, void* dst, int64_t hidden, float w, bool vec, int lane)
{
    using T = typename El<DT>::T;
    constexpr int N = 16 / sizeof(T);
    if (vec) {
        const int64_t chunks = hidden / N;
        const uint4* s = reinterpret_cast<const uint4*>(src);
        uint4* d = reinterpret_cast<uint4*>(dst);
        for (int64_t c = lane; c < chunks; c += 64 * 4) {
            Chunk<T> v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u].raw = (src && c + 64 * u < chunks) ? s[c + 64 * u] : make_uint4(0, 0, 0, 0);
            if (SCALE && src) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int k = 0; k < N; ++k) v[u].e[k] = El<DT>::from_f32(El<DT>::to_f32(v[u].e[k]) * w);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (c + 64 * u < chunks) d[c + 64 * u] = v[u].raw;
        }
    } else {
        const T* s = reinterpret_cast<const T*>(src);
        T* d = reinterpret_cast<T*>(dst);
        for (int64_t c = lane; c < hidden; c += 64) {
            T v = src ? s[c] : (T)0;
            if (SCALE && src) v = El<DT>::from_f32(El<DT>::to_f32(v) * w);
            d[c] = v;
        }
    }
}

struct PermuteArgs {
    const void* x;
    void* out;
    const int32_t* indices;  // [n]
    const void* weights;     // [n] or null
    int w_dtype;
    const int32_t* bins;     // binned forms: inclusive prefix sums of the tokens per expert, [experts]
    int32_t* inverse;        // scatter: [n]
    const void* grad;        // scatter_wgrad: [tokens, hidden]
    int64_t n;               // tokens * top_k
    int64_t hidden;
    int32_t top_k, experts, capacity;
    bool vec;
};

// Source slot of row r of the expert-sorted side: dropless r -> r; binned (e, j) -> bins[e-1] + j, or -1 when
// expert e has fewer than j + 1 tokens.  Returns the token-slot index (indices[...]) or -1.
template <bool BINNED>
__device__ __forceinline__ int64_t slot_of_row(const PermuteArgs& a, int64_t r)
{
    int64_t pos = r;
    if (BINNED) {
        const int e = (int)(r / a.capacity), j = (int)(r % a.capacity);
        const int start = e ? a.bins[e - 1] : 0;
        if (j >= a.bins[e] - start) return -1;
        pos = start + j;
    }
    if (pos >= a.n) return -1;
    const int64_t idx = a.indices[pos];
    return (idx < 0 || idx >= a.n) ? -1 : idx;
}

template <int DT, bool SCALE, bool BINNED>
__global__ __launch_bounds__(kThreads) void gather_kernel(PermuteArgs a, int64_t rows)
{
    const int lane = threadIdx.x & 63;
    using T = typename El<DT>::T;
    for (int64_t r = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6); r < rows;
         r += (int64_t)gridDim.x * kWavesPerBlock) {
        const int64_t idx = slot_of_row<BINNED>(a, r);
        const T* src = idx < 0 ? nullptr : reinterpret_cast<const T*>(a.x) + (idx / a.top_k) * a.hidden;
        const float w = (SCALE && idx >= 0) ? load_weight(a.weights, a.w_dtype, idx) : 1.0f;
        copy_row<DT, SCALE>(src, reinterpret_cast<T*>(a.out) + r * a.hidden, a.hidden, w, a.vec, lane);
    }
}

template <typename T>
__global__ void fill_kernel(T* p, int64_t n, T v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

template <bool BINNED>
__global__ void inverse_kernel(PermuteArgs a, int64_t rows)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int64_t idx = slot_of_row<BINNED>(a, r);
    if (idx >= 0) a.inverse[idx] = (int32_t)r;
}

// out[t] = sum over the token's top_k slots of round(x[inverse[slot]] * w[slot]); slots nobody filled add zero
template <int DT, bool SCALE>
__global__ __launch_bounds__(kThreads) void scatter_reduce_kernel(PermuteArgs a, int64_t tokens)
{
    using T = typename El<DT>::T;
    constexpr int N = 16 / sizeof(T);
    const int lane = threadIdx.x & 63;
    const T* x = reinterpret_cast<const T*>(a.x);
    const int k = a.top_k;
    for (int64_t t = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6); t < tokens;
         t += (int64_t)gridDim.x * kWavesPerBlock) {
    T* out = reinterpret_cast<T*>(a.out) + t * a.hidden;
    if (a.vec) {
        const int64_t chunks = a.hidden / N;
        // The token's rows and weights are fetched once, slot j by lane j, and handed round as wave-uniform values (top_k
        // up to 64; beyond, every term reads its own).  A lane then has four chunks of two rows in flight at a time: a
        // chain of one index load and one row load per term left the memory system idle most of the time.
        const bool held = k <= 64;
        int32_t my_r = -1;
        float my_w = 1.0f;
        if (held && lane < k) {
            my_r = a.inverse[t * k + lane];
            if (SCALE && my_r >= 0) my_w = load_weight(a.weights, a.w_dtype, t * k + lane);
        }
        auto term = [&](int j, int32_t& r, float& w) __attribute__((always_inline)) {
            if (held) {
                r = __builtin_amdgcn_readlane(my_r, j);
                w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_w), j));
            } else {
                r = a.inverse[t * k + j];
                w = (SCALE && r >= 0) ? load_weight(a.weights, a.w_dtype, t * k + j) : 1.0f;
            }
        };
        constexpr int U = 4;
        for (int64_t c0 = lane; c0 < chunks; c0 += 64 * U) {
            float acc[U][N];
            Chunk<T> first[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                first[u].raw = make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < N; ++e) acc[u][e] = 0.0f;
            }
            auto fetch = [&](int32_t r, Chunk<T> (&v)[U]) __attribute__((always_inline)) {
                const uint4* row = reinterpret_cast<const uint4*>(x + (int64_t)(r < 0 ? 0 : r) * a.hidden);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    v[u].raw = (r >= 0 && c0 + 64 * u < chunks) ? load_stream16(row + c0 + 64 * u) : make_uint4(0, 0, 0, 0);
            };
            auto add = [&](int32_t r, float w, Chunk<T> (&v)[U]) __attribute__((always_inline)) {
                if (r < 0) return;  // (uniform) an unfilled slot adds nothing, not even +0 to a -0
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (SCALE) {
#pragma unroll
                        for (int e = 0; e < N; ++e) v[u].e[e] = El<DT>::from_f32(El<DT>::to_f32(v[u].e[e]) * w);
                    }
                    if (k == 1) first[u] = v[u];
#pragma unroll
                    for (int e = 0; e < N; ++e) acc[u][e] += El<DT>::to_f32(v[u].e[e]);
                }
            };
            int j = 0;
            for (; j + 1 < k; j += 2) {  // two terms' rows in flight; added in slot order
                int32_t r0, r1;
                float w0, w1;
                term(j, r0, w0);
                term(j + 1, r1, w1);
                Chunk<T> v0[U], v1[U];
                fetch(r0, v0);
                fetch(r1, v1);
                add(r0, w0, v0);
                add(r1, w1, v1);
            }
            if (j < k) {
                int32_t r0;
                float w0;
                term(j, r0, w0);
                Chunk<T> v0[U];
                fetch(r0, v0);
                add(r0, w0, v0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (c0 + 64 * u >= chunks) continue;
                Chunk<T> o;
#pragma unroll
                for (int e = 0; e < N; ++e) o.e[e] = El<DT>::from_f32(acc[u][e]);
                reinterpret_cast<uint4*>(out)[c0 + 64 * u] = (k == 1) ? first[u].raw : o.raw;  // top_k 1 is a pure move (keeps -0)
            }
        }
    } else {
        for (int64_t c = lane; c < a.hidden; c += 64) {
            float acc = 0.0f;
            T first = 0;
            for (int j = 0; j < k; ++j) {
                const int64_t slot = t * k + j;
                const int32_t r = a.inverse[slot];
                if (r < 0) continue;
                T v = x[(int64_t)r * a.hidden + c];
                if (SCALE) v = El<DT>::from_f32(El<DT>::to_f32(v) * load_weight(a.weights, a.w_dtype, slot));
                if (k == 1) first = v;
                acc += El<DT>::to_f32(v);
            }
            out[c] = (k == 1) ? first : El<DT>::from_f32(acc);
        }
    }
    }
}

// The scatter of few slots in one launch.  A call with few tokens is a chain of short launches, and three of them - clearing the
// inverse, filling it, one wave a token - were its last 17 us (48 tokens of 8 slots, 2048 columns; now 6.4).  Here
// a workgroup finds the rows of its token among all slots itself, and its lanes have one 16-byte chunk of a row each, eight rows in
// flight.  Sums as above; a slot named twice takes the later row.
constexpr int64_t kFewSlots = 8192;
constexpr int kFewTopK = 64;

// So the slots are read as often as there are workgroups: up to 2^22 of them in all, 2^23 where half the lanes have no chunk to wait
// for.  us, this and the three launches, tokens x slots of a token x bf16 columns: 512 x 8 x 4096 (2^22) 13.5 / 21.1, 1024 x 4 x 2048 9.5 / 11.6, 2048 x 1 x
// 2048 10.9 / 13.1; 1024 x 8 x 2048 (2^23) 17.6 / 14.8, x 1024 9.7 / 13.3; 2048 x 2 x 2048 13.8 / 13.0, x 1024 10.5 / 11.2; 2048 x 4 x 1024 (2^24)
// 15.9 / 13.2, x 64 12.3 / 11.0; 8192 x 1 x 4096 (2^27) 101 / 59.
bool scatter_in_one_launch(const PermuteArgs& a, int64_t tokens, int64_t chunks)
{
    const int64_t columns = ceil_div(chunks, kThreads);
    return a.vec && a.n <= kFewSlots && a.top_k <= kFewTopK && columns <= 65535 && tokens * a.n * columns <= (chunks <= 128 ? 1 << 23 : 1 << 22);
}

template <int DT, bool SCALE>
__global__ __launch_bounds__(kThreads) void scatter_few_kernel(PermuteArgs a)
{
    using T = typename El<DT>::T;
    constexpr int N = 16 / sizeof(T);
    __shared__ int32_t row_of[kFewTopK];
    __shared__ float weight_of[kFewTopK];
    const int tid = threadIdx.x, k = a.top_k, n = (int)a.n;
    const int first = (int)blockIdx.x * k;
    if (tid < k) {
        row_of[tid] = -1;
        weight_of[tid] = SCALE ? load_weight(a.weights, a.w_dtype, first + tid) : 1.0f;
    }
    __syncthreads();
#pragma unroll 8
    for (int r = tid; r < n; r += kThreads) {
        const uint32_t j = (uint32_t)a.indices[r] - (uint32_t)first;
        if (j < (uint32_t)k) atomicMax(&row_of[j], r);
    }
    __syncthreads();
    const T* x = reinterpret_cast<const T*>(a.x);
    const int64_t c = (int64_t)blockIdx.y * kThreads + tid;
    if (c >= a.hidden / N) return;
    constexpr int U = 8;
    float acc[N];
    Chunk<T> first_term;
    first_term.raw = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < N; ++e) acc[e] = 0.0f;
    for (int j0 = 0; j0 < k; j0 += U) {
        Chunk<T> v[U];
        int32_t row[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            row[u] = j0 + u < k ? row_of[j0 + u] : -1;
            v[u].raw = make_uint4(0, 0, 0, 0);
            if (row[u] >= 0) v[u].raw = reinterpret_cast<const uint4*>(x + (int64_t)row[u] * a.hidden)[c];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (row[u] < 0) continue;  // (uniform) an unfilled slot adds nothing, not even +0 to a -0
            if (SCALE) {
                const float w = weight_of[j0 + u];
#pragma unroll
                for (int e = 0; e < N; ++e) v[u].e[e] = El<DT>::from_f32(El<DT>::to_f32(v[u].e[e]) * w);
            }
            if (k == 1) first_term = v[u];
#pragma unroll
            for (int e = 0; e < N; ++e) acc[e] += El<DT>::to_f32(v[u].e[e]);
        }
    }
    Chunk<T> o;
#pragma unroll
    for (int e = 0; e < N; ++e) o.e[e] = El<DT>::from_f32(acc[e]);
    reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.out) + (int64_t)blockIdx.x * a.hidden)[c] = k == 1 ? first_term.raw : o.raw;
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// out[slot] = dot(x[r], grad[slot / top_k]) for every filled row r of the expert-sorted side
template <int DT, bool BINNED>
__global__ __launch_bounds__(kThreads) void scatter_wgrad_kernel(PermuteArgs a, int64_t rows)
{
    using T = typename El<DT>::T;
    constexpr int N = 16 / sizeof(T);
    const int lane = threadIdx.x & 63;
    for (int64_t r = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6); r < rows;
         r += (int64_t)gridDim.x * kWavesPerBlock) {
    const int64_t idx = slot_of_row<BINNED>(a, r);
    if (idx < 0) continue;
    const T* x = reinterpret_cast<const T*>(a.x) + r * a.hidden;
    const T* g = reinterpret_cast<const T*>(a.grad) + (idx / a.top_k) * a.hidden;
    float acc = 0.0f;
    if (a.vec) {
        const int64_t chunks = a.hidden / N;
        constexpr int U = 4;  // chunks in flight per lane; summed in the order of a chunk-by-chunk loop
        for (int64_t c0 = lane; c0 < chunks; c0 += 64 * U) {
            Chunk<T> xv[U], gv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool ok = c0 + 64 * u < chunks;
                xv[u].raw = ok ? load_stream16(reinterpret_cast<const uint4*>(x) + c0 + 64 * u) : make_uint4(0, 0, 0, 0);
                gv[u].raw = ok ? reinterpret_cast<const uint4*>(g)[c0 + 64 * u] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (c0 + 64 * u >= chunks) continue;
#pragma unroll
                for (int e = 0; e < N; ++e) acc += El<DT>::to_f32(xv[u].e[e]) * El<DT>::to_f32(gv[u].e[e]);
            }
        }
    } else {
        for (int64_t c = lane; c < a.hidden; c += 64) acc += El<DT>::to_f32(x[c]) * El<DT>::to_f32(g[c]);
    }
    acc = wave_sum(acc);
    if (lane == 0) reinterpret_cast<T*>(a.out)[idx] = El<DT>::from_f32(acc);
    }
}

// ---- host side --------------------------------------------------------------------------------------------
int elem_size(int dt) { return dt == MI8_F32 ? 4 : (dt == MI8_RAW8 ? 1 : 2); }
bool valid_dt(int dt, bool allow_raw) { return dt == MI8_BF16 || dt == MI8_F32 || dt == MI8_F16 || (allow_raw && dt == MI8_RAW8); }
bool valid_w(int dt) { return dt == MI8_BF16 || dt == MI8_F32 || dt == MI8_F16; }
// one wave per row; long inputs are walked by a fixed-size grid (8 blocks per CU's worth) so that waves stay
// resident and keep several rows in flight
unsigned wave_blocks(int64_t rows)
{
    const int64_t need = ceil_div(rows, kWavesPerBlock);
    return (unsigned)(need < kMaxBlocks ? need : kMaxBlocks);
}

bool rows_vectorisable(int64_t hidden, int dt, const void* p0, const void* p1, const void* p2 = nullptr)
{
    return (hidden * elem_size(dt)) % 16 == 0 && aligned16(p0) && aligned16(p1) && aligned16(p2);
}

int check_common(const char* what, const void* x, const void* out, const int32_t* indices, int dtype, bool allow_raw,
                 const void* weights, int w_dtype, int64_t tokens, int64_t hidden, int32_t top_k)
{
    MI8_REQUIRE(x && out && indices, MI8_ERR_ARG, "%s: null pointer", what);
    MI8_REQUIRE(valid_dt(dtype, allow_raw), MI8_ERR_ARG, "%s: unknown element type %d", what, dtype);
    MI8_REQUIRE(!weights || (valid_w(w_dtype) && dtype != MI8_RAW8), MI8_ERR_ARG,
                "%s: weights need a floating-point element type and weight type", what);
    MI8_REQUIRE(tokens > 0 && hidden > 0 && top_k > 0, MI8_ERR_ARG, "%s: empty problem (tokens %lld, hidden %lld, top_k %d)",
                what, (long long)tokens, (long long)hidden, top_k);
    MI8_REQUIRE(tokens * top_k < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "%s: more than 2^31 token slots", what);
    return MI8_OK;
}

int check_bins(const char* what, const int32_t* bins, int32_t experts, int64_t capacity)
{
    MI8_REQUIRE(bins && experts > 0 && capacity > 0, MI8_ERR_ARG, "%s: bins, experts and capacity are required", what);
    MI8_REQUIRE((int64_t)experts * capacity < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "%s: more than 2^31 binned rows", what);
    return MI8_OK;
}

template <bool BINNED>
int launch_gather(PermuteArgs& a, int dtype, int64_t rows, hipStream_t st)
{
    const bool scale = a.weights != nullptr;
#define MI8_G(DT_)                                                                                              \
    if (scale)                                                                                                  \
        hipLaunchKernelGGL((gather_kernel<DT_, true, BINNED>), dim3(wave_blocks(rows)), dim3(kThreads), 0, st, a, rows); \
    else                                                                                                        \
        hipLaunchKernelGGL((gather_kernel<DT_, false, BINNED>), dim3(wave_blocks(rows)), dim3(kThreads), 0, st, a, rows)
    switch (dtype) {
        case MI8_BF16: MI8_G(MI8_BF16); break;
        case MI8_F16: MI8_G(MI8_F16); break;
        case MI8_F32: MI8_G(MI8_F32); break;
        default: hipLaunchKernelGGL((gather_kernel<MI8_RAW8, false, BINNED>), dim3(wave_blocks(rows)), dim3(kThreads), 0, st, a, rows);
    }
#undef MI8_G
    return launch_status(BINNED ? "mi8_moe_binned_gather" : "mi8_moe_gather");
}

template <bool BINNED>
int launch_scatter(PermuteArgs& a, int dtype, int64_t rows, int64_t tokens, hipStream_t st)
{
    const bool scale = a.weights != nullptr;
    const int64_t chunks = a.hidden * elem_size(dtype) / 16;
    if (!BINNED && scatter_in_one_launch(a, tokens, chunks)) {
        const dim3 grid((unsigned)tokens, (unsigned)ceil_div(chunks, kThreads));
#define MI8_S(DT_)                                                                                                   \
    if (scale)                                                                                                       \
        hipLaunchKernelGGL((scatter_few_kernel<DT_, true>), grid, dim3(kThreads), 0, st, a);                         \
    else                                                                                                             \
        hipLaunchKernelGGL((scatter_few_kernel<DT_, false>), grid, dim3(kThreads), 0, st, a)
        switch (dtype) {
            case MI8_BF16: MI8_S(MI8_BF16); break;
            case MI8_F16: MI8_S(MI8_F16); break;
            default: MI8_S(MI8_F32);
        }
#undef MI8_S
        return launch_status("mi8_moe_scatter");
    }
    const unsigned tb = 256;
    // tokens beyond an expert's capacity fill no slot; neither does a slot that `indices` fails to name
    hipLaunchKernelGGL(fill_kernel<int32_t>, dim3((unsigned)ceil_div(a.n, tb)), dim3(tb), 0, st, a.inverse, a.n, (int32_t)-1);
    hipLaunchKernelGGL((inverse_kernel<BINNED>), dim3((unsigned)ceil_div(rows, tb)), dim3(tb), 0, st, a, rows);
#define MI8_S(DT_)                                                                                               \
    if (scale)                                                                                                   \
        hipLaunchKernelGGL((scatter_reduce_kernel<DT_, true>), dim3(wave_blocks(tokens)), dim3(kThreads), 0, st, a, tokens); \
    else                                                                                                         \
        hipLaunchKernelGGL((scatter_reduce_kernel<DT_, false>), dim3(wave_blocks(tokens)), dim3(kThreads), 0, st, a, tokens)
    switch (dtype) {
        case MI8_BF16: MI8_S(MI8_BF16); break;
        case MI8_F16: MI8_S(MI8_F16); break;
        default: MI8_S(MI8_F32);
    }
#undef MI8_S
    return launch_status(BINNED ? "mi8_moe_binned_scatter" : "mi8_moe_scatter");
}

template <bool BINNED>
int launch_wgrad(PermuteArgs& a, int dtype, int64_t rows, hipStream_t st)
{
    switch (dtype) {
        case MI8_BF16:
            hipLaunchKernelGGL((scatter_wgrad_kernel<MI8_BF16, BINNED>), dim3(wave_blocks(rows)), dim3(kThreads), 0, st, a, rows);
            break;
        case MI8_F16:
            hipLaunchKernelGGL((scatter_wgrad_kernel<MI8_F16, BINNED>), dim3(wave_blocks(rows)), dim3(kThreads), 0, st, a, rows);
            break;
        default:
            hipLaunchKernelGGL((scatter_wgrad_kernel<MI8_F32, BINNED>), dim3(wave_blocks(rows)), dim3(kThreads), 0, st, a, rows);
    }
    return launch_status(BINNED ? "mi8_moe_binned_scatter_wgrad" : "mi8_moe_scatter_wgrad");
}

// ---- slots sorted by expert -----------------------------------------------------------------------------
// Stable sort of up to kSortSlots expert ids in one launch: the place of slot e is the number of slots before it that
// have its id or a smaller one, plus the number of slots after it with a smaller one.  A workgroup places 64 slots, one
// per lane; its 16 waves count over a sixteenth of the ids each (wave-uniform, so scalar loads and two vector
// instructions an id).  A call with few tokens is a chain of short launches: the conversion, sort, prefix sum and their
// copies were eleven of them.  Counting is n^2, so larger inputs have a sort of their own.  us on the device, this and the
// chain it replaces: 384 slots 3.6 / 27, 2048 7.4 / 30, 8192 15.8 / 37.
constexpr int kSortThreads = 1024;
constexpr int64_t kSortSlots = 8192;

// the inclusive prefix sums of the experts' counts, by one wave
__device__ __forceinline__ void write_bins(const int64_t* __restrict__ sizes, int experts, int32_t* __restrict__ bins, int lane)
{
    int64_t sum = 0;
    for (int base = 0; base < experts; base += 64) {
        int64_t v = base + lane < experts ? sizes[base + lane] : 0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int64_t o = __shfl_up(v, d, 64);
            if (lane >= d) v += o;
        }
        if (base + lane < experts) bins[base + lane] = (int32_t)(sum + v);
        sum += __shfl(v, 63, 64);
    }
}

template <typename ID>
__global__ __launch_bounds__(kSortThreads) void sort_slots_kernel(const ID* __restrict__ ids, int n,
                                                                  const int64_t* __restrict__ sizes, int experts,
                                                                  int32_t* __restrict__ indices, int32_t* __restrict__ bin_ids,
                                                                  int32_t* __restrict__ bins)
{
    __shared__ int32_t part[kSortThreads / 64][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int first = (int)blockIdx.x * 64, e = first + lane;
    const int32_t id = e < n ? (int32_t)ids[e] : 0;
    const int per = (n + kSortThreads / 64 - 1) / (kSortThreads / 64);
    const int lo = per * wave < n ? per * wave : n, hi = lo + per < n ? lo + per : n;
    int32_t before = 0;
    int j = lo;
    const int end_before = hi < first ? hi : first;
#pragma unroll 8
    for (; j < end_before; ++j) before += (int32_t)ids[j] <= id ? 1 : 0;
    const int end_own = hi < first + 64 ? hi : first + 64;
    for (; j < end_own; ++j) {
        const int32_t other = (int32_t)ids[j];
        before += other < id || (other == id && j < e) ? 1 : 0;
    }
#pragma unroll 8
    for (; j < hi; ++j) before += (int32_t)ids[j] < id ? 1 : 0;
    part[wave][lane] = before;
    __syncthreads();
    if (wave == 0 && e < n) {
        int32_t at = 0;
#pragma unroll
        for (int w = 0; w < kSortThreads / 64; ++w) at += part[w][lane];
        indices[at] = e;
        bin_ids[at] = id;
    }
    if (wave == 1 && blockIdx.x == 0) write_bins(sizes, experts, bins, lane);
}

// The same for more slots: a stable counting sort in two launches, which count the ids of every 1024 slots and place them.  (A
// radix sort of 131072 slots with its conversions and the scan of the sizes is 16 dependent launches, 93 us; with these two a step of 16384 tokens takes 67 us less.)
// Every workgroup of the second reads the counts of all, so the reads grow with the square of the slots, and the radix sort
// has what passes kSortCounts of them.  us, this and that: 8 experts, 2^22 slots 74 / 221 (168 million counts); 64, 2^20 33 / 191, 2^21 87 / 153 (277),
// 2^22 270 / 222; 256, 2^19 33 / 155, 2^20 90 / 197 (271), 2^21 309 / 154.
// An id that names no expert sorts as any other number would.  Where all that are too small, or all that are too large, are one
// number, as those of dropped slots are, they are one more bucket (131072 slots 18 us).  Else the first launch's sorted lists of
// them, one a workgroup, are searched by every such slot (all 131072 of any numbers 450 us, radix sort 66).
constexpr int kSortExperts = 256;  // (16 tables of that many counts in LDS)
constexpr int64_t kSortCounts = 300000000;

__device__ __forceinline__ int sort_bucket(int32_t id, int experts) { return id < 0 ? 0 : id >= experts ? experts + 1 : id + 1; }

// the lists: behind the counts, 1024 words a workgroup
__device__ __forceinline__ int32_t* others_of(int32_t* counts, int experts) { return counts + (int64_t)gridDim.x * (experts + 2); }
__device__ __forceinline__ const int32_t* others_of(const int32_t* counts, int experts) { return counts + (int64_t)gridDim.x * (experts + 2); }

// the place of a workgroup's slot `at` among those of its slots whose ids name no expert
__device__ __forceinline__ int32_t rank_of_other(const int32_t* id_of, int at, int experts)
{
    const int32_t id = id_of[at];
    int32_t rank = 0;
#pragma unroll 4
    for (int j = 0; j < kSortThreads; j += 4) {
        const int4 four = reinterpret_cast<const int4*>(id_of)[j / 4];
        const int32_t v[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) rank += (uint32_t)v[i] >= (uint32_t)experts && (v[i] < id || (v[i] == id && j + i < at)) ? 1 : 0;
    }
    return rank;
}

// how many entries of the other workgroups' lists come before one of this workgroup's: eight lists are searched at a time
__device__ __forceinline__ int32_t others_before(const int32_t* __restrict__ counts, int experts, int32_t id)
{
    const int32_t* __restrict__ others = others_of(counts, experts);
    const int blocks = (int)gridDim.x, own = (int)blockIdx.x;
    constexpr int U = 8;
    int32_t sum = 0;
    for (int first = 0; first < blocks; first += U) {
        int len[U], at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int block = first + u;
            const int32_t* c = counts + (int64_t)(block < blocks ? block : own) * (experts + 2);
            len[u] = block < blocks && block != own ? c[0] + c[experts + 1] : 0;
            at[u] = 0;
        }
        for (int step = kSortThreads; step; step >>= 1) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (at[u] + step <= len[u]) {
                    const int32_t v = others[(int64_t)(first + u) * kSortThreads + at[u] + step - 1];
                    if (v < id || (v == id && first + u < own)) at[u] += step;
                }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) sum += at[u];
    }
    return sum;
}

template <typename ID>
__global__ __launch_bounds__(kSortThreads) void count_slots_kernel(const ID* __restrict__ ids, int n, int experts, int32_t* __restrict__ counts)
{
    __shared__ int32_t count[kSortExperts + 2], least[2], most[2], filled[2];  // (the last three: ids too small, too large)
    __shared__ __attribute__((aligned(16))) int32_t id_of[kSortThreads];
    const int tid = threadIdx.x, e = (int)blockIdx.x * kSortThreads + tid;
    const int32_t id = e < n ? (int32_t)ids[e] : 0;
    const int b = sort_bucket(id, experts), side = b != 0;
    const bool other = b == 0 || b == experts + 1;  // (not the lanes beyond n)
    id_of[tid] = id;
    if (tid < experts + 2) count[tid] = 0;
    if (tid < 2) {
        least[tid] = INT32_MAX;
        most[tid] = INT32_MIN;
        filled[tid] = 0;
    }
    __syncthreads();
    if (e < n) atomicAdd(&count[b], 1);
    if (other) {
        atomicMin(&least[side], id);
        atomicMax(&most[side], id);
    }
    __syncthreads();
    if (tid < experts + 2) counts[(int64_t)blockIdx.x * (experts + 2) + tid] = count[tid];
    if (other) {
        const int at = least[side] == most[side] ? (side ? count[0] : 0) + atomicAdd(&filled[side], 1) : rank_of_other(id_of, tid, experts);
        others_of(counts, experts)[(int64_t)blockIdx.x * kSortThreads + at] = id;
    }
}

template <typename ID>
__global__ __launch_bounds__(kSortThreads) void place_slots_kernel(const ID* __restrict__ ids, int n, const int64_t* __restrict__ sizes,
                                                                   int experts, const int32_t* __restrict__ counts,
                                                                   int32_t* __restrict__ indices, int32_t* __restrict__ bin_ids,
                                                                   int32_t* __restrict__ bins)
{
    constexpr int kWaves = kSortThreads / 64;
    __shared__ int32_t of_wave[kWaves][kSortExperts + 2], before[kSortExperts + 2], total[kSortExperts + 2];
    __shared__ int32_t slot_at[kSortThreads], least[2], most[2];  // (ids too small, too large)
    __shared__ __attribute__((aligned(16))) int32_t id_of[kSortThreads];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, buckets = experts + 2;
    for (int b = tid; b < kWaves * (kSortExperts + 2); b += kSortThreads) (&of_wave[0][0])[b] = 0;
    if (tid < buckets) before[tid] = total[tid] = 0;
    if (tid < 2) {
        least[tid] = INT32_MAX;
        most[tid] = INT32_MIN;
    }
    __syncthreads();
    // slots of each bucket in the blocks before this one and in all: as many threads a bucket as there are
    const int parts = kSortThreads / buckets, part = tid / buckets, bucket = tid - part * buckets;
    if (part < parts) {
        int32_t sum = 0, mine = 0;
#pragma unroll 4
        for (int b = part; b < (int)gridDim.x; b += parts) {
            const int32_t c = counts[(int64_t)b * buckets + bucket];
            sum += c;
            if (b < (int)blockIdx.x) mine += c;
        }
        atomicAdd(&total[bucket], sum);
        atomicAdd(&before[bucket], mine);
    }
    // place among the wave's slots of one bucket
    const int e = (int)blockIdx.x * kSortThreads + tid;
    const int32_t id = e < n ? (int32_t)ids[e] : 0;
    const int b = sort_bucket(id, experts);
    id_of[tid] = id;
    uint64_t same = __ballot(e < n);
    for (int bit = 0; (buckets - 1) >> bit; ++bit) {
        const uint64_t set = __ballot((b >> bit) & 1);
        same &= (b >> bit) & 1 ? set : ~set;
    }
    const int rank = __popcll(same & (((uint64_t)1 << lane) - 1));
    if (e < n && rank == 0) of_wave[wave][b] = __popcll(same);
    __syncthreads();
    const int others = total[0] + total[experts + 1];
    for (int i = tid; i < (others ? 2 * (int)gridDim.x : 0); i += kSortThreads) {
        const int32_t* c = counts + (int64_t)(i >> 1) * buckets;
        const int32_t low = c[0], len = i & 1 ? c[experts + 1] : low;
        if (len) {
            const int32_t* list = others_of(counts, experts) + (int64_t)(i >> 1) * kSortThreads + (i & 1 ? low : 0);
            atomicMin(&least[i & 1], list[0]);
            atomicMax(&most[i & 1], list[len - 1]);
        }
    }
    if (wave == 0) {  // where each bucket starts
        int32_t sum = 0;
        for (int base = 0; base < buckets; base += 64) {
            const int32_t own = base + lane < buckets ? total[base + lane] : 0;
            int32_t v = own;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int32_t o = __shfl_up(v, d, 64);
                if (lane >= d) v += o;
            }
            if (base + lane < buckets) before[base + lane] += sum + v - own;
            sum += __shfl(v, 63, 64);
        }
    }
    __syncthreads();
    const bool several = least[0] < most[0] || least[1] < most[1], other = b == 0 || b == experts + 1;
    if (e < n && !(several && other)) {
        int32_t at = before[b] + rank;
        for (int w = 0; w < wave; ++w) at += of_wave[w][b];
        indices[at] = e;
        bin_ids[at] = id;
    }
    if (several) {  // (uniform) lane i takes the i-th of the workgroup's list, so that a wave searches close by
        if (other) slot_at[rank_of_other(id_of, tid, experts)] = tid;
        __syncthreads();
        const int32_t* c = counts + (int64_t)blockIdx.x * buckets;
        if (tid < c[0] + c[experts + 1]) {
            const int slot = slot_at[tid];
            const int32_t its_id = id_of[slot];
            const int32_t at = (its_id < 0 ? 0 : n - others) + tid + others_before(counts, experts, its_id);
            indices[at] = (int)blockIdx.x * kSortThreads + slot;
            bin_ids[at] = its_id;
        }
    }
    if (wave == 1 && blockIdx.x == 0) write_bins(sizes, experts, bins, lane);
}

}  // namespace
}  // namespace mi8

using namespace mi8;

extern "C" int64_t mi8_moe_sort_workspace_words(int64_t n, int32_t experts)
{
    if (n <= 0 || n >= (1 << 30) || experts <= 0 || experts > kSortExperts) return 0;
    const int64_t blocks = ceil_div(n, kSortThreads);
    return blocks * blocks * (experts + 2) <= kSortCounts ? blocks * (experts + 2 + kSortThreads) : 0;
}

extern "C" int mi8_moe_sort_many_slots(const void* ids, int ids_are_64, int64_t n, const int64_t* sizes, int32_t experts,
                                       int32_t* workspace, int32_t* indices, int32_t* bin_ids, int32_t* bins, void* stream)
{
    MI8_REQUIRE(ids && sizes && workspace && indices && bin_ids && bins, MI8_ERR_ARG, "mi8_moe_sort_many_slots: null pointer");
    MI8_REQUIRE(mi8_moe_sort_workspace_words(n, experts) > 0, MI8_ERR_UNSUPPORTED,
                "mi8_moe_sort_many_slots: needs 1..%d experts and no more slots than mi8_moe_sort_workspace_words takes (got %lld, %d)", kSortExperts,
                (long long)n, experts);
    const dim3 grid((unsigned)ceil_div(n, kSortThreads)), threads(kSortThreads);
    hipStream_t st = (hipStream_t)stream;
    if (ids_are_64) {
        hipLaunchKernelGGL(count_slots_kernel<int64_t>, grid, threads, 0, st, (const int64_t*)ids, (int)n, experts, workspace);
        hipLaunchKernelGGL(place_slots_kernel<int64_t>, grid, threads, 0, st, (const int64_t*)ids, (int)n, sizes, experts, workspace, indices,
                           bin_ids, bins);
    } else {
        hipLaunchKernelGGL(count_slots_kernel<int32_t>, grid, threads, 0, st, (const int32_t*)ids, (int)n, experts, workspace);
        hipLaunchKernelGGL(place_slots_kernel<int32_t>, grid, threads, 0, st, (const int32_t*)ids, (int)n, sizes, experts, workspace, indices,
                           bin_ids, bins);
    }
    return launch_status("mi8_moe_sort_many_slots");
}

extern "C" int64_t mi8_moe_sort_slots_max(void) { return kSortSlots; }

extern "C" int mi8_moe_sort_slots(const void* ids, int ids_are_64, int64_t n, const int64_t* sizes, int32_t experts,
                                  int32_t* indices, int32_t* bin_ids, int32_t* bins, void* stream)
{
    MI8_REQUIRE(ids && sizes && indices && bin_ids && bins, MI8_ERR_ARG, "mi8_moe_sort_slots: null pointer");
    MI8_REQUIRE(n > 0 && n <= kSortSlots && experts > 0, MI8_ERR_UNSUPPORTED,
                "mi8_moe_sort_slots: needs 1..%lld slots and an expert (got %lld, %d)", (long long)kSortSlots, (long long)n, experts);
    const dim3 grid((unsigned)ceil_div(n, 64));
    if (ids_are_64)
        hipLaunchKernelGGL(sort_slots_kernel<int64_t>, grid, dim3(kSortThreads), 0, (hipStream_t)stream, (const int64_t*)ids,
                           (int)n, sizes, experts, indices, bin_ids, bins);
    else
        hipLaunchKernelGGL(sort_slots_kernel<int32_t>, grid, dim3(kSortThreads), 0, (hipStream_t)stream, (const int32_t*)ids,
                           (int)n, sizes, experts, indices, bin_ids, bins);
    return launch_status("mi8_moe_sort_slots");
}

extern "C" int mi8_moe_gather(const void* x, int dtype, int64_t tokens, int64_t hidden, const int32_t* indices,
                              const void* weights, int w_dtype, int32_t top_k, void* out, void* stream)
{
    int rc = check_common("mi8_moe_gather", x, out, indices, dtype, true, weights, w_dtype, tokens, hidden, top_k);
    if (rc != MI8_OK) return rc;
    PermuteArgs a{x, out, indices, weights, w_dtype, nullptr, nullptr, nullptr, tokens * top_k, hidden, top_k, 0, 0,
                  rows_vectorisable(hidden, dtype, x, out)};
    return launch_gather<false>(a, dtype, a.n, (hipStream_t)stream);
}

extern "C" int mi8_moe_binned_gather(const void* x, int dtype, int64_t tokens, int64_t hidden, const int32_t* indices,
                                     const void* weights, int w_dtype, const int32_t* bins, int32_t experts,
                                     int64_t capacity, int32_t top_k, void* out, void* stream)
{
    int rc = check_common("mi8_moe_binned_gather", x, out, indices, dtype, true, weights, w_dtype, tokens, hidden, top_k);
    if (rc == MI8_OK) rc = check_bins("mi8_moe_binned_gather", bins, experts, capacity);
    if (rc != MI8_OK) return rc;
    PermuteArgs a{x, out, indices, weights, w_dtype, bins, nullptr, nullptr, tokens * top_k, hidden, top_k, experts,
                  (int32_t)capacity, rows_vectorisable(hidden, dtype, x, out)};
    return launch_gather<true>(a, dtype, (int64_t)experts * capacity, (hipStream_t)stream);
}

extern "C" int mi8_moe_scatter(const void* x, int dtype, int64_t tokens, int64_t hidden, const int32_t* indices,
                               const void* weights, int w_dtype, int32_t top_k, int32_t* inverse_workspace, void* out,
                               void* stream)
{
    int rc = check_common("mi8_moe_scatter", x, out, indices, dtype, false, weights, w_dtype, tokens, hidden, top_k);
    if (rc != MI8_OK) return rc;
    MI8_REQUIRE(inverse_workspace, MI8_ERR_ARG, "mi8_moe_scatter: the inverse workspace (tokens * top_k int32) is required");
    PermuteArgs a{x, out, indices, weights, w_dtype, nullptr, inverse_workspace, nullptr, tokens * top_k, hidden, top_k, 0,
                  0, rows_vectorisable(hidden, dtype, x, out)};
    return launch_scatter<false>(a, dtype, a.n, tokens, (hipStream_t)stream);
}

extern "C" int mi8_moe_binned_scatter(const void* x, int dtype, int64_t tokens, int64_t hidden, const int32_t* indices,
                                      const void* weights, int w_dtype, const int32_t* bins, int32_t experts,
                                      int64_t capacity, int32_t top_k, int32_t* inverse_workspace, void* out,
                                      void* stream)
{
    int rc = check_common("mi8_moe_binned_scatter", x, out, indices, dtype, false, weights, w_dtype, tokens, hidden, top_k);
    if (rc == MI8_OK) rc = check_bins("mi8_moe_binned_scatter", bins, experts, capacity);
    if (rc != MI8_OK) return rc;
    MI8_REQUIRE(inverse_workspace, MI8_ERR_ARG, "mi8_moe_binned_scatter: the inverse workspace (tokens * top_k int32) is required");
    PermuteArgs a{x, out, indices, weights, w_dtype, bins, inverse_workspace, nullptr, tokens * top_k, hidden, top_k,
                  experts, (int32_t)capacity, rows_vectorisable(hidden, dtype, x, out)};
    return launch_scatter<true>(a, dtype, (int64_t)experts * capacity, tokens, (hipStream_t)stream);
}

extern "C" int mi8_moe_scatter_wgrad(const void* x, const void* grad, int dtype, int64_t tokens, int64_t hidden,
                                     const int32_t* indices, int32_t top_k, void* out, void* stream)
{
    int rc = check_common("mi8_moe_scatter_wgrad", x, out, indices, dtype, false, nullptr, 0, tokens, hidden, top_k);
    if (rc != MI8_OK) return rc;
    MI8_REQUIRE(grad, MI8_ERR_ARG, "mi8_moe_scatter_wgrad: grad is null");
    PermuteArgs a{x, out, indices, nullptr, 0, nullptr, nullptr, grad, tokens * top_k, hidden, top_k, 0, 0,
                  rows_vectorisable(hidden, dtype, x, grad)};
    return launch_wgrad<false>(a, dtype, a.n, (hipStream_t)stream);
}

extern "C" int mi8_moe_binned_scatter_wgrad(const void* x, const void* grad, int dtype, int64_t tokens, int64_t hidden,
                                            const int32_t* indices, const int32_t* bins, int32_t experts,
                                            int64_t capacity, int32_t top_k, void* out, void* stream)
{
    int rc = check_common("mi8_moe_binned_scatter_wgrad", x, out, indices, dtype, false, nullptr, 0, tokens, hidden, top_k);
    if (rc == MI8_OK) rc = check_bins("mi8_moe_binned_scatter_wgrad", bins, experts, capacity);
    if (rc != MI8_OK) return rc;
    MI8_REQUIRE(grad, MI8_ERR_ARG, "mi8_moe_binned_scatter_wgrad: grad is null");
    hipStream_t st = (hipStream_t)stream;
    // slots of dropped tokens get no contribution: the output starts from zero
    const int64_t n = tokens * top_k;
    if (elem_size(dtype) == 4)
        hipLaunchKernelGGL(fill_kernel<uint32_t>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, st, (uint32_t*)out, n, 0u);
    else
        hipLaunchKernelGGL(fill_kernel<uint16_t>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, st, (uint16_t*)out, n,
                           (uint16_t)0);
    PermuteArgs a{x, out, indices, nullptr, 0, bins, nullptr, grad, tokens * top_k, hidden, top_k, experts,
                  (int32_t)capacity, rows_vectorisable(hidden, dtype, x, grad)};
    return launch_wgrad<true>(a, dtype, (int64_t)experts * capacity, st);
}
