// Several tensors quantised in one launch per pass: the input and the weights of a layer, the gradients of its outputs.
//
// What bounds it: the tensors of a small or middle-sized layer are a few MB each, so a launch of its own per tensor and pass
// is latency - filling and draining the chip around 1-6 us of traffic - and a call from the host.  One grid over the tiles
// of all of them pays that once per pass.  The second pass loads its tile before it reduces the partial maxima: neither waits
// for the other.  A call among others, us, tensor by tensor / together: one projection of 116 tokens, 4096 x 4096, input and
// weight 51.1 / 37.9; of 2048 tokens, 4096 x 11008, 132.9 / 128.6; forward and backward of four projections on 1537 tokens of 2048
// with scales per row and column (ten tensors, 30 launches before, 8 now) 633 / 470.
#include <algorithm>

#include "../../include/mi8.h"
#include "mi8_cast_tile.h"

namespace mi8 {
namespace {

// ---- amax of several tensors, then one scale each (tensorwise) ------------------------------------------------------

struct CastItem {
    const void* x;
    int64_t rows, cols;
    const uint32_t* slots;  // partial maxima; null: scale_in
    const float* scale_in;
    uint8_t* out;
    int64_t ld_out;
    uint8_t* out_t;
    int64_t ld_t, t_end;
    float* scale_out;
    int n_slots;
    int fp32;
    int tiles_n;
    int first;  // the item's first workgroup in the cast pass
};

struct AmaxItem {
    const void* x;
    int64_t n;
    uint32_t* slots;
    int fp32;
    int first, blocks;  // workgroups, one slot each
};

struct AmaxItems {
    AmaxItem t[MI8_CAST_BATCH];
    int count;
};

struct CastItems {
    CastItem t[MI8_CAST_BATCH];
    int count;
    bool pow2, stream;
};

template <typename Items>
__device__ __forceinline__ int item_of_block(const Items& a, int block)
{
    int t = 0;
#pragma unroll
    for (int i = 1; i < MI8_CAST_BATCH; ++i)
        if (i < a.count && block >= a.t[i].first) t = i;
    return t;
}

template <int HP>
__device__ __forceinline__ uint32_t amax_of_range(const void* p, int64_t n, int block, int blocks)
{
    constexpr int kPerVec = HP == MI8_BF16 ? 8 : 4;
    const uint4* x = reinterpret_cast<const uint4*>(p);
    const int64_t nvec = n / kPerVec;
    uint32_t acc[4] = {0, 0, 0, 0};
    const BlockRange r = block_range(nvec, block, blocks);
    int64_t i = r.lo + threadIdx.x;
    for (; i + 3 * kThreads < r.hi; i += 4 * kThreads) {
        const uint4 v0 = x[i], v1 = x[i + kThreads], v2 = x[i + 2 * kThreads], v3 = x[i + 3 * kThreads];
        absmax_accumulate<HP>(v0, acc);
        absmax_accumulate<HP>(v1, acc);
        absmax_accumulate<HP>(v2, acc);
        absmax_accumulate<HP>(v3, acc);
    }
    for (; i < r.hi; i += kThreads) absmax_accumulate<HP>(x[i], acc);
    return absmax_fold<HP>(acc);  // (n % 16 == 0: no tail)
}

__global__ __launch_bounds__(kThreads) void amax_items_kernel(AmaxItems a)
{
    __shared__ uint32_t smem[4];
    const AmaxItem& t = a.t[item_of_block(a, (int)blockIdx.x)];
    const int block = (int)blockIdx.x - t.first;
    uint32_t m = t.fp32 ? amax_of_range<MI8_F32>(t.x, t.n, block, t.blocks) : amax_of_range<MI8_BF16>(t.x, t.n, block, t.blocks);
    m = block_umax(m, smem);
    if (threadIdx.x == 0) t.slots[block] = m;
}

template <int HP, int FP8, bool SW>
__device__ __forceinline__ void cast_item(const CastItem& t, int tile, bool pow2, bool stream, uint32_t* lds_t, uint32_t* smem)
{
    const int64_t row0 = (int64_t)(tile / t.tiles_n) * kTile, col0 = (int64_t)(tile % t.tiles_n) * kTile;
    RawTile<HP> values;
    values.load(t.x, t.rows, t.cols, row0, col0);
    float s;
    if (t.slots) {
        uint32_t m = 0;
        for (int i = threadIdx.x; i < t.n_slots; i += kThreads) m = umax32(m, t.slots[i]);
        m = block_umax(m, smem);
        s = scale_from_amax_bits<FP8>(m, pow2);  // every lane: same bits in, same bits out
    } else {
        s = t.scale_in[0];
    }
    if (threadIdx.x == 0 && tile == 0) t.scale_out[0] = s;
    float sc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sc[i] = s;
    tile_quantise<FP8, SW>(values, t.rows, t.cols, row0, col0, sc, t.out, t.ld_out, t.out_t, t.ld_t, row0, t.t_end, lds_t, stream);
}

// MIX: bf16, float32, or both
enum { kAllBf16, kAllF32, kMixed };

template <int MIX, int FP8, bool SW>
__global__ __launch_bounds__(kThreads) void cast_items_kernel(CastItems a)
{
    __shared__ __attribute__((aligned(16))) uint32_t lds_t[kTile * kTile / 4];
    __shared__ uint32_t smem[4];
    const int block = (int)blockIdx.x;
    const CastItem& t = a.t[item_of_block(a, block)];
    if (MIX == kAllF32 || (MIX == kMixed && t.fp32))
        cast_item<MI8_F32, FP8, SW>(t, block - t.first, a.pow2, a.stream, lds_t, smem);
    else
        cast_item<MI8_BF16, FP8, SW>(t, block - t.first, a.pow2, a.stream, lds_t, smem);
}

// ---- a scale per row (row-major copy) and a scale per column (transposed copy) of several tensors -----------------------
// Pass 1 leaves partial maxima in plain tables, nothing to clear and no atomics: per column over chunks of at most
// chunk_tiles * 128 rows, per row over the 128 columns of a tile.  Pass 2 folds the partials of its 128 rows and columns,
// 16 bytes a load.
//
// Both passes are bound by memory, so by the bytes in flight: kernels of their own where all tensors are bf16 (68 and 88 VGPRs
// instead of 110 and 122 with a branch on the type), a tile kept as bf16 until it is quantised, and a pass 1 that loads the
// next half tile while it folds this one.  16384 x 4096 bf16 (134 MB): 84 us before these three, 75 now (5.4 TB/s with the second
// read); three weights of 65536 x 2048: 540 and 474.

struct TwoCastItem {
    const void* x;
    int64_t rows, cols;
    uint8_t* out_r;
    int64_t ld_r;
    float* row_scale;
    uint8_t* out_t;
    int64_t ld_t;
    float* col_scale;
    uint32_t* col_part;  // [chunks][128 tiles_n], group after group
    uint32_t* row_part;  // [tiles_n][128 tiles_m]
    int fp32;
    int tiles_m, tiles_n, chunk_tiles;
    int group_tiles, group_chunks;  // row tiles and chunks of a group
    int first, first_chunk;  // first workgroup in the cast pass and in the amax pass
};

struct TwoCastItems {
    TwoCastItem t[MI8_CAST_BATCH];
    int count;
    bool pow2, stream;
};

template <int HP>
__device__ __forceinline__ void two_amax_body(const TwoCastItem& t, int block, uint32_t (&red)[16][kTile + 1])
{
    const int tid = threadIdx.x;
    const int cl = tid & 15, rg = tid >> 4;
    const int ct = block % t.tiles_n, chunk = block / t.tiles_n;
    const int64_t c8 = (int64_t)ct * kTile + 8 * cl;
    const char* xb = reinterpret_cast<const char*>(t.x) + c8 * HpVec<HP>::kBytes;
    const int64_t pitch = t.cols * HpVec<HP>::kBytes;
    constexpr int NV = HpVec<HP>::kBytes == 2 ? 1 : 2;
    uint32_t acc[NV][4];
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[v][k] = 0;
    uint32_t* const row_out = t.row_part + (int64_t)ct * t.tiles_m * kTile;
    const int group = chunk / t.group_chunks;
    const int first = group * t.group_tiles + (chunk - group * t.group_chunks) * t.chunk_tiles, end = (group + 1) * t.group_tiles;
    const int last = first + t.chunk_tiles < end ? first + t.chunk_tiles : end;
    // half a tile of rows in flight while the half before it is folded
    constexpr int kHalf = kTile / 32;
    uint4 v[2][kHalf][NV];
    const auto load_half = [&](uint4(&to)[kHalf][NV], int64_t row0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kHalf; ++i)
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                to[i][k] = make_uint4(0, 0, 0, 0);
                if (c8 < t.cols && row0 + 16 * i < t.rows)
                    to[i][k] = reinterpret_cast<const uint4*>(xb + (row0 + 16 * i) * pitch)[k];
            }
    };
    const auto fold_half = [&](const uint4(&from)[kHalf][NV], int64_t row0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
            uint32_t rowacc[4] = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                absmax_accumulate<HP>(from[i][k], acc[k]);
                absmax_accumulate<HP>(from[i][k], rowacc);
            }
            uint32_t m = absmax_fold<HP>(rowacc);  // the 16 lanes that share this row fold their eight columns each
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) m = umax32(m, (uint32_t)__shfl_xor((int)m, off, 16));
            if (cl == 0) row_out[row0 + 16 * i] = m;  // (the table has whole tiles of rows)
        }
    };
    int64_t row0 = (int64_t)first * kTile + rg;
    load_half(v[0], row0);
    for (int rt = first; rt < last; ++rt, row0 += kTile) {
        load_half(v[1], row0 + kTile / 2);
        fold_half(v[0], row0);
        if (rt + 1 < last) load_half(v[0], row0 + kTile);
        fold_half(v[1], row0 + kTile / 2);
    }
    if constexpr (HP == MI8_BF16) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            red[rg][8 * cl + 2 * k] = (acc[0][k] & 0xFFFFu) << 16;
            red[rg][8 * cl + 2 * k + 1] = acc[0][k] & 0xFFFF0000u;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            red[rg][8 * cl + k] = acc[0][k];
            red[rg][8 * cl + 4 + k] = acc[NV - 1][k];
        }
    }
    __syncthreads();
    if (tid < kTile) {
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) m = umax32(m, red[k][tid]);
        t.col_part[((int64_t)chunk * t.tiles_n + ct) * kTile + tid] = m;
    }
}

template <int MIX>
__global__ __launch_bounds__(kThreads) void two_amax_items_kernel(TwoCastItems a)
{
    __shared__ uint32_t red[16][kTile + 1];
    int i = 0;
#pragma unroll
    for (int k = 1; k < MI8_CAST_BATCH; ++k)
        if (k < a.count && (int)blockIdx.x >= a.t[k].first_chunk) i = k;
    const TwoCastItem& t = a.t[i];
    if (MIX == kAllF32 || (MIX == kMixed && t.fp32))
        two_amax_body<MI8_F32>(t, (int)blockIdx.x - t.first_chunk, red);
    else
        two_amax_body<MI8_BF16>(t, (int)blockIdx.x - t.first_chunk, red);
}

template <int HP, int FP8, bool SW>
__device__ __forceinline__ void two_cast_item(const TwoCastItem& t, int tile, bool pow2, bool stream, uint32_t* lds_t, uint32_t (&parts)[2][4][kTile],
                                              float (&s_scale)[2][kTile])
{
    const int rt = tile / t.tiles_n, ct = tile % t.tiles_n;
    const int64_t row0 = (int64_t)rt * kTile, col0 = (int64_t)ct * kTile;
    const int tid = threadIdx.x;
    RawTile<HP> values;
    values.load(t.x, t.rows, t.cols, row0, col0);
    // the first half of the workgroup folds the columns' partials, the second the rows': four lanes share four of them
    const bool of_rows = tid >= kTile;
    {
        const int part = (tid >> 5) & 3, at = (tid & 31) * 4;
        const int n = of_rows ? t.tiles_n : t.group_chunks;
        const int64_t pitch = (int64_t)kTile * (of_rows ? t.tiles_m : t.tiles_n);
        const uint32_t* p = (of_rows ? t.row_part + row0 : t.col_part + col0 + (rt / t.group_tiles) * t.group_chunks * pitch) + at;
        uint4 m = make_uint4(0, 0, 0, 0);
#pragma unroll 8
        for (int k = part; k < n; k += 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(p + k * pitch);
            m = make_uint4(umax32(m.x, v.x), umax32(m.y, v.y), umax32(m.z, v.z), umax32(m.w, v.w));
        }
        *reinterpret_cast<uint4*>(&parts[of_rows][part][at]) = m;
    }
    __syncthreads();
    {
        const int i = tid & (kTile - 1);
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) m = umax32(m, parts[of_rows][k][i]);
        const float s = scale_from_amax_bits<FP8>(m, pow2);
        s_scale[of_rows][i] = s;
        if (of_rows ? ct == 0 && row0 + i < t.rows : rt % t.group_tiles == 0 && col0 + i < t.cols)
            (of_rows ? t.row_scale + row0 : t.col_scale + (rt / t.group_tiles) * t.cols + col0)[i] = s;
    }
    __syncthreads();
    float sc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sc[i] = s_scale[0][8 * (tid & 15) + i];
    tile_quantise<FP8, SW>(values, t.rows, t.cols, row0, col0, sc, nullptr, 0, t.out_t, t.ld_t, row0, t.ld_t, lds_t, stream, t.out_r, t.ld_r,
                           s_scale[1], row0);
}

template <int MIX, int FP8, bool SW>
__global__ __launch_bounds__(kThreads) void two_cast_items_kernel(TwoCastItems a)
{
    __shared__ __attribute__((aligned(16))) uint32_t lds_t[kTile * kTile / 4];
    __shared__ __attribute__((aligned(16))) uint32_t parts[2][4][kTile];
    __shared__ float s_scale[2][kTile];  // of the tile's columns, of its rows
    const int block = (int)blockIdx.x;
    const TwoCastItem& t = a.t[item_of_block(a, block)];
    if (MIX == kAllF32 || (MIX == kMixed && t.fp32))
        two_cast_item<MI8_F32, FP8, SW>(t, block - t.first, a.pow2, a.stream, lds_t, parts, s_scale);
    else
        two_cast_item<MI8_BF16, FP8, SW>(t, block - t.first, a.pow2, a.stream, lds_t, parts, s_scale);
}

bool valid_hp(int v) { return v == MI8_BF16 || v == MI8_F32; }

// row tiles per chunk of the column partials: at most 32 chunks of a group of rows (or of all) to fold (16384 x 4096: 75 us; 64 chunks
// 76.6, 16 chunks 88); the last chunk of a group is shorter, so that a chunk has rows of one group only
// (three weights of 8 x 5504 x 1024, 43 tiles a group: 165 us, in chunks that divide a group - here all of it - 239)
int chunk_tiles_for(int64_t group_tiles) { return (int)ceil_div(group_tiles, 32); }

template <typename Kernel, typename Args>
int launch_items(Kernel kern, const Args& a, int64_t blocks, hipStream_t st, const char* what)
{
    MI8_REQUIRE(blocks < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "%s: grid too large", what);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), 0, st, a);
    return launch_status(what);
}

template <typename Items>
int mix_of(const Items& a)
{
    int fp32 = 0;
    for (int i = 0; i < a.count; ++i) fp32 += a.t[i].fp32;
    return fp32 == 0 ? kAllBf16 : fp32 == a.count ? kAllF32 : kMixed;
}

#define MI8_BY_TYPE(KERNEL, MIX_)                                                                                             \
    (fp8_dtype == MI8_E4M3 ? (sw ? launch_items(KERNEL<MIX_, MI8_E4M3, true>, a, blocks, st, what)                            \
                                 : launch_items(KERNEL<MIX_, MI8_E4M3, false>, a, blocks, st, what))                          \
                           : (sw ? launch_items(KERNEL<MIX_, MI8_E5M2, true>, a, blocks, st, what)                            \
                                 : launch_items(KERNEL<MIX_, MI8_E5M2, false>, a, blocks, st, what)))

int launch_cast(const CastItems& a, int fp8_dtype, bool sw, int64_t blocks, hipStream_t st, const char* what)
{
    const int mix = mix_of(a);
    return mix == kAllBf16 ? MI8_BY_TYPE(cast_items_kernel, kAllBf16) : mix == kAllF32 ? MI8_BY_TYPE(cast_items_kernel, kAllF32)
                                                                                      : MI8_BY_TYPE(cast_items_kernel, kMixed);
}

int launch_two_cast(const TwoCastItems& a, int fp8_dtype, bool sw, int64_t chunk_blocks, int64_t blocks, hipStream_t st, const char* what)
{
    const int mix = mix_of(a);
    const auto amax = mix == kAllBf16 ? two_amax_items_kernel<kAllBf16> : mix == kAllF32 ? two_amax_items_kernel<kAllF32> : two_amax_items_kernel<kMixed>;
    if (int rc = launch_items(amax, a, chunk_blocks, st, what)) return rc;
    return mix == kAllBf16 ? MI8_BY_TYPE(two_cast_items_kernel, kAllBf16) : mix == kAllF32 ? MI8_BY_TYPE(two_cast_items_kernel, kAllF32)
                                                                                          : MI8_BY_TYPE(two_cast_items_kernel, kMixed);
}
#undef MI8_BY_TYPE

}  // namespace
}  // namespace mi8

using namespace mi8;

extern "C" int mi8_cast_tensorwise_batch(const mi8_cast_item* items, int32_t count, int fp8_dtype, uint32_t flags, void* stream)
{
    const char* what = "mi8_cast_tensorwise_batch";
    MI8_REQUIRE(items, MI8_ERR_ARG, "%s: null pointer", what);
    MI8_REQUIRE(count > 0 && count <= MI8_CAST_BATCH, MI8_ERR_ARG, "%s: %d tensors (1..%d)", what, count, MI8_CAST_BATCH);
    MI8_REQUIRE(fp8_dtype == MI8_E4M3 || fp8_dtype == MI8_E5M2, MI8_ERR_ARG, "%s: unknown fp8 dtype %d", what, fp8_dtype);
    AmaxItems am{};
    CastItems ca{};
    ca.count = count;
    ca.pow2 = (flags & MI8_FLAG_POW2_SCALE) != 0;
    int64_t amax_blocks = 0, cast_blocks = 0, bytes = 0, end = 0;
    for (int i = 0; i < count; ++i) {
        const mi8_cast_item& t = items[i];
        MI8_REQUIRE(t.x && t.scale_out && (t.out || t.out_t) && (t.slots || t.scale_in || t.amax_ws), MI8_ERR_ARG, "%s: tensor %d: null pointer", what, i);
        MI8_REQUIRE(valid_hp(t.hp_dtype), MI8_ERR_ARG, "%s: tensor %d: unknown hp dtype %d", what, i, t.hp_dtype);
        MI8_REQUIRE(t.rows > 0 && t.cols > 0, MI8_ERR_ARG, "%s: tensor %d is empty", what, i);
        MI8_REQUIRE(t.cols % 16 == 0, MI8_ERR_UNSUPPORTED, "%s: tensor %d: cols (%lld) must be a multiple of 16", what, i, (long long)t.cols);
        MI8_REQUIRE(aligned16(t.x) && aligned16(t.out) && aligned16(t.out_t), MI8_ERR_UNSUPPORTED, "%s: tensor %d: pointers must be 16-byte aligned", what, i);
        MI8_REQUIRE(!t.slots || (t.n_slots > 0 && t.n_slots <= MI8_AMAX_SLOTS), MI8_ERR_ARG, "%s: tensor %d: n_slots %d out of range", what, i, t.n_slots);
        const int64_t t_end = round_up(t.rows, t.pad_t128 ? 128 : 16);
        MI8_REQUIRE(!t.out || (t.ld_out >= t.cols && t.ld_out % 16 == 0), MI8_ERR_UNSUPPORTED, "%s: tensor %d: ld_out (%lld)", what, i, (long long)t.ld_out);
        MI8_REQUIRE(!t.out_t || (t.ld_t >= t_end && t.ld_t % 16 == 0), MI8_ERR_UNSUPPORTED, "%s: tensor %d: ld_t (%lld)", what, i, (long long)t.ld_t);
        const int fp32 = t.hp_dtype == MI8_F32;
        const uint32_t* slots = t.slots;
        int n_slots = t.n_slots;
        if (!slots && !t.scale_in) {
            n_slots = mi8_amax_slots_for(t.rows * t.cols);
            slots = t.amax_ws;
            am.t[am.count++] = AmaxItem{t.x, t.rows * t.cols, t.amax_ws, fp32, (int)amax_blocks, n_slots};
            amax_blocks += n_slots;
        }
        const int64_t tiles_n = ceil_div(t.cols, kTile), tiles = tiles_n * ceil_div(t.rows, kTile);
        MI8_REQUIRE(cast_blocks + tiles < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "%s: grid too large", what);
        ca.t[i] = CastItem{t.x, t.rows, t.cols, slots, t.scale_in, (uint8_t*)t.out, t.ld_out, (uint8_t*)t.out_t, t.ld_t, t_end,
                           t.scale_out, n_slots, fp32, (int)tiles_n, (int)cast_blocks};
        cast_blocks += tiles;
        bytes += t.rows * t.cols * ((t.out ? 1 : 0) + (t.out_t ? 1 : 0));
        end = std::max({end, t.out ? t.rows * t.ld_out : 0, t.out_t ? t.cols * t.ld_t : 0});
    }
    ca.stream = streams_outputs(bytes, end);
    hipStream_t st = (hipStream_t)stream;
    if (am.count)
        if (int rc = launch_items(amax_items_kernel, am, amax_blocks, st, what)) return rc;
    return launch_cast(ca, fp8_dtype, (flags & MI8_FLAG_SW_CVT) != 0, cast_blocks, st, what);
}

extern "C" int64_t mi8_two_cast_workspace_words(int64_t rows, int64_t cols)
{
    if (rows <= 0 || cols <= 0) return 0;
    const int64_t tiles_m = ceil_div(rows, kTile), tiles_n = ceil_div(cols, kTile);
    return 2 * tiles_n * tiles_m * kTile;  // (a chunk has at least one row tile)
}

extern "C" int mi8_cast_rows_and_colwise_t_batch(const mi8_two_cast_item* items, int32_t count, int fp8_dtype, uint32_t flags,
                                                 void* stream)
{
    const char* what = "mi8_cast_rows_and_colwise_t_batch";
    MI8_REQUIRE(items, MI8_ERR_ARG, "%s: null pointer", what);
    MI8_REQUIRE(count > 0 && count <= MI8_CAST_BATCH, MI8_ERR_ARG, "%s: %d tensors (1..%d)", what, count, MI8_CAST_BATCH);
    MI8_REQUIRE(fp8_dtype == MI8_E4M3 || fp8_dtype == MI8_E5M2, MI8_ERR_ARG, "%s: unknown fp8 dtype %d", what, fp8_dtype);
    for (int i = 0; i < count; ++i) {
        const mi8_two_cast_item& t = items[i];
        MI8_REQUIRE(t.x && t.out_rows && t.row_scale && t.out_t && t.col_scale && t.workspace, MI8_ERR_ARG, "%s: tensor %d: null pointer", what, i);
        MI8_REQUIRE(valid_hp(t.hp_dtype), MI8_ERR_ARG, "%s: tensor %d: unknown hp dtype %d", what, i, t.hp_dtype);
        MI8_REQUIRE(t.rows > 0 && t.cols > 0 && t.rows < (1 << 30) && t.cols < (1 << 30), MI8_ERR_ARG, "%s: tensor %d: %lld x %lld", what, i,
                    (long long)t.rows, (long long)t.cols);
        MI8_REQUIRE(t.cols % 16 == 0, MI8_ERR_UNSUPPORTED, "%s: tensor %d: cols (%lld) must be a multiple of 16", what, i, (long long)t.cols);
        MI8_REQUIRE(aligned16(t.x) && aligned16(t.out_rows) && aligned16(t.out_t) && aligned16(t.workspace), MI8_ERR_UNSUPPORTED,
                    "%s: tensor %d: pointers must be 16-byte aligned", what, i);
        MI8_REQUIRE(t.ld_rows >= t.cols && t.ld_rows % 16 == 0, MI8_ERR_UNSUPPORTED, "%s: tensor %d: ld_rows (%lld)", what, i, (long long)t.ld_rows);
        MI8_REQUIRE(t.ld_t >= round_up(t.rows, kTile) && t.ld_t % 16 == 0, MI8_ERR_UNSUPPORTED,
                    "%s: tensor %d: ld_t (%lld) must be a multiple of 16 and at least the rows rounded up to 128", what, i, (long long)t.ld_t);
        MI8_REQUIRE(t.group_rows == 0 || (t.group_rows > 0 && t.group_rows % kTile == 0 && t.rows % t.group_rows == 0), MI8_ERR_UNSUPPORTED,
                    "%s: tensor %d: group_rows (%lld) must be a multiple of 128 that divides the rows (%lld)", what, i,
                    (long long)t.group_rows, (long long)t.rows);
    }
    TwoCastItems a{};
    a.count = count;
    a.pow2 = (flags & MI8_FLAG_POW2_SCALE) != 0;
    int64_t blocks = 0, chunk_blocks = 0, bytes = 0, end = 0;
    for (int i = 0; i < count; ++i) {
        const mi8_two_cast_item& t = items[i];
        const int64_t tiles_m = ceil_div(t.rows, kTile), tiles_n = ceil_div(t.cols, kTile);
        const int64_t group_tiles = t.group_rows ? t.group_rows / kTile : tiles_m;  // (of the rows that share column scales)
        const int chunk = chunk_tiles_for(group_tiles);
        const int64_t group_chunks = ceil_div(group_tiles, chunk), chunks = tiles_m / group_tiles * group_chunks;
        MI8_REQUIRE(blocks + tiles_m * tiles_n < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "%s: grid too large", what);
        a.t[i] = TwoCastItem{t.x, t.rows, t.cols, (uint8_t*)t.out_rows, t.ld_rows, t.row_scale, (uint8_t*)t.out_t, t.ld_t, t.col_scale,
                             t.workspace, t.workspace + chunks * tiles_n * kTile, t.hp_dtype == MI8_F32, (int)tiles_m, (int)tiles_n,
                             chunk, (int)group_tiles, (int)group_chunks, (int)blocks, (int)chunk_blocks};
        blocks += tiles_m * tiles_n;
        chunk_blocks += chunks * tiles_n;
        bytes += 2 * t.rows * t.cols;
        end = std::max({end, t.rows * t.ld_rows, t.cols * t.ld_t});
    }
    a.stream = streams_outputs(bytes, end);
    return launch_two_cast(a, fp8_dtype, (flags & MI8_FLAG_SW_CVT) != 0, chunk_blocks, blocks, (hipStream_t)stream, what);
}
