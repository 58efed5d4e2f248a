// Pieces shared by the amax and cast kernels: maxima of magnitudes, and the 128 x 128 tile that is read once, quantised and
// written row-major and transposed.
#pragma once
#include "mi8_common.h"

namespace mi8 {
namespace {

constexpr int kThreads = 256;

// ------------------------------------------------------------------------------------------------
// tensorwise amax -> per-workgroup partial maxima
// ------------------------------------------------------------------------------------------------

typedef unsigned short us2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_absmax_u16(uint32_t acc, uint32_t v)
{
    // two bf16 per dword: clear both sign bits, packed unsigned 16-bit max (v_pk_max_u16)
    us2 a = __builtin_bit_cast(us2, acc);
    us2 b = __builtin_bit_cast(us2, v & 0x7FFF7FFFu);
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(a, b));
}

template <int HP>
__device__ __forceinline__ void absmax_accumulate(uint4 v, uint32_t (&acc)[4])
{
    if constexpr (HP == MI8_BF16) {
        acc[0] = pk_absmax_u16(acc[0], v.x);
        acc[1] = pk_absmax_u16(acc[1], v.y);
        acc[2] = pk_absmax_u16(acc[2], v.z);
        acc[3] = pk_absmax_u16(acc[3], v.w);
    } else {
        acc[0] = umax32(acc[0], v.x & 0x7FFFFFFFu);
        acc[1] = umax32(acc[1], v.y & 0x7FFFFFFFu);
        acc[2] = umax32(acc[2], v.z & 0x7FFFFFFFu);
        acc[3] = umax32(acc[3], v.w & 0x7FFFFFFFu);
    }
}

// fold the four accumulators into one float32 |x| bit pattern
template <int HP>
__device__ __forceinline__ uint32_t absmax_fold(const uint32_t (&acc)[4])
{
    if constexpr (HP == MI8_BF16) {
        uint32_t m = pk_absmax_u16(pk_absmax_u16(acc[0], acc[1]), pk_absmax_u16(acc[2], acc[3]));
        uint32_t hi = m >> 16, lo = m & 0xFFFFu;
        return umax32(hi, lo) << 16;
    } else {
        return umax32(umax32(acc[0], acc[1]), umax32(acc[2], acc[3]));
    }
}

__device__ __forceinline__ uint32_t block_umax(uint32_t v, uint32_t* smem /* >= 4 words */)
{
    v = wave_umax(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) smem[wave] = v;
    __syncthreads();
    v = umax32(umax32(smem[0], smem[1]), umax32(smem[2], smem[3]));
    __syncthreads();
    return v;
}

constexpr int kTile = 128;

// Source row of logical row r when the casts read their input through a token permutation (the rows of a
// dropless-MoE expert batch: row r is the token that owns slot gather[r], top_k slots per token); -1 for a slot
// index outside [0, src_rows * top_k) - a dropped token, which reads as a row of zeros.
__device__ __forceinline__ int64_t gathered_row(const int32_t* gather, int top_k, int64_t src_rows, int64_t r, bool ok)
{
    if (!ok) return -1;
    const int32_t slot = gather[r];  // (src_rows * top_k < 2^31: a 32-bit division)
    return (slot < 0 || slot >= src_rows * top_k) ? -1 : (int64_t)((uint32_t)slot / (uint32_t)top_k);
}

// Weight of a slot of the weighted gather: the row is the token's row times this weight, the product rounded to the element type
// as the gather kernel does.
__device__ __forceinline__ float slot_weight(const void* w, int w_dtype, int64_t slot)
{
    if (w_dtype == MI8_F32) return reinterpret_cast<const float*>(w)[slot];
    const uint16_t v = reinterpret_cast<const uint16_t*>(w)[slot];
    return w_dtype == MI8_BF16 ? bits_to_f32((uint32_t)v << 16) : (float)__builtin_bit_cast(_Float16, v);
}

// the 16 bytes of a row times the row's gather weight, each product rounded to the element type
template <int HP>
__device__ __forceinline__ uint4 scale_vec(uint4 v, float w)
{
    uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (HP == MI8_BF16) {
            d[i] = pack_bf16(bits_to_f32(d[i] << 16) * w, bits_to_f32(d[i] & 0xFFFF0000u) * w);
        } else {
            d[i] = f32_to_bits(bits_to_f32(d[i]) * w);
        }
    }
    return make_uint4(d[0], d[1], d[2], d[3]);
}

// LDS holds the transposed tile as 128 columns x 128 row-bytes.  Two columns share a 256-byte line; the
// 16-byte chunk index inside the line is XORed with a function of the column's group of eight so that
// both the dword writes (lanes spread over 16 column groups x 4 row groups) and the 16-byte reads
// (lanes spread over 8 columns x 8 chunks) touch every bank once.
__device__ __forceinline__ int tile_lds_chunk(int col, int part /* 0..7: which 16 row-bytes */)
{
    const int grp = col >> 3;
    const int key = (((grp >> 3) & 1) << 3) | (grp & 7);
    return (col >> 1) * 16 + ((((col & 1) << 3) | part) ^ key);
}

// A thread's share of the 128 x 128 tile at (row0, col0) as it is in memory (bf16: half the registers of its values): rows
// 32 wave + 16 it + 4 (lane / 16) + j, eight columns from 8 (lane % 16); rows >= row_end and columns >= cols read as zero.
// The loads need nothing but the position, so that they can be in flight while the scales are made.
// GATHER: row r is row src[r - row0] of x, a row of zeros where that is negative.
template <int HP>
struct RawTile {
    static constexpr int NV = HpVec<HP>::kBytes / 2;  // 16-byte vectors per eight elements
    uint4 v[2][4][NV];
    __device__ __forceinline__ static int row_of(int it, int j) { return 32 * ((int)threadIdx.x >> 6) + 16 * it + 4 * (((int)threadIdx.x & 63) >> 4) + j; }
    template <bool GATHER = false>
    __device__ __forceinline__ void load(const void* x, int64_t row_end, int64_t cols, int64_t row0, int64_t col0, const int32_t* src = nullptr)
    {
        const int64_t c8 = col0 + 8 * (threadIdx.x & 15);
        const char* xb = reinterpret_cast<const char*>(x);
#pragma unroll
        for (int it = 0; it < 2; ++it)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t r = row0 + row_of(it, j);
                const int64_t from = GATHER ? (int64_t)src[row_of(it, j)] : r;
                const bool ok = c8 < cols && r < row_end && from >= 0;
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    v[it][j][k] = make_uint4(0, 0, 0, 0);
                    const char* p = xb + (from * cols + c8) * HpVec<HP>::kBytes + 16 * k;
                    // (gathered: a token's row is read top_k times, it stays cached)
                    if (ok) v[it][j][k] = GATHER ? *reinterpret_cast<const uint4*>(p) : load_stream16(p);
                }
            }
    }
    // the weighted gather's product; weights[row]: 1 for a row of zeros
    __device__ __forceinline__ void scale_rows(const float* weights, bool col_ok)
    {
#pragma unroll
        for (int it = 0; it < 2; ++it)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int k = 0; k < NV; ++k)
                    if (col_ok) v[it][j][k] = scale_vec<HP>(v[it][j][k], weights[row_of(it, j)]);
    }
    __device__ __forceinline__ void operator()(int it, int j, float (&f)[8]) const
    {
        const uint4 a = v[it][j][0], b = v[it][j][NV - 1];
        if constexpr (HP == MI8_BF16) {
            const uint32_t d[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f[2 * k] = bits_to_f32(d[k] << 16);
                f[2 * k + 1] = bits_to_f32(d[k] & 0xFFFF0000u);
            }
        } else {
            const uint32_t d[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) f[k] = bits_to_f32(d[k]);
        }
    }
};

// Quantise a loaded tile (values(it, j, f): a thread's eight of row 16 it + j) with the eight per-column scales of this lane
// (all equal for a tensorwise cast).
// Row-major bytes go to out[r, c]; the transposed bytes go to out_t[c, dst0 + (r - row0)] as 16-byte chunks,
// chunks at or beyond dst_end are not written.  stream: see streams_outputs.
template <int FP8, bool SW, typename Values>
__device__ __forceinline__ void tile_quantise(const Values& values, int64_t row_end, int64_t cols, int64_t row0, int64_t col0,
                                              const float (&sc)[8], uint8_t* out, int64_t ld_out, uint8_t* out_t, int64_t ld_t,
                                              int64_t dst0, int64_t dst_end, uint32_t* lds_t,
                                              bool stream, uint8_t* out_r = nullptr, int64_t ld_r = 0, const float* row_scale = nullptr,
                                              int64_t row_scale_row0 = 0)
{
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int cl = lane & 15, g = lane >> 4;
    const int64_t c8 = col0 + 8 * cl;
    const bool col_ok = c8 < cols;

    // the rows' own scales, read ahead of the stores below (a read placed between them would wait for them)
    float srow[2][4];
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t r = row0 + 32 * wave + 16 * it + 4 * g + j;
            srow[it][j] = (out_r && r < row_end) ? row_scale[r - row_scale_row0] : 0.0f;  // (row_scale[0] = row row_scale_row0)
        }

#pragma unroll
    for (int it = 0; it < 2; ++it) {
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t r = row0 + 32 * wave + 16 * it + 4 * g + j;
            const bool ok = col_ok && r < row_end;
            float v[8];
            values(it, j, v);
            lo[j] = quant4<FP8, SW>(v[0], v[1], v[2], v[3], sc[0], sc[1], sc[2], sc[3]);
            hi[j] = quant4<FP8, SW>(v[4], v[5], v[6], v[7], sc[4], sc[5], sc[6], sc[7]);
            if (!ok) lo[j] = hi[j] = 0;  // padding is zero bytes whatever the scale is (0 * NaN is NaN)
            if (out && ok) store_out8(out, r * ld_out + c8, lo[j], hi[j], stream);
            if (out_r && ok) {  // the same values quantised with the row's own scale
                const float sr = srow[it][j];
                const uint32_t rl = quant4<FP8, SW>(v[0], v[1], v[2], v[3], sr, sr, sr, sr);
                const uint32_t rh = quant4<FP8, SW>(v[4], v[5], v[6], v[7], sr, sr, sr, sr);
                store_out8(out_r, r * ld_r + c8, rl, rh, stream);
            }
        }
        if (out_t) {
            uint32_t t[8];
            transpose4x4_bytes(lo[0], lo[1], lo[2], lo[3], t[0], t[1], t[2], t[3]);
            transpose4x4_bytes(hi[0], hi[1], hi[2], hi[3], t[4], t[5], t[6], t[7]);
            const int rd = 8 * wave + 4 * it + g;  // which dword of the column's 32 row-dwords
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int col = 8 * cl + i;
                lds_t[tile_lds_chunk(col, rd >> 2) * 4 + (rd & 3)] = t[i];
            }
        }
    }

    if (out_t) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = tid + kThreads * i;
            const int col = q >> 3, part = q & 7;
            const uint4 v = reinterpret_cast<const uint4*>(lds_t)[tile_lds_chunk(col, part)];
            const int64_t c = col0 + col;
            const int64_t d = dst0 + 16 * part;
            if (c < cols && d < dst_end) store_out16(out_t, c * ld_t + d, v, stream);
        }
    }
}

}  // namespace
}  // namespace mi8
