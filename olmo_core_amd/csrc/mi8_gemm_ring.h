// The fp8 GEMM tile routine for everything the persistent kernel (mi8_gemm_m16.hip) is too coarse for: any M, N,
// K % 16 == 0, bf16 or fp32 output, single scales or scale vectors; shared by the dense, split-K and grouped kernels.
//
// What bounds it: these are products with fewer tiles than fill the chip once or twice at 256 x 256, so a tile's time is
// latency (the first operand bytes, one barrier and one LDS round trip per 128-byte K step, the epilogue) and, once two
// workgroups share a compute unit, the operand bytes that come out of L2: (BM + BN) * 128 per step at about 80 B/ns and
// compute unit.  Hence small tiles (32 to 128 rows by 64 or 128 columns, four waves of (BM / 2) x (BN / 2)), operands that go from L2
// straight to LDS (buffer loads with the LDS destination, no registers and no vector address arithmetic: one resident
// lane offset per load and a uniform K offset), a ring of ST stages so that ST - 1 steps are in flight, and an LDS
// footprint that lets two workgroups live on a compute unit, one computing while the other waits.
//
// A step's fragments are read from LDS during the step before (two sets of registers), so that the reads (0.37 us a step of
// a 128 x 128 tile) and the MFMAs (0.23 us) run side by side: what bounds a step is then the operands' way out of L2, 0.27 us
// with few compute units busy and 0.40 with all of them, where it took 0.60 with the reads between a barrier and the MFMAs.
// Tiles that share a compute unit in pairs (two stages), or that have no registers left (256 x 256), keep one set:
// there the other workgroup or wave fills the gap.
//
// The MFMA (v_mfma_f32_16x16x128_f8f6f4), the order of K and the scale arithmetic are those of the persistent kernel: a
// product has the same bits on either.  us per launch in a graph, one set of fragments / two: 777 x 4096 x 11008 55.8 / 41.1
// (128 x 128), 1537 x 2048 x 2048 14.8 / 11.3, 1999 x 1024 x 2816 12.9 / 10.0 (64 x 128), 200 x 4096 x 4096 12.1 / 9.3 (64 x 64).
// 256 x 256 tiles at 16384 x 4096 x 11024: matrix pipe busy 59 %, bank conflicts 2 % of the LDS cycles, operands fetched into
// L2 4.8 times.
//
// LDS stage: [row][128 bytes], A rows then B rows; 16-byte chunk c of row r sits at c ^ swz16(r) (the swizzle of the
// persistent kernel), applied by permuting which global chunk a lane fetches.
#pragma once
#include <type_traits>

#include "mi8_gemm.h"
#include "mi8_swiglu.h"

namespace mi8 {
namespace gemm {
namespace {

typedef float ring_v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* ring_lds_t;
typedef const __attribute__((address_space(3))) v4i* ring_frag_t;

// 16 bytes per lane from a raw buffer into LDS at dst + 16 * lane (dst uniform); lanes past the descriptor's end write zeros
__device__ __forceinline__ void ring_load(__amdgpu_buffer_rsrc_t d, uint8_t* dst, int lane_offset, int offset)
{
#ifdef __HIP_DEVICE_COMPILE__  // (the builtin exists in the device pass only)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(d, (ring_lds_t)dst, 16, lane_offset, offset, 0, 0);
#endif
}

// all but the last N vector memory operations and every LDS operation of this wave have completed
template <int N>
__device__ __forceinline__ void ring_wait()
{
    static_assert(N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70);
}

// the same for all but the loads of `steps` steps (0 .. MOST) of LD loads each
template <int LD, int MOST>
__device__ __forceinline__ void ring_wait_steps(int steps)
{
    if constexpr (MOST == 0) {
        ring_wait<0>();
    } else {
        if (steps >= MOST)
            ring_wait<LD * MOST>();
        else
            ring_wait_steps<LD, MOST - 1>(steps);
    }
}

template <int BM, int BN, int ST>
constexpr int kRingLdsBytes = ST * (BM + BN) * BK;

constexpr int kRingThreads = 256;

// C[m0 .. m0 + BM, n0 .. n0 + BN] of g's product (K may be 0: zeros).  g.sa == null: the raw fp32 sums are wanted.
// SLICED: K is summed in slices of g.slice_steps, each from zero, added in order (the sums of split K without its planes).
// NW waves, two of them side by side along M.
// DUAL (32 or 64 rows by 64 B rows, single scales): C[.., n0 .. n0 + 32] = silu(A B^T) * (A B3^T).  B rows 32 w .. of the stage, those of the
// wave column w, are 16 rows of B and the same 16 of B3, so that a lane holds both products of the same elements.
template <int BM, int BN, int ST, int CBSZ, int BLGP, bool SLICED = false, int NW = kRingThreads / 64, bool DUAL = false>
__device__ __forceinline__ void ring_tile(const GemmArgs& g, const int m0, const int n0, uint8_t* lds)
{
    constexpr int WAVES_N = NW / 2;
    constexpr int WTM = BM / 2, WTN = BN / WAVES_N;  // wave tile
    constexpr int TM = WTM / 16, TN = WTN / 16;
    constexpr int STAGE = (BM + BN) * BK;
    constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW, LD = LA + LB;  // loads per wave and step: 8 rows x 128 bytes each
    static_assert(LA * 8 * NW == BM && LB * 8 * NW == BN && ST >= 2 && LD * (ST - 1) < 64, "tile shape");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int r16 = lane & 15, kb = lane >> 4;

    // ---- operand loads: load i of wave w fills rows 8 (NW i + w) .. + 7; rows past the edge re-read the last one
    constexpr int BNC = DUAL ? BN / 2 : BN;  // columns of C
    static_assert(!DUAL || (BM <= 64 && BN == 64 && NW == 4 && TN == 2), "dual tile shape");
    const int rows_a = g.M - m0 < BM ? g.M - m0 : BM, rows_b = g.N - n0 < BNC ? g.N - n0 : BNC;
    const uint8_t* const b_base = DUAL && (wave & 2) ? g.B3 : g.B;  // (a wave's loads of B are of one matrix)
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(g.A + (int64_t)m0 * g.lda), 0, (int)(uint32_t)((int64_t)(rows_a - 1) * g.lda + g.K), 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(b_base + (int64_t)n0 * g.ldb), 0, (int)(uint32_t)((int64_t)(rows_b - 1) * g.ldb + g.K), 0x00020000);
    const int lr = lane >> 3, chunk16 = ((lane & 7) ^ swz16(lr)) * 16;
    int off[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {
        const bool is_a = i < LA;
        int r = 8 * (NW * (is_a ? i : i - LA) + wave) + lr;
        if (DUAL && !is_a) r = 16 * (r >> 5) + (r & 15);
        const int last = (is_a ? rows_a : rows_b) - 1;
        r = r < last ? r : last;
        off[i] = (int)((uint32_t)r * (uint32_t)(is_a ? g.lda : g.ldb)) + chunk16;
    }
    const int nk = (g.K + BK - 1) / BK;
    const bool ragged = g.K < nk * BK;
    auto issue_one = [&](int i, int k, int slot) __attribute__((always_inline)) {
        const bool is_a = i < LA;
        ring_load(is_a ? da : db, lds + slot * STAGE + ((is_a ? 0 : BM) + 8 * (NW * (is_a ? i : i - LA) + wave)) * BK, off[i], k * BK);
    };
    auto issue = [&](int k, int slot) __attribute__((always_inline)) {
        uint8_t* st = lds + slot * STAGE;
        const int at = k * BK;
        if (ragged && k == nk - 1) {  // bytes past K are fed as zeros: those lanes point past the descriptor's end
#pragma unroll
            for (int i = 0; i < LD; ++i) {
                const bool is_a = i < LA;
                ring_load(is_a ? da : db, st + ((is_a ? 0 : BM) + 8 * (NW * (is_a ? i : i - LA) + wave)) * BK,
                          at + chunk16 < g.K ? off[i] + at : (int)0xFFFFFFF0, 0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < LD; ++i) issue_one(i, k, slot);
        }
    };

    // ---- fragment reads: half q of a lane's 32 K bytes; MFMA tile t adds 2048 t
    uint32_t fa_at[2], fb_at[2];
    {
        const uint32_t lds0 = (uint32_t)(uintptr_t)(ring_lds_t)lds;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t chunk = (uint32_t)((2 * kb + q) ^ swz16(r16)) << 4;
            fa_at[q] = lds0 + (uint32_t)((wm * WTM + r16) * BK) + chunk;
            fb_at[q] = lds0 + (uint32_t)((BM + wn * WTN + r16) * BK) + chunk;
        }
    }

    ring_v4f acc[TM][TN], sum[SLICED ? TM : 1][SLICED ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = (ring_v4f){0, 0, 0, 0};
    int slice_left = g.slice_steps;
    if constexpr (SLICED) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) sum[i][j] = (ring_v4f){0, 0, 0, 0};
    }

    // x-th fragment register pair of a step: halves q = 0, 1 of the A tiles, then of the B tiles
    struct ReadAt { uint32_t a[2], b[2]; };
    auto read_at = [&](int slot) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t)(slot * STAGE);
        ReadAt r{{fa_at[0] + at, fa_at[1] + at}, {fb_at[0] + at, fb_at[1] + at}};
        asm volatile("" : "+v"(r.a[0]), "+v"(r.a[1]), "+v"(r.b[0]), "+v"(r.b[1]));  // (the tiles' offsets go into the instructions)
        return r;
    };
    auto read_one = [&](v4i (&fa)[TM][2], v4i (&fb)[TN][2], int x, const ReadAt& r) __attribute__((always_inline)) {
        const int t = x >> 1, q = x & 1;
        if (t < TM)
            fa[t][q] = *reinterpret_cast<ring_frag_t>((uintptr_t)(r.a[q] + t * 16 * BK));
        else
            fb[t - TM][q] = *reinterpret_cast<ring_frag_t>((uintptr_t)(r.b[q] + (t - TM) * 16 * BK));
    };
    // D' = B . A^T: the first operand is the B fragment (its type code goes to cbsz)
    auto mma_one = [&](const v4i (&fa)[TM][2], const v4i (&fb)[TN][2], int x) __attribute__((always_inline)) {
        const int i = x / TN, j = x % TN;
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
            __builtin_shufflevector(fb[j][0], fb[j][1], 0, 1, 2, 3, 4, 5, 6, 7),
            __builtin_shufflevector(fa[i][0], fa[i][1], 0, 1, 2, 3, 4, 5, 6, 7), acc[i][j], BLGP, CBSZ, 0, 0, 0, 0);
    };
    auto end_of_step = [&]() __attribute__((always_inline)) {
        if constexpr (SLICED) {
            if (--slice_left == 0) {
                slice_left = g.slice_steps;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        sum[i][j] += acc[i][j];
                        acc[i][j] = (ring_v4f){0, 0, 0, 0};
                    }
            }
        }
    };
    constexpr int kMma = TM * TN, kReads = 2 * (TM + TN);
    // Two sets of fragments: a step multiplies from one while the next step's are read into the other, and the loads of step
    // k + ST go into the slot of step k, whose fragments have all been read.
    constexpr bool kTwoSets = ST > 2 && 8 * kReads + 4 * kMma * (SLICED ? 2 : 1) <= 192;
    if constexpr (kTwoSets) {
        v4i fa[2][TM][2], fb[2][TN][2];
        int slot = 0;
        auto k_step = [&](int k, auto set_tag, auto steady_tag) __attribute__((always_inline)) {
            constexpr int S = decltype(set_tag)::value;
            auto body = [&](auto with_reads, auto with_loads) __attribute__((always_inline)) {
                const ReadAt at = read_at(slot == ST - 1 ? 0 : slot + 1);
#pragma unroll
                for (int x = 0; x < kMma; ++x) {
                    mma_one(fa[S], fb[S], x);
                    if constexpr (decltype(with_reads)::value) {
#pragma unroll
                        for (int y = x * kReads / kMma; y < (x + 1) * kReads / kMma; ++y) read_one(fa[S ^ 1], fb[S ^ 1], y, at);
                    }
                    if constexpr (decltype(with_loads)::value) {
#pragma unroll
                        for (int y = x * LD / kMma; y < (x + 1) * LD / kMma; ++y) issue_one(y, k + ST, slot);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // this wave's fragments of step k have arrived and its loads of step k + 1 have landed (those of up to ST - 2
            // later steps may be in flight); after the barrier every wave's
            constexpr bool kSteady = decltype(steady_tag)::value;
            const int ahead = kSteady ? ST - 2 : nk - 2 - k;
            ring_wait_steps<LD, ST - 2>(ahead);
            asm volatile("s_barrier" ::: "memory");
            if constexpr (kSteady) {
                body(std::true_type{}, std::true_type{});
            } else {
                if (k + ST < nk) issue(k + ST, slot);
                if (k + 1 < nk)
                    body(std::true_type{}, std::false_type{});
                else
                    body(std::false_type{}, std::false_type{});
            }
            slot = slot == ST - 1 ? 0 : slot + 1;
            end_of_step();
        };
        if (nk > 0) {
#pragma unroll
            for (int s = 0; s < ST; ++s)
                if (s < nk) issue(s, s);
            ring_wait_steps<LD, ST - 1>(nk - 1);
            asm volatile("s_barrier" ::: "memory");
            const ReadAt at = read_at(0);
#pragma unroll
            for (int x = 0; x < kReads; ++x) read_one(fa[0], fb[0], x, at);
        }
        const std::integral_constant<int, 0> set0;
        const std::integral_constant<int, 1> set1;
        int k = 0;
        for (; k + 1 + ST < nk - (ragged ? 1 : 0); k += 2) {  // both steps have whole loads to issue
            k_step(k, set0, std::true_type{});
            k_step(k + 1, set1, std::true_type{});
        }
        for (; k + 1 < nk; k += 2) {
            k_step(k, set0, std::false_type{});
            k_step(k + 1, set1, std::false_type{});
        }
        if (k < nk) k_step(k, set0, std::false_type{});
    } else {
#pragma unroll
        for (int s = 0; s < ST - 1; ++s)
            if (s < nk) issue(s, s);
        int slot = 0;
        for (int k = 0; k < nk; ++k) {
            // this wave's loads of step k have landed (those of up to ST - 2 later steps may be in flight) ...
            ring_wait_steps<LD, ST - 2>(nk - 1 - k);
            // ... every wave's have, and every wave has its fragments of step k - 1, whose slot is filled next
            asm volatile("s_barrier" ::: "memory");
            if (k + ST - 1 < nk) issue(k + ST - 1, slot == 0 ? ST - 1 : slot - 1);
            const ReadAt at = read_at(slot);
            v4i fa[TM][2], fb[TN][2];
#pragma unroll
            for (int x = 0; x < kReads; ++x) read_one(fa, fb, x, at);
#pragma unroll
            for (int x = 0; x < kMma; ++x) mma_one(fa, fb, x);
            slot = slot == ST - 1 ? 0 : slot + 1;
            end_of_step();
        }
    }
    if constexpr (SLICED) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j] + acc[i][j];
    }

    if constexpr (DUAL) {
        const float isa = 1.0f / g.sa[0], f1 = isa * (1.0f / g.sb[0]), f3 = isa * (1.0f / g.sb3[0]);
        const int col = n0 + 16 * wn + 4 * kb;  // (N % 8 == 0)
        uint32_t hm = 0;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = m0 + wm * WTM + 16 * i + r16;
            const ring_v4f x1 = acc[i][0], x3 = acc[i][TN - 1];
            const uint2 h = swiglu_fwd4(make_uint2(pack_bf16x2(x1[0] * f1, x1[1] * f1), pack_bf16x2(x1[2] * f1, x1[3] * f1)),
                                        make_uint2(pack_bf16x2(x3[0] * f3, x3[1] * f3), pack_bf16x2(x3[2] * f3, x3[3] * f3)));
            if (row < g.M && col < g.N) {
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.C) + (int64_t)row * g.ldc + col) = h;
                hm = umax32(hm, (max_code8(h.x, h.y, h.x, h.y) & 0xFFFFu) << 16);
            }
        }
        hm = wave_umax(hm);
        __syncthreads();  // (the ring is free now)
        uint32_t* maxima = reinterpret_cast<uint32_t*>(lds);
        if (lane == 0) maxima[wave] = hm;
        __syncthreads();
        if (tid == 0) g.slots_out[n0 / BNC] = umax32(umax32(maxima[0], maxima[1]), umax32(maxima[2], maxima[3]));
        return;
    }
    // ---- epilogue: acc[i][j][e] of lane l is C[row = 16 i + l % 16][col = 16 j + 4 (l / 16) + e] of the wave tile.
    // Single scales are inverted with an IEEE division, scale vectors with v_rcp_f32 (exact for the power-of-two scales
    // of the axiswise recipes, within 1 ulp otherwise).
    const int row0 = m0 + wm * WTM + r16, col0 = n0 + wn * WTN + 4 * kb;
    const float isa1 = g.sa && !g.sa_vec ? 1.0f / g.sa[0] : 1.0f, isb1 = g.sb && !g.sb_vec ? 1.0f / g.sb[0] : 1.0f;
    const bool both_single = !g.sa_vec && !g.sb_vec;
    float isb[TN][4];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            isb[j][e] = g.sb_vec ? (col0 + 16 * j + e < g.N ? __builtin_amdgcn_rcpf(g.sb[col0 + 16 * j + e]) : 0.0f) : isb1;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = row0 + 16 * i;
        const float isa = g.sa_vec ? (row < g.M ? __builtin_amdgcn_rcpf(g.sa[row]) : 0.0f) : isa1;
        const float one = isa1 * isb1;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = both_single ? acc[i][j][e] * one : acc[i][j][e] * isa * isb[j][e];
    }
    if (g.c_f32 == 2) {  // (uniform)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] = round_to_bf16(acc[i][j][e]);
    }
    const bool wide = (reinterpret_cast<uintptr_t>(g.C) & 15) == 0 && ((g.ldc | g.N) & (g.c_f32 ? 3 : 7)) == 0;
    if (!wide) {
        // Rows that are not whole 16-byte chunks leave an element per lane, or four bf16 values where rows are whole 8-byte
        // chunks, consecutive lanes on consecutive columns (16 rows of the wave tile at a time through LDS; the ring is free
        // now).  Stored from the accumulators, whose lanes hold 16 rows of four columns each, 14592 x 3967 x 1040 in float32
        // took 188 us where this takes 127, 65536 rows in 32 groups x 1020 x 1024 213 where this takes 153.
        const bool quads = !g.c_f32 && ((g.ldc | g.N) & 3) == 0 && (reinterpret_cast<uintptr_t>(g.C) & 7) == 0;
        constexpr int PITCH = WTN + 4;
        static_assert(NW * 16 * PITCH * 4 <= ST * STAGE, "output staging");
        __syncthreads();
        float* stg = reinterpret_cast<float*>(lds) + wave * (16 * PITCH);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j) *reinterpret_cast<ring_v4f*>(stg + r16 * PITCH + 16 * j + 4 * kb) = acc[i][j];
            if (quads) {
                constexpr int QPR = WTN / 4;
#pragma unroll
                for (int it = 0; it < 16 * QPR / 64; ++it) {
                    const int rw = (it * 64 + lane) / QPR, cw = lane % QPR * 4;
                    const ring_v4f v = *reinterpret_cast<const ring_v4f*>(stg + rw * PITCH + cw);
                    const int row = m0 + wm * WTM + 16 * i + rw, col = n0 + wn * WTN + cw;
                    if (row >= g.M || col >= g.N) continue;
                    uint2* c = reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.C) + (int64_t)row * g.ldc + col);
                    uint2 r = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                    if (g.accumulate) r = make_uint2(add_bf16x2(r.x, c->x), add_bf16x2(r.y, c->y));
                    *c = r;
                }
                continue;
            }
#pragma unroll
            for (int it = 0; it < 16 * WTN / 64; ++it) {
                const int rw = (it * 64 + lane) / WTN, cw = lane % WTN;
                const float v = stg[rw * PITCH + cw];
                const int row = m0 + wm * WTM + 16 * i + rw, col = n0 + wn * WTN + cw;
                if (row >= g.M || col >= g.N) continue;
                const int64_t at = (int64_t)row * g.ldc + col;
                if (g.c_f32) {
                    float* c = reinterpret_cast<float*>(g.C) + at;
                    *c = g.accumulate ? *c + v : v;
                } else {
                    uint16_t* c = reinterpret_cast<uint16_t*>(g.C) + at;
                    uint16_t r = f32_to_bf16_bits(v);
                    if (g.accumulate)
                        r = f32_to_bf16_bits(bits_to_f32((uint32_t)*c << 16) + bits_to_f32((uint32_t)r << 16));
                    *c = r;
                }
            }
        }
        return;
    }
    if (g.c_f32) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = row0 + 16 * i;
            if (row >= g.M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = col0 + 16 * j;
                if (col >= g.N) continue;
                ring_v4f* c = reinterpret_cast<ring_v4f*>(reinterpret_cast<float*>(g.C) + (int64_t)row * g.ldc + col);
                *c = g.accumulate ? *c + acc[i][j] : acc[i][j];
            }
        }
        return;
    }
    uint16_t* C = reinterpret_cast<uint16_t*>(g.C);
    // bf16 rows leave through LDS (the ring is free now): whole row segments of the wave tile, 16 bytes per lane
    constexpr int PITCH = WTN * 2 + 16;  // (the pad spreads the rows of a store over the banks)
    constexpr int SR = NW * WTM * PITCH <= ST * STAGE ? WTM : WTM / 2;  // rows of the wave tile staged at a time
    static_assert(NW * SR * PITCH <= ST * STAGE, "output staging");
    __syncthreads();
    uint8_t* stg = lds + wave * (SR * PITCH);
    constexpr int LPR = WTN / 8, RPI = 64 / LPR;  // lanes per row, rows per store
#pragma unroll
    for (int part = 0; part < WTM / SR; ++part) {
#pragma unroll
        for (int i = 0; i < SR / 16; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const ring_v4f v = acc[part * (SR / 16) + i][j];
                *reinterpret_cast<uint2*>(stg + (16 * i + r16) * PITCH + (16 * j + 4 * kb) * 2) =
                    make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
            }
#pragma unroll
        for (int it = 0; it < SR / RPI; ++it) {
            const int rw = it * RPI + lane / LPR, c8 = (lane % LPR) * 8;
            v4i v = *reinterpret_cast<const v4i*>(stg + rw * PITCH + c8 * 2);
            const int row = m0 + wm * WTM + part * SR + rw, col = n0 + wn * WTN + c8;
            if (row < g.M && col < g.N) {
                v4i* c = reinterpret_cast<v4i*>(C + (int64_t)row * g.ldc + col);
                if (g.accumulate) v = add_bf16x8(v, *c);
                *c = v;
            }
        }
    }
}

}  // namespace
}  // namespace gemm
}  // namespace mi8
