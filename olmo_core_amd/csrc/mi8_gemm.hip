// Scaled float8 GEMM on CDNA4 matrix cores:  C[M,N] = bf16( (A[M,K] . B[N,K]^T) * (1/sa) * (1/sb) ).
//
// Both operands are K-contiguous ("TN"), which is what the fp8 MFMAs want: every lane feeds 32 consecutive K bytes of
// one row.
//
// This file holds the kernels over the general tile routine of mi8_gemm_ring.h (any M, N; K % 16 == 0; bf16 or fp32
// output), their split-K form for problems with few output tiles, and the entry points, which pick a kernel by shape:
// the persistent direct-to-LDS kernel of mi8_gemm_m16.hip for large problems, the weight-streaming kernel of
// mi8_gemm_skinny.hip for a few rows of A.
#include "mi8_gemm_ring.h"

namespace mi8 {
using namespace gemm;
namespace {

template <int BM, int BN, int ST, int OCC, int CBSZ, int BLGP, bool SLICED, int NW>
__global__ __launch_bounds__(NW * 64, OCC) void gemm_fp8_ring_kernel(GemmArgs g)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    int tm, tn;
    if (!tile_of_block(g, tm, tn)) return;
    ring_tile<BM, BN, ST, CBSZ, BLGP, SLICED, NW>(g, tm * BM, tn * BN, lds);
}

// A few rows through both input projections of a SwiGLU block and the activation (see ring_tile); K in eighths.  Bound by
// reading the weights, 3.7 TB/s at 90 MB and 5.0 at 283 (weights from HBM; six stages instead of four change nothing).
template <int BM>
__global__ __launch_bounds__(kRingThreads, BM == 32 ? 3 : 2) void dual_ring_kernel(GemmArgs g)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    int tm, tn;
    if (!tile_of_block(g, tm, tn)) return;
    ring_tile<BM, 64, 4, 0, 0, true, kRingThreads / 64, true>(g, 0, tn * 32, lds);
}

// ---- split K ---------------------------------------------------------------------------------------
// A problem with few output tiles and a long K leaves most compute units idle while every busy one pays a
// memory latency per 128-byte K step.  Here blockIdx.y cuts K into slices: every (tile, slice) workgroup runs
// the same tile routine on its slice (operand pointers moved along the rows, which are K-contiguous) and stores
// the raw fp32 sums into its own plane of a workspace; a second kernel adds the planes in a fixed order (the
// result does not depend on scheduling), applies the scales and rounds.

struct SplitArgs {
    GemmArgs g;          // the problem; C, ldc, scales describe the final output
    float* planes;       // [splits][M][ld_plane] fp32
    int64_t ld_plane;    // round_up(N, 4)
    int steps_per_split; // 128-byte K steps per slice; the last slice may be shorter, none is empty
    int splits;
};

template <int BM, int BN, int ST, int OCC, int CBSZ, int BLGP>
__global__ __launch_bounds__(kRingThreads, OCC) void gemm_fp8_splitk_kernel(SplitArgs a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    GemmArgs g = a.g;
    int tm, tn;
    if (!tile_of_block(g, tm, tn)) return;
    const int split = (int)blockIdx.y;
    const int k0 = split * a.steps_per_split * BK;
    const int left = g.K - k0;
    g.A += k0;
    g.B += k0;
    g.K = left < a.steps_per_split * BK ? left : a.steps_per_split * BK;
    g.C = a.planes + (int64_t)split * g.M * a.ld_plane;
    g.c_f32 = 1;
    g.accumulate = 0;
    g.ldc = a.ld_plane;
    g.sa = g.sb = nullptr;
    g.sa_vec = g.sb_vec = 0;
    ring_tile<BM, BN, ST, CBSZ, BLGP>(g, tm * BM, tn * BN, lds);
}

// out[m][n] (+)= round( (sum over planes, in plane order) * (1/sa) * (1/sb) ); four columns per thread.  Bound by the
// latency of the plane reads: kInFlight are in flight at a time, seven where there are more than four planes, so that eight
// are one round of reads (one after the other: 7-11 us where this takes 4-5).
template <int kInFlight>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(SplitArgs a)
{
    const GemmArgs& g = a.g;
    const int64_t quads_per_row = a.ld_plane / 4;
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= (int64_t)g.M * quads_per_row) return;
    const int m = (int)(q / quads_per_row);
    const int n = (int)(q % quads_per_row) * 4;
    const int64_t plane = (int64_t)g.M * a.ld_plane;
    const float* p = a.planes + (int64_t)m * a.ld_plane + n;
    ring_v4f s = *reinterpret_cast<const ring_v4f*>(p);
    for (int i = 1; i < a.splits; i += kInFlight) {
        ring_v4f t[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
            if (i + u < a.splits) t[u] = *reinterpret_cast<const ring_v4f*>(p + (i + u) * plane);
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
            if (i + u < a.splits) s += t[u];
    }
    // same scale arithmetic as the tile routine's own epilogue
    const float isa = g.sa_vec ? __builtin_amdgcn_rcpf(g.sa[m]) : 1.0f / g.sa[0];
    const float isb_single = g.sb_vec ? 0.0f : 1.0f / g.sb[0];
    const bool both_single = !g.sa_vec && !g.sb_vec;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (n + j >= g.N) break;
        const float isb = g.sb_vec ? __builtin_amdgcn_rcpf(g.sb[n + j]) : isb_single;
        float r = both_single ? s[j] * (isa * isb) : s[j] * isa * isb;
        if (g.c_f32 == 2) r = round_to_bf16(r);
        if (g.c_f32) {
            float* c = reinterpret_cast<float*>(g.C) + (int64_t)m * g.ldc + n + j;
            *c = g.accumulate ? *c + r : r;
        } else {
            uint16_t* c = reinterpret_cast<uint16_t*>(g.C) + (int64_t)m * g.ldc + n + j;
            uint16_t h = f32_to_bf16_bits(r);
            if (g.accumulate) h = f32_to_bf16_bits(bits_to_f32((uint32_t)*c << 16) + bits_to_f32((uint32_t)h << 16));
            *c = h;
        }
    }
}

// ---- several products in one launch ------------------------------------------------------------------
// A layer of ordinary size is a handful of products that each fill a part of the chip for 10-20 us, of which a launch of
// their own wastes the start, the last round of tiles and the way to the next one.  Here the tiles of all of them form one
// grid.  A product may add to the one before it (C += product, the terms of a grad_input): then one workgroup runs the
// chain on its tile, so that every element is read and written by one lane, in order.  Every product's tiles are dealt to
// the XCDs by themselves (an eighth each, contiguous), since products differ in length.
struct BatchArgs {
    GemmArgs g[MI8_GEMM_BATCH];
    int next[MI8_GEMM_BATCH];            // the product that adds to this one's output, or -1
    int first_slot[MI8_GEMM_BATCH + 1];  // tiles per XCD before the i-th chain
    int head[MI8_GEMM_BATCH];            // first product of the i-th chain
    int chains;
};

template <int BM, int BN, int ST, int OCC, int CBSZ, int BLGP, bool SLICED>
__global__ __launch_bounds__(kRingThreads, OCC) void gemm_fp8_batch_kernel(BatchArgs a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
    int c = 0;
#pragma unroll
    for (int i = 1; i < MI8_GEMM_BATCH; ++i)
        if (i < a.chains && slot >= a.first_slot[i]) c = i;
    const int per_xcd = a.first_slot[c + 1] - a.first_slot[c];
    const int t = xcd * per_xcd + slot - a.first_slot[c];
    int i = a.head[c];
    if (t >= a.g[i].tiles_m * a.g[i].tiles_n) return;
    int tm, tn;
    tile_coords(a.g[i], t, tm, tn);
    for (;;) {
        ring_tile<BM, BN, ST, CBSZ, BLGP, SLICED>(a.g[i], tm * BM, tn * BN, lds);
        i = a.next[i];
        if (i < 0) break;
        __syncthreads();  // the output staging has been read
    }
}

// ---- tile shapes of the ring kernels and what a problem costs on them ---------------------------------------------

struct RingShape {
    const char* name;
    int bm, bn;
    float step0, step1;  // us per 128-byte K step with one workgroup on a compute unit: few units busy .. all of them
    float step2;         // ... and for a pair of them sharing one (0: only one fits)
    float tile;          // us per tile outside the K loop
    float many, many_tile;  // step (of one or of the pair) and tile where units get three tiles and more: operands from further away
};

// (fitted to 113 products each, 65 x 768 x 2048 to 1999 x 5632 x 1024 and 700 x 5120 x 27648, which the model below meets
// within 5-8 % rms, the shape it picks on average 1 % behind the fastest; the last two to products up to 16384 x 11008 x 4112)
constexpr RingShape kRing[] = {
    {"64x64_ring4", 64, 64, 0.113f, 0.181f, 0.335f, 1.33f, 0.39f, 1.2f},
    {"128x64_ring3", 128, 64, 0.169f, 0.294f, 0.524f, 1.67f, 0.64f, 1.2f},
    {"64x128_ring3", 64, 128, 0.171f, 0.295f, 0.533f, 1.72f, 0.64f, 1.2f},
    {"128x128_ring2", 128, 128, 0.543f, 0.639f, 0.918f, 1.62f, 1.0f, 1.5f},
    {"128x128_ring3", 128, 128, 0.267f, 0.45f, 0.0f, 3.0f, 0.60f, 1.5f},
    // Eight waves, for the large products that the persistent kernel does not take: a quarter of the barriers and half the
    // operand bytes of 128 x 128 tiles.  us, 128x128_ring2 / this: 16384 x 4096 x 11024 834 / 601, 16384 x 11008 x 4112 865 / 676,
    // 4096 x 4096 x 4112 84 / 63, 3000 x 3000 x 4112 in float32 76 / 57, 16384 x 11008 x 4096 in float32 734 / 671.
    {"256x256_ring2", 256, 256, 1.6f, 1.6f, 0.0f, 5.0f, 1.6f, 5.0f},
};
constexpr int kNumRing = sizeof(kRing) / sizeof(kRing[0]);
constexpr int kRing256 = kNumRing - 1;  // never cut along K
constexpr int kRingLastSliced = 2;      // (128 x 128 tiles have no registers left for a second set of sums)
constexpr float kLaunchUs = 2.6f;

// time of a problem of `slices` independent slices of `steps` K steps on tile shape r, launch included
float ring_cost(const RingShape& r, int64_t M, int64_t N, int64_t steps, int64_t slices)
{
    const int64_t tiles = ((M + r.bm - 1) / r.bm) * ((N + r.bn - 1) / r.bn) * slices;
    const int64_t per_cu = (tiles + 255) / 256;
    const float busy = (float)tiles / 256.0f;  // (the units share what the L2s deliver)
    const float tile = per_cu > 2 ? r.many_tile : r.tile;
    const float alone = per_cu > 2 ? r.many : r.step0 + (r.step1 - r.step0) * (busy < 1.0f ? busy : 1.0f);
    const float pair = per_cu > 2 ? r.many : r.step2;
    const float work = per_cu == 1 || r.step2 == 0.0f ? per_cu * (steps * alone + tile) : 0.5f * per_cu * (steps * pair + tile);
    // A short K leaves the stores: these kernels write 3.2 MB a us (27648 x 5120 x 256: 91-100 us, the persistent kernel 66-76).
    const float stores = (float)(M * N) * (slices > 1 ? 4.0f * slices : 2.0f) / 3.2e6f;
    return kLaunchUs + (work > stores ? work : stores);
}

// the fastest of the four-wave shapes (sliced: of those that are also built to add slices of K one after the other)
int best_ring(int64_t M, int64_t N, int64_t steps, int64_t slices, float* cost, bool sliced = false)
{
    int best = 0;
    float c = 0.0f;
    for (int i = 0; i < kRing256; ++i) {
        if (sliced && i > kRingLastSliced) break;
        const float t = ring_cost(kRing[i], M, N, steps, slices);
        if (i == 0 || t < c) {
            best = i;
            c = t;
        }
    }
    *cost = c;
    return best;
}

// A few rows (more than 16: up to there the few-rows kernel always) sum K in eighths on whichever kernel, so the choice is
// free: the few-rows kernel, whose workgroups take 32 rows of B and wait out a memory latency per step and wave; ring tiles
// that walk all of K; ring tiles for each eighth, whose planes a second launch adds.  Constants met within 15 % on 768 x 2048
// .. 5120 x 27648 and 17 .. 64 rows (us, in this order; 48 x 2816 x 1024: 6.4, 5.6, 6.9; 48 x 8192 x 2048: 9.2, 6.7, 9.6;
// 64 x 4096 x 4096: 13.0, 8.8, 12.5; 23 x 4096 x 11008: 28, 17.3, 14.0).
enum FewRowsKernel { kFewRows, kFewRing, kFewPlanes };

// slices that are not empty
int eighths(int64_t K) { return (int)(((K + BK - 1) / BK + eighth_steps(K) - 1) / eighth_steps(K)); }

FewRowsKernel choose_few_rows(int64_t M, int64_t N, int64_t K)
{
    if (M <= 16) return kFewRows;
    const float steps = (float)((K + BK - 1) / BK), bytes = (float)N * (float)K;
    const float rounds = (float)((N + 32 * 256 - 1) / (32 * 256));
    const float rows = 1.6f + rounds * (1.6f + eighth_steps(K) * (M <= 32 ? 1.75f : 2.6f));
    const float walk = 4.2f + 0.145f * steps, read = 2.0f + bytes / 5.3e6f;
    const float ring = walk > read ? walk : read;
    const float planes = steps < 2.0f ? 1e30f : 5.0f + bytes / 5.3e6f + (float)(M * N) * 1.5e-5f;
    if (rows <= ring && rows <= planes) return kFewRows;
    return ring <= planes ? kFewRing : kFewPlanes;
}

// Slices for a problem, 1 = do not split.  Slices are a summation order of their own, so they follow from the sizes alone
// and stay what they are when kernels get faster: few tiles and a K of at least eight steps, at least four of them a slice.
// Which kernel sums in that order is decided apart from it (splitk_entry).  The estimate behind the line: us per K step of a
// 64 x 64, 128 x 64 (64 x 128), 128 x 128 tile alone on a compute unit and of a pair sharing one, 0 where a pair does not fit.
float slices_estimate(int64_t M, int64_t N, int64_t steps, int64_t slices)
{
    struct Line {
        int bm, bn;
        float step1, step2, tile;
    };
    constexpr Line lines[] = {{64, 64, 0.28f, 0.39f, 1.2f}, {128, 64, 0.40f, 0.64f, 1.2f}, {64, 128, 0.40f, 0.64f, 1.2f},
                              {128, 128, 0.72f, 1.0f, 1.5f}, {128, 128, 0.60f, 0.0f, 1.5f}};
    float best = 1e30f;
    for (const Line& r : lines) {
        const int64_t per_cu = (ceil_div(M, r.bm) * ceil_div(N, r.bn) * slices + 255) / 256;
        const float work = per_cu == 1 || r.step2 == 0.0f ? per_cu * (steps * r.step1 + r.tile) : 0.5f * per_cu * (steps * r.step2 + r.tile);
        const float stores = (float)(M * N) * (slices > 1 ? 4.0f * slices : 2.0f) / 3.2e6f;
        const float t = 2.6f + (work > stores ? work : stores);
        best = t < best ? t : best;
    }
    return best;
}

int suggested_splits(int64_t M, int64_t N, int64_t K)
{
    const int64_t tiles256 = ((M + 255) / 256) * ((N + 255) / 256), tiles64 = ((M + 63) / 64) * ((N + 63) / 64);
    const int64_t steps = (K + BK - 1) / BK;
    if (M <= kSkinnyMaxM) return choose_few_rows(M, N, K) == kFewRows ? 1 : eighths(K);
    if (tiles256 > 96 || steps < 8) return 1;
    float best = slices_estimate(M, N, steps, 1);
    if (M >= 256 && N >= 256 && K % BK == 0 && N % 8 == 0) {
        const float t = m16_cost(M, N, K, false);
        best = t < best ? t : best;
    }
    if (tiles64 <= 192) best = 1e30f;
    int64_t splits = 1;
    for (int64_t s = 2; s <= 32 && s <= steps / 4; ++s) {
        const int64_t per = (steps + s - 1) / s;
        if ((s - 1) * per >= steps) continue;  // the last slice would be empty
        const float t = slices_estimate(M, N, per, s) + 2.2f + (float)(M * N) * (4.0f * s + 2.0f) / 4.0e6f;
        if (t < best) {
            best = t;
            splits = s;
        }
    }
    return (int)splits;
}

// ---- variants: the ring tile shapes, then the other two kernels ----------------------------------------------------

constexpr int kM16 = kNumRing, kSkinny = kNumRing + 1, kEighths = kNumRing + 2, kNumVariants = kNumRing + 3;

template <typename Args, typename Kernel>
int launch_ring_kernel(Kernel kern, std::atomic<uint64_t>& configured, int lds_bytes, const Args& a, int tiles, int slices,
                       int threads, hipStream_t st, const char* what)
{
    if (int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured, what)) return rc;
    hipLaunchKernelGGL(kern, dim3((tiles + 7) / 8 * 8, slices), dim3(threads), lds_bytes, st, a);
    return launch_status(what);
}

template <int BM, int BN, int ST, int OCC, int CBSZ, int BLGP, bool SLICED = false, int NW = kRingThreads / 64>
int launch_ring(GemmArgs& g, SplitArgs* split, hipStream_t st)
{
    GemmArgs& p = split ? split->g : g;
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    const int tiles = p.tiles_m * p.tiles_n;
    static std::atomic<uint64_t> configured[2];
    if constexpr (NW * 64 == kRingThreads)  // (slices are for problems of few tiles: none of the larger workgroups' business)
        if (split)
            return launch_ring_kernel(gemm_fp8_splitk_kernel<BM, BN, ST, OCC, CBSZ, BLGP>, configured[1], kRingLdsBytes<BM, BN, ST>,
                                      *split, tiles, split->splits, kRingThreads, st, "mi8_gemm_fp8_splitk");
    return launch_ring_kernel(gemm_fp8_ring_kernel<BM, BN, ST, OCC, CBSZ, BLGP, SLICED, NW>, configured[0], kRingLdsBytes<BM, BN, ST>,
                              g, tiles, 1, NW * 64, st, "mi8_gemm_fp8");
}

// K summed in slices of g.slice_steps steps by one workgroup a tile
template <int CBSZ, int BLGP>
int launch_sliced_shape(int shape, GemmArgs& g, hipStream_t st)
{
    switch (shape) {
        case 0: return launch_ring<64, 64, 4, 2, CBSZ, BLGP, true>(g, nullptr, st);
        case 1: return launch_ring<128, 64, 3, 2, CBSZ, BLGP, true>(g, nullptr, st);
        default: return launch_ring<64, 128, 3, 2, CBSZ, BLGP, true>(g, nullptr, st);
    }
}

template <int CBSZ, int BLGP>
int launch_ring_shape(int shape, GemmArgs& g, SplitArgs* split, hipStream_t st)
{
    if (g.slice_steps) return launch_sliced_shape<CBSZ, BLGP>(shape, g, st);
    switch (shape) {
        case 0: return launch_ring<64, 64, 4, 2, CBSZ, BLGP>(g, split, st);
        case 1: return launch_ring<128, 64, 3, 2, CBSZ, BLGP>(g, split, st);
        case 2: return launch_ring<64, 128, 3, 2, CBSZ, BLGP>(g, split, st);
        case 3: return launch_ring<128, 128, 2, 2, CBSZ, BLGP>(g, split, st);
        case 4: return launch_ring<128, 128, 3, 1, CBSZ, BLGP>(g, split, st);
        case kRing256: return launch_ring<256, 256, 2, 1, CBSZ, BLGP, false, 8>(g, nullptr, st);
    }
    set_error("mi8_gemm_fp8: unknown variant %d", shape);
    return MI8_ERR_ARG;
}

int launch_ring_typed(int shape, int a_dtype, int b_dtype, GemmArgs& g, SplitArgs* split, hipStream_t st)
{
    if (a_dtype == MI8_E4M3)
        return b_dtype == MI8_E4M3 ? launch_ring_shape<0, 0>(shape, g, split, st) : launch_ring_shape<0, 1>(shape, g, split, st);
    return b_dtype == MI8_E4M3 ? launch_ring_shape<1, 0>(shape, g, split, st) : launch_ring_shape<1, 1>(shape, g, split, st);
}

}  // namespace
int gemm::launch_dual_ring(GemmArgs& g, hipStream_t st)
{
    g.tiles_m = 1;
    g.tiles_n = dual_ring_slots(g.N);
    g.slice_steps = eighth_steps(g.K);
    static std::atomic<uint64_t> configured[2];
    const char* what = "mi8_few_rows_swiglu";
    if (g.M <= 32) return launch_ring_kernel(dual_ring_kernel<32>, configured[0], kRingLdsBytes<32, 64, 4>, g, g.tiles_n, 1, kRingThreads, st, what);
    return launch_ring_kernel(dual_ring_kernel<64>, configured[1], kRingLdsBytes<64, 64, 4>, g, g.tiles_n, 1, kRingThreads, st, what);
}
namespace {

// ---- several products in one launch: launch and cost ------------------------------------------------------------------

template <int BM, int BN, int ST, int OCC, int CBSZ, int BLGP, bool SLICED>
int launch_batch(BatchArgs& a, hipStream_t st)
{
    int slots = 0;
    for (int c = 0; c < a.chains; ++c) {
        a.first_slot[c] = slots;
        for (int i = a.head[c]; i >= 0; i = a.next[i]) {
            a.g[i].tiles_m = (a.g[i].M + BM - 1) / BM;
            a.g[i].tiles_n = (a.g[i].N + BN - 1) / BN;
        }
        slots += (a.g[a.head[c]].tiles_m * a.g[a.head[c]].tiles_n + 7) / 8;
    }
    for (int c = a.chains; c <= MI8_GEMM_BATCH; ++c) a.first_slot[c] = slots;
    static std::atomic<uint64_t> configured;
    const auto kern = gemm_fp8_batch_kernel<BM, BN, ST, OCC, CBSZ, BLGP, SLICED>;
    constexpr int lds_bytes = kRingLdsBytes<BM, BN, ST>;
    if (int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured, "mi8_gemm_fp8_batch")) return rc;
    hipLaunchKernelGGL(kern, dim3(8 * slots), dim3(kRingThreads), lds_bytes, st, a);
    return launch_status("mi8_gemm_fp8_batch");
}

template <int CBSZ, int BLGP>
int launch_batch_shape(int shape, bool sliced, BatchArgs& a, hipStream_t st)
{
    if (sliced) {
        if (shape == 0) return launch_batch<64, 64, 4, 2, CBSZ, BLGP, true>(a, st);
        if (shape == 1) return launch_batch<128, 64, 3, 2, CBSZ, BLGP, true>(a, st);
        return launch_batch<64, 128, 3, 2, CBSZ, BLGP, true>(a, st);
    }
    switch (shape) {
        case 0: return launch_batch<64, 64, 4, 2, CBSZ, BLGP, false>(a, st);
        case 1: return launch_batch<128, 64, 3, 2, CBSZ, BLGP, false>(a, st);
        case 2: return launch_batch<64, 128, 3, 2, CBSZ, BLGP, false>(a, st);
        case 3: return launch_batch<128, 128, 2, 2, CBSZ, BLGP, false>(a, st);
        default: return launch_batch<128, 128, 3, 1, CBSZ, BLGP, false>(a, st);
    }
}

// K steps that a product of these sizes sums from zero before they join the sum, 0: all of them (the order of its sums
// wherever it runs: see eighth_steps and suggested_splits)
int slice_steps_of(int64_t M, int64_t N, int64_t K)
{
    if (M <= kSkinnyMaxM) return eighth_steps(K);
    const int splits = suggested_splits(M, N, K);
    return splits > 1 ? (int)ceil_div(ceil_div(K, BK), splits) : 0;
}

// us of one launch over all tiles on shape r.  Chains are walked tile by tile; where units get more than one tile the load
// evens out but for half of the longest.  (128 x 128 pairs in a training step, model / measured: three products of
// 1537 x 2048 x 2048 36 / 42, grad_input and grad_weight of one of them 26 / 24, all six of three 78 / 70; in launches of their
// own 16 each.)
float batch_cost(const RingShape& r, const BatchArgs& a)
{
    int64_t tiles = 0;
    float longest = 0.0f, total = 0.0f, stores = 0.0f;
    for (int c = 0; c < a.chains; ++c) {
        const GemmArgs& h = a.g[a.head[c]];
        tiles += ceil_div(h.M, r.bm) * ceil_div(h.N, r.bn);
    }
    const bool one_round = tiles <= 256, many = tiles > 512;
    const float busy = tiles < 256 ? (float)tiles / 256.0f : 1.0f, tile = many ? r.many_tile : r.tile;
    const bool pairs = !one_round && r.step2 != 0.0f;
    const float step = pairs ? (many ? r.many : r.step2) : many && !pairs ? r.many : r.step0 + (r.step1 - r.step0) * busy;
    for (int c = 0; c < a.chains; ++c) {
        const GemmArgs& h = a.g[a.head[c]];
        float t = 0.0f;
        for (int i = a.head[c]; i >= 0; i = a.next[i]) {
            t += (float)ceil_div(a.g[i].K, BK) * step + tile;
            stores += (float)h.M * (float)h.N * (a.g[i].c_f32 ? 4.0f : 2.0f) * (a.g[i].accumulate ? 2.0f : 1.0f) / 3.2e6f;
        }
        longest = t > longest ? t : longest;
        total += t * (float)(ceil_div(h.M, r.bm) * ceil_div(h.N, r.bn)) / (pairs ? 512.0f : 256.0f);
    }
    const float work = one_round ? longest : 1.15f * total + 0.5f * longest;
    return kLaunchUs + (work > stores ? work : stores);
}

}  // namespace
}  // namespace mi8

using namespace mi8;

namespace {
// What the persistent kernel asks of a product's sizes.  (It shifts its last tile row / column back over the previous one when
// M or N is not a whole number of half tiles (128 x 256) and rewrites the overlap with identical values: not possible when
// accumulating.  Its output stores address a tile's 256 rows with 32-bit byte offsets: ldc < 2^22.)
bool m16_takes(int64_t M, int64_t N, int64_t K, int64_t ldc, int out_dtype, bool accumulate)
{
    return K % 128 == 0 && M >= 256 && N >= 256 && N % 8 == 0 && ldc % 8 == 0 && ldc < (out_dtype == MI8_BF16 ? 1 << 22 : 1 << 21) &&
           (out_dtype == MI8_BF16 || (out_dtype == MI8_F32_OF_BF16 && !accumulate)) &&
           (!accumulate || (M % 128 == 0 && N % 256 == 0));
}

// A few rows of A: see choose_few_rows; everything else goes to whichever of the ring tile shapes and the persistent
// kernel the measured costs above say is fastest for this number of tiles and K steps (all of them give the same bits).
int chosen_variant(int64_t M, int64_t N, int64_t K, bool m16_fits)
{
    if (M <= kSkinnyMaxM) {  // (a caller that wants the planes asks for split K)
        const FewRowsKernel few = choose_few_rows(M, N, K);
        return few == kFewRows || (few == kFewPlanes && M <= 32) ? kSkinny : kEighths;
    }
    float cost;
    const int64_t steps = ceil_div(K, BK);
    const int ring = best_ring(M, N, steps, 1, &cost);
    if (m16_fits) return m16_cost(M, N, K, true) < cost ? kM16 : ring;
    // (rows that do not start on a cache line cost the small tiles, which read them more often, a quarter more, the large
    // ones 5-7 %: 16384 x 4096 x 11008 and 11024, 616 and 834 us, 550 and 601)
    return ring_cost(kRing[kRing256], M, N, steps, 1) < (K % BK ? 1.25f : 1.0f) * cost ? kRing256 : ring;
}
}  // namespace

extern "C" int mi8_gemm_variant_for(int64_t M, int64_t N, int64_t K, int out_dtype, int accumulate)
{
    if (M <= 0 || N <= 0 || K <= 0 || (accumulate && out_dtype == MI8_F32_OF_BF16)) return -1;
    return chosen_variant(M, N, K, m16_takes(M, N, K, N, out_dtype, accumulate != 0));
}

extern "C" int mi8_gemm_num_variants(void) { return kNumVariants; }

extern "C" const char* mi8_gemm_variant_name(int variant)
{
    if (variant < 0 || variant >= kNumVariants) return nullptr;
    return variant == kM16 ? "256x256_dma_w4x128_m16x128" : variant == kSkinny ? "rows64x16_k8_m16x128"
           : variant == kEighths ? "64x64_ring4_eighths" : kRing[variant].name;
}

namespace {
int gemm_fp8_entry(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb, int64_t M, int64_t N,
                   int64_t K, const float* sa, int sa_is_vector, const float* sb, int sb_is_vector, void* out,
                   int out_dtype, int64_t ldc, int variant, bool accumulate, void* stream)
{
    MI8_REQUIRE(a && b && sa && sb && out, MI8_ERR_ARG, "mi8_gemm_fp8: null pointer");
    MI8_REQUIRE((a_dtype == MI8_E4M3 || a_dtype == MI8_E5M2) && (b_dtype == MI8_E4M3 || b_dtype == MI8_E5M2),
                MI8_ERR_ARG, "mi8_gemm_fp8: unknown fp8 dtype");
    MI8_REQUIRE(M > 0 && N > 0 && K > 0, MI8_ERR_ARG, "mi8_gemm_fp8: empty problem %lld x %lld x %lld",
                (long long)M, (long long)N, (long long)K);
    MI8_REQUIRE(variant >= -1 && variant < kNumVariants, MI8_ERR_ARG, "mi8_gemm_fp8: unknown variant %d", variant);
    MI8_REQUIRE(K % 16 == 0 && lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8: K (%lld), lda (%lld), ldb (%lld) must be multiples of 16 with lda, ldb >= K",
                (long long)K, (long long)lda, (long long)ldb);
    MI8_REQUIRE(ldc >= N, MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8: ldc (%lld) < N (%lld)", (long long)ldc, (long long)N);
    MI8_REQUIRE(aligned16(a) && aligned16(b), MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8: operands must be 16-byte aligned");
    MI8_REQUIRE(M * lda < (int64_t)1 << 32 && N * ldb < (int64_t)1 << 32 && M < (1 << 30) && N < (1 << 30) &&
                    K < (1 << 30),
                MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8: operand larger than 4 GiB");
    MI8_REQUIRE(gemm_out_dtype(out_dtype), MI8_ERR_ARG, "mi8_gemm_fp8: unknown output dtype %d",
                out_dtype);
    MI8_REQUIRE(!accumulate || out_dtype != MI8_F32_OF_BF16, MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8_accumulate: a sum is not rounded to bf16 values");
    GemmArgs g{(const uint8_t*)a, (const uint8_t*)b, out, c_f32_of(out_dtype), lda, ldb, ldc, (int)M, (int)N, (int)K,
               sa, sb, sa_is_vector ? 1 : 0, sb_is_vector ? 1 : 0, 0, 0, accumulate ? 1 : 0};
    hipStream_t st = (hipStream_t)stream;
    const bool dma_ok = m16_takes(M, N, K, ldc, out_dtype, accumulate) && aligned16(out) && (!sb_is_vector || aligned16(sb)) &&
                        (sa_is_vector != 0) == (sb_is_vector != 0);
    if (variant < 0) variant = chosen_variant(M, N, K, dma_ok);
    if (variant == kSkinny) return launch_skinny(g, a_dtype, b_dtype, st);
    if (variant == kM16) {
        MI8_REQUIRE(dma_ok, MI8_ERR_UNSUPPORTED,
                    "mi8_gemm_fp8: the direct-to-LDS variant needs M, N >= 256, K %% 128 == 0, N %% 8 == 0, ldc %% 8 == 0, "
                    "scales that are both single values or both vectors, and a 16-byte aligned output of bf16 values (M=%lld N=%lld K=%lld ldc=%lld)",
                    (long long)M, (long long)N, (long long)K, (long long)ldc);
        return launch_m16(g, a_dtype, b_dtype, st);
    }
    if (variant == kEighths) {
        g.slice_steps = eighth_steps(K);
        variant = 0;
    }
    return launch_ring_typed(variant, a_dtype, b_dtype, g, nullptr, st);
}
}  // namespace

extern "C" int mi8_gemm_fp8(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                            int64_t M, int64_t N, int64_t K, const float* sa, int sa_is_vector, const float* sb,
                            int sb_is_vector, void* out, int out_dtype, int64_t ldc, int variant, void* stream)
{
    return gemm_fp8_entry(a, a_dtype, lda, b, b_dtype, ldb, M, N, K, sa, sa_is_vector, sb, sb_is_vector, out, out_dtype,
                          ldc, variant, false, stream);
}

extern "C" int mi8_gemm_fp8_accumulate(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                                       int64_t M, int64_t N, int64_t K, const float* sa, int sa_is_vector,
                                       const float* sb, int sb_is_vector, void* out, int out_dtype, int64_t ldc,
                                       void* stream)
{
    return gemm_fp8_entry(a, a_dtype, lda, b, b_dtype, ldb, M, N, K, sa, sa_is_vector, sb, sb_is_vector, out, out_dtype,
                          ldc, -1, true, stream);
}

// 1 if mi8_gemm_fp8_swiglu takes the shape AND the library would not cut either projection along K (then the fused
// launch reproduces the three-call route bit for bit: all kernels that do not split sum in one order), for products of many tiles,
// which are never cut
extern "C" int mi8_gemm_fp8_swiglu_matches_separate(int64_t M, int64_t H, int64_t K)
{
    if (M < 256 || H < 256 || K <= 0 || K % 128 || H % 8) return 0;
    const int64_t tiles256 = ((M + 255) / 256) * ((H + 255) / 256);
    return tiles256 > 96 ? 1 : 0;
}

// The same for any number of tiles: with few the fused launch, in whole, half and quarter tiles, is the faster one too.  us fused /
// two products in one launch and the activation: 256 x 11008 x 4096 29.2 / 43.8, 300 44.5 / 56.9; 640 x 8192 x 2048 28.3 / 37.8;
// 1999 x 2816 x 1024 20.8 / 28.3; 777 x 2048 x 768 9.4 / 14.8, 256 8.6 / 9.3; 256 x 512 x 512 7.5 / 8.0.  A block without gradients: 400 x 512 x
// 512 39.9 / 43.0, 512 x 8192 x 512 41.7 / 47.9; of 230 sizes with K of 512 to 2048 none was slower.  The line at K = 512 is not one of speed (3000 x 2048 x
// 384 40.8 / 46.0, 777 x 2048 x 256 39.4 / 42.3, none of 219 sizes slower): the tests of calls that are recorded and replaced pin the
// separate launches with blocks 256 wide, and the feed-forward blocks of perf/cases.py are 768 wide or more.
extern "C" int mi8_gemm_fp8_swiglu_pays(int64_t M, int64_t H, int64_t K)
{
    if (mi8_gemm_fp8_swiglu_matches_separate(M, H, K)) return 1;
    if (M < 256 || H < 256 || K < 512 || K % 128 || H % 8) return 0;
    return suggested_splits(M, H, K) == 1 ? 1 : 0;
}

extern "C" int mi8_gemm_fp8_swiglu(const void* a, int a_dtype, int64_t lda, const void* b1, const void* b3, int b_dtype,
                                   int64_t ldb, int64_t M, int64_t H, int64_t K, const float* sa, const float* sb1,
                                   const float* sb3, void* x1, void* x3, void* h, int64_t ldc, uint32_t* slots_h,
                                   int32_t* n_slots_used, uint16_t* x_codes, void* stream)
{
    MI8_REQUIRE(a && b1 && b3 && sa && sb1 && sb3 && x1 && x3 && h && slots_h && n_slots_used, MI8_ERR_ARG,
                "mi8_gemm_fp8_swiglu: null pointer");
    MI8_REQUIRE((a_dtype == MI8_E4M3 || a_dtype == MI8_E5M2) && (b_dtype == MI8_E4M3 || b_dtype == MI8_E5M2),
                MI8_ERR_ARG, "mi8_gemm_fp8_swiglu: unknown fp8 dtype");
    MI8_REQUIRE(M >= 256 && H >= 128 && K > 0 && K % 128 == 0 && H % 8 == 0, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_swiglu: needs M >= 256, H >= 128, H %% 8 == 0, K %% 128 == 0 (got %lld x %lld x %lld); use "
                "mi8_gemm_fp8 twice and mi8_swiglu_fwd",
                (long long)M, (long long)H, (long long)K);
    MI8_REQUIRE(lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K && ldc >= H && ldc % 8 == 0, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_swiglu: lda, ldb must be multiples of 16 and >= K, ldc a multiple of 8 and >= H");
    MI8_REQUIRE(aligned16(a) && aligned16(b1) && aligned16(b3) && aligned16(x1) && aligned16(x3) && aligned16(h),
                MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8_swiglu: operands and outputs must be 16-byte aligned");
    MI8_REQUIRE(M * lda < (int64_t)1 << 32 && H * ldb < (int64_t)1 << 32 && M < (1 << 30) && H < (1 << 30) &&
                    K < (1 << 30),
                MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8_swiglu: operand larger than 4 GiB");
    MI8_REQUIRE(!x_codes || H % 64 == 0, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_swiglu: row-segment codes need H (%lld) to be a multiple of 64", (long long)H);
    GemmArgs g{(const uint8_t*)a, (const uint8_t*)b1, x1, 0, lda, ldb, ldc, (int)M, (int)H, (int)K, sa, sb1, 0, 0, 0, 0, 0};
    int used = 0;
    const int rc = launch_m16_swiglu(g, (const uint8_t*)b3, sb3, (uint16_t*)x3, (uint16_t*)h, slots_h, &used, x_codes,
                                     a_dtype, b_dtype, (hipStream_t)stream);
    *n_slots_used = used;
    return rc;
}

extern "C" int32_t mi8_gemm_fp8_swiglu_slots(int64_t M, int64_t H, int64_t K)
{
    if (M < 256 || H < 128 || K <= 0 || M >= (1 << 30) || H >= (1 << 30) || K >= (1 << 30)) return 0;
    return m16_swiglu_slots(M, H, K);
}

// 1 if mi8_gemm_fp8_codes takes the shape: shapes that the library never cuts along K (so that the output has the bits
// of the plain call) whose row segments line up with the output tiles
extern "C" int mi8_gemm_fp8_codes_supported(int64_t M, int64_t N, int64_t K)
{
    if (M < 256 || N < 256 || K <= 0 || K % 128 || N % 64) return 0;
    const int64_t tiles256 = ((M + 255) / 256) * ((N + 255) / 256);
    return tiles256 > 96 ? 1 : 0;
}

extern "C" int mi8_gemm_fp8_codes(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb, int64_t M,
                                  int64_t N, int64_t K, const float* sa, const float* sb, void* out, int64_t ldc,
                                  uint16_t* codes, void* stream)
{
    MI8_REQUIRE(a && b && sa && sb && out && codes, MI8_ERR_ARG, "mi8_gemm_fp8_codes: null pointer");
    MI8_REQUIRE((a_dtype == MI8_E4M3 || a_dtype == MI8_E5M2) && (b_dtype == MI8_E4M3 || b_dtype == MI8_E5M2),
                MI8_ERR_ARG, "mi8_gemm_fp8_codes: unknown fp8 dtype");
    MI8_REQUIRE(mi8_gemm_fp8_codes_supported(M, N, K), MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_codes: needs N %% 64 == 0, K %% 128 == 0 and more than 96 tiles of 256 x 256 (got %lld x %lld x "
                "%lld); use mi8_gemm_fp8 and mi8_rowseg_max_codes",
                (long long)M, (long long)N, (long long)K);
    MI8_REQUIRE(lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K && ldc >= N && ldc % 8 == 0, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_codes: lda, ldb must be multiples of 16 and >= K, ldc a multiple of 8 and >= N");
    MI8_REQUIRE(aligned16(a) && aligned16(b) && aligned16(out), MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_codes: operands and output must be 16-byte aligned");
    MI8_REQUIRE(M * lda < (int64_t)1 << 32 && N * ldb < (int64_t)1 << 32 && M < (1 << 30) && N < (1 << 30) && K < (1 << 30),
                MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8_codes: operand larger than 4 GiB");
    GemmArgs g{(const uint8_t*)a, (const uint8_t*)b, out, 0, lda, ldb, ldc, (int)M, (int)N, (int)K, sa, sb, 0, 0, 0, 0, 0};
    return launch_m16_codes(g, codes, a_dtype, b_dtype, (hipStream_t)stream);
}

extern "C" int mi8_gemm_splitk_suggest(int64_t M, int64_t N, int64_t K)
{
    if (M <= 0 || N <= 0 || K <= 0) return 1;
    return suggested_splits(M, N, K);
}

extern "C" int64_t mi8_gemm_splitk_workspace_bytes(int64_t M, int64_t N, int splits)
{
    if (M <= 0 || N <= 0 || splits <= 0) return 0;
    return (int64_t)splits * M * ((N + 3) / 4 * 4) * (int64_t)sizeof(float);
}

namespace {
int splitk_entry(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                                   int64_t M, int64_t N, int64_t K, const float* sa, int sa_is_vector,
                                   const float* sb, int sb_is_vector, void* out, int out_dtype, int64_t ldc,
                                   int splits, void* workspace, int64_t workspace_bytes, bool accumulate, void* stream)
{
    MI8_REQUIRE(a && b && sa && sb && out && workspace, MI8_ERR_ARG, "mi8_gemm_fp8_splitk: null pointer");
    MI8_REQUIRE((a_dtype == MI8_E4M3 || a_dtype == MI8_E5M2) && (b_dtype == MI8_E4M3 || b_dtype == MI8_E5M2),
                MI8_ERR_ARG, "mi8_gemm_fp8_splitk: unknown fp8 dtype");
    MI8_REQUIRE(M > 0 && N > 0 && K > 0, MI8_ERR_ARG, "mi8_gemm_fp8_splitk: empty problem %lld x %lld x %lld",
                (long long)M, (long long)N, (long long)K);
    MI8_REQUIRE(K % 16 == 0 && lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_splitk: K (%lld), lda (%lld), ldb (%lld) must be multiples of 16 with lda, ldb >= K",
                (long long)K, (long long)lda, (long long)ldb);
    MI8_REQUIRE(ldc >= N, MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8_splitk: ldc (%lld) < N (%lld)", (long long)ldc,
                (long long)N);
    MI8_REQUIRE(aligned16(a) && aligned16(b) && aligned16(workspace), MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_splitk: operands and workspace must be 16-byte aligned");
    MI8_REQUIRE(M * lda < (int64_t)1 << 32 && N * ldb < (int64_t)1 << 32 && M < (1 << 30) && N < (1 << 30) &&
                    K < (1 << 30),
                MI8_ERR_UNSUPPORTED, "mi8_gemm_fp8_splitk: operand larger than 4 GiB");
    MI8_REQUIRE(gemm_out_dtype(out_dtype), MI8_ERR_ARG,
                "mi8_gemm_fp8_splitk: unknown output dtype %d", out_dtype);
    MI8_REQUIRE(!accumulate || out_dtype != MI8_F32_OF_BF16, MI8_ERR_UNSUPPORTED,
                "mi8_gemm_fp8_splitk_accumulate: a sum is not rounded to bf16 values");
    const int64_t steps = (K + BK - 1) / BK;
    MI8_REQUIRE(splits >= 1 && splits <= 64 && splits <= steps, MI8_ERR_ARG,
                "mi8_gemm_fp8_splitk: splits (%d) must be in 1..min(64, K steps = %lld)", splits, (long long)steps);
    const int64_t per = (steps + splits - 1) / splits;
    const int used = (int)((steps + per - 1) / per);  // slices that are not empty
    MI8_REQUIRE(workspace_bytes >= mi8_gemm_splitk_workspace_bytes(M, N, used), MI8_ERR_ARG,
                "mi8_gemm_fp8_splitk: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
                (long long)mi8_gemm_splitk_workspace_bytes(M, N, used));
    SplitArgs s{};
    s.g = GemmArgs{(const uint8_t*)a, (const uint8_t*)b, out, c_f32_of(out_dtype), lda, ldb, ldc, (int)M,
                   (int)N, (int)K, sa, sb, sa_is_vector ? 1 : 0, sb_is_vector ? 1 : 0, 0, 0, accumulate ? 1 : 0};
    s.planes = (float*)workspace;
    s.ld_plane = (N + 3) / 4 * 4;
    s.steps_per_split = (int)per;
    s.splits = used;
    hipStream_t st = (hipStream_t)stream;
    // The planes are left out where one workgroup a tile adds the slices sooner (the eighths of a few rows: choose_few_rows).
    // Both fitted to 550 products of 65 to 700 rows and 2 to 8 slices; us in planes / whole: 128 x 4096 x 4096 in four 13.5 / 8.6,
    // 300 x 2048 x 2048 in three 11.7 / 6.7, 128 x 2048 x 8192 in three 10.6 / 11.6, 200 x 5120 x 27648 in six 43.8 / 61.2.
    float planes, whole;
    const int shape = best_ring(M, N, per, used, &planes);
    int sliced = best_ring(M, N, steps, 1, &whole, true);
    planes += 2.9f + (float)(M * N) * (0.89e-6f * used + 0.66e-6f);
    bool leave_out = whole < planes;
    if (M <= kSkinnyMaxM && used == eighths(K)) {
        leave_out = choose_few_rows(M, N, K) == kFewRing;
        sliced = 0;
    }
    if (leave_out) {
        s.g.slice_steps = (int)per;
        return launch_ring_typed(sliced, a_dtype, b_dtype, s.g, nullptr, st);
    }
    if (int rc = launch_ring_typed(shape, a_dtype, b_dtype, s.g, &s, st)) return rc;
    const int64_t quads = M * (s.ld_plane / 4);
    const auto reduce = used > 4 ? splitk_reduce_kernel<7> : used > 2 ? splitk_reduce_kernel<3> : splitk_reduce_kernel<1>;
    hipLaunchKernelGGL(reduce, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, s);
    return launch_status("mi8_gemm_fp8_splitk");
}
}  // namespace

extern "C" int mi8_gemm_fp8_splitk(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                                   int64_t M, int64_t N, int64_t K, const float* sa, int sa_is_vector,
                                   const float* sb, int sb_is_vector, void* out, int out_dtype, int64_t ldc,
                                   int splits, void* workspace, int64_t workspace_bytes, void* stream)
{
    return splitk_entry(a, a_dtype, lda, b, b_dtype, ldb, M, N, K, sa, sa_is_vector, sb, sb_is_vector, out, out_dtype, ldc,
                        splits, workspace, workspace_bytes, false, stream);
}

extern "C" int mi8_gemm_fp8_splitk_accumulate(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                                              int64_t M, int64_t N, int64_t K, const float* sa, int sa_is_vector,
                                              const float* sb, int sb_is_vector, void* out, int out_dtype, int64_t ldc,
                                              int splits, void* workspace, int64_t workspace_bytes, void* stream)
{
    return splitk_entry(a, a_dtype, lda, b, b_dtype, ldb, M, N, K, sa, sa_is_vector, sb, sb_is_vector, out, out_dtype, ldc,
                        splits, workspace, workspace_bytes, true, stream);
}

namespace {
int batch_args(const mi8_gemm_product* p, int32_t count, BatchArgs& a, bool& sliced)
{
    const char* what = "mi8_gemm_fp8_batch";
    MI8_REQUIRE(p, MI8_ERR_ARG, "%s: null pointer", what);
    MI8_REQUIRE(count > 0 && count <= MI8_GEMM_BATCH, MI8_ERR_ARG, "%s: %d products (1..%d)", what, count, MI8_GEMM_BATCH);
    a.chains = 0;
    sliced = false;
    for (int i = 0; i < count; ++i) {
        const mi8_gemm_product& q = p[i];
        MI8_REQUIRE(q.a && q.b && q.sa && q.sb && q.out, MI8_ERR_ARG, "%s: product %d: null pointer", what, i);
        MI8_REQUIRE(q.M > 0 && q.N > 0 && q.K > 0, MI8_ERR_ARG, "%s: product %d: empty problem %lld x %lld x %lld", what, i,
                    (long long)q.M, (long long)q.N, (long long)q.K);
        MI8_REQUIRE(q.K % 16 == 0 && q.lda % 16 == 0 && q.ldb % 16 == 0 && q.lda >= q.K && q.ldb >= q.K && q.ldc >= q.N,
                    MI8_ERR_UNSUPPORTED, "%s: product %d: K (%lld), lda (%lld), ldb (%lld) must be multiples of 16 with lda, ldb >= K, ldc (%lld) >= N",
                    what, i, (long long)q.K, (long long)q.lda, (long long)q.ldb, (long long)q.ldc);
        MI8_REQUIRE(aligned16(q.a) && aligned16(q.b), MI8_ERR_UNSUPPORTED, "%s: product %d: operands must be 16-byte aligned", what, i);
        MI8_REQUIRE(q.M < (1 << 30) && q.N < (1 << 30) && q.K < (1 << 30) && q.M * q.lda < (int64_t)1 << 32 && q.N * q.ldb < (int64_t)1 << 32,
                    MI8_ERR_UNSUPPORTED, "%s: product %d: operand larger than 4 GiB", what, i);
        MI8_REQUIRE(gemm_out_dtype(q.out_dtype), MI8_ERR_ARG, "%s: product %d: unknown output dtype %d", what, i, q.out_dtype);
        MI8_REQUIRE(!q.add_to_previous || (i > 0 && q.M == p[i - 1].M && q.N == p[i - 1].N && q.out == p[i - 1].out && q.ldc == p[i - 1].ldc &&
                                           q.out_dtype == p[i - 1].out_dtype),
                    MI8_ERR_ARG, "%s: product %d adds to the one before it: one output and sizes are wanted", what, i);
        MI8_REQUIRE(!q.add_to_previous || q.out_dtype != MI8_F32_OF_BF16, MI8_ERR_UNSUPPORTED, "%s: product %d: a sum is not rounded to bf16 values",
                    what, i);
        a.g[i] = GemmArgs{(const uint8_t*)q.a, (const uint8_t*)q.b, q.out, c_f32_of(q.out_dtype), q.lda, q.ldb, q.ldc, (int)q.M,
                          (int)q.N, (int)q.K, q.sa, q.sb, q.sa_is_vector ? 1 : 0, q.sb_is_vector ? 1 : 0, 0, 0, q.add_to_previous ? 1 : 0,
                          slice_steps_of(q.M, q.N, q.K)};
        sliced = sliced || a.g[i].slice_steps;
        a.next[i] = -1;
        if (q.add_to_previous)
            a.next[i - 1] = i;
        else
            a.head[a.chains++] = i;
    }
    return MI8_OK;
}

int best_batch_shape(const BatchArgs& a, bool sliced, float* cost)
{
    int best = 0;
    for (int i = 0; i <= (sliced ? kRingLastSliced : kRing256 - 1); ++i) {
        const float t = batch_cost(kRing[i], a);
        if (i == 0 || t < *cost) {
            best = i;
            *cost = t;
        }
    }
    return best;
}
}  // namespace

// One launch against a launch each: us, estimates as above; in a step operands come from memory rather than from the last
// repetition's L2, so a product on its own takes 1.2 times its estimate, and every launch that follows another 2 us.  Fitted to 66 sets
// of two to six products, 400-4000 rows of 1024 and 2048 (replayed graphs, operands of four sets in turn): 0.3 % over the better of the two
// on average, 5 % before the two constants; the largest misses 5 %.  us together / apart: the six products of three projections'
// backward, 1537 x 2048 61 / 84, 4000 x 2048 146 / 153; grad_input and grad_weight of one 21 / 27, 4000 rows 47 / 41; of two
// projections 1024 -> 2816, 3000 rows 46 / 61.
extern "C" int mi8_gemm_fp8_batch_pays(const mi8_gemm_product* products, int32_t count)
{
    BatchArgs a;
    bool sliced;
    if (batch_args(products, count, a, sliced) != MI8_OK) return 0;
    float together = 0.0f, apart = 2.0f * (float)(count - 1);
    best_batch_shape(a, sliced, &together);
    for (int i = 0; i < count; ++i) {
        const GemmArgs& g = a.g[i];
        const bool acc = g.accumulate != 0;
        float t;
        best_ring(g.M, g.N, ceil_div(g.K, BK), 1, &t, g.slice_steps != 0);
        if (m16_takes(g.M, g.N, g.K, g.ldc, g.c_f32 == 0 ? MI8_BF16 : g.c_f32 == 1 ? MI8_F32 : MI8_F32_OF_BF16, acc) && aligned16(g.C) && !g.slice_steps) {
            const float p = m16_cost(g.M, g.N, g.K, true);
            t = p < t ? p : t;
        }
        apart += 1.2f * t;
    }
    return together < apart ? 1 : 0;
}

extern "C" int mi8_gemm_fp8_batch(const mi8_gemm_product* products, int32_t count, int a_dtype, int b_dtype, void* stream)
{
    MI8_REQUIRE((a_dtype == MI8_E4M3 || a_dtype == MI8_E5M2) && (b_dtype == MI8_E4M3 || b_dtype == MI8_E5M2), MI8_ERR_ARG,
                "mi8_gemm_fp8_batch: unknown fp8 dtype");
    BatchArgs a;
    bool sliced;
    if (int rc = batch_args(products, count, a, sliced)) return rc;
    float cost = 0.0f;
    const int shape = best_batch_shape(a, sliced, &cost);
    if (sliced)  // (whole products among sliced ones: one slice)
        for (int i = 0; i < count; ++i)
            if (!a.g[i].slice_steps) a.g[i].slice_steps = 1 << 30;
    hipStream_t st = (hipStream_t)stream;
    if (a_dtype == MI8_E4M3)
        return b_dtype == MI8_E4M3 ? launch_batch_shape<0, 0>(shape, sliced, a, st) : launch_batch_shape<0, 1>(shape, sliced, a, st);
    return b_dtype == MI8_E4M3 ? launch_batch_shape<1, 0>(shape, sliced, a, st) : launch_batch_shape<1, 1>(shape, sliced, a, st);
}
