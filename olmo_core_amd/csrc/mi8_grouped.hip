// Ragged grouped fp8 GEMMs for the dropless-MoE expert layer: rows of the activation matrix are split into
// consecutive groups (one per expert, sizes known only on the device), every group multiplies its own weight.
//
//   grouped_gemm  : out[rows_e, :] = A[rows_e, :K] . B_e[:N, :K]^T      (forward and grad_input; ragged M)
//   grouped_wgrad : out[e]         = A_t[:, seg_e] . B_t[:, seg_e]^T     (grad_weight; ragged K, segments padded
//                                                                          to multiples of 128 with zero bytes)
//
// Each workgroup finds its group in the device-resident sizes, builds a per-group view of the operands and runs the
// general tile routine on it; workgroups beyond the real number of tiles exit.
#include "mi8_gemm_ring.h"
#include "mi8_groups.h"

namespace mi8 {
using namespace gemm;
namespace {

struct GroupedArgs {
    const uint8_t* A;  // [T, lda]
    const uint8_t* B;  // group e starts at B + e * b_group_stride, rows N, pitch ldb
    void* C;           // [T, ldc]
    int c_f32;
    int64_t lda, ldb, ldc, b_group_stride, sb_group_stride;
    const int64_t* sizes;
    int E;
    int64_t T;
    int N, K;
    const float* sa;  // [T]
    const float* sb;  // group e: sb + e * sb_group_stride, N values
    int tiles_n;
    int accumulate;   // C += the rounded product
};

template <int BM, int BN, int ST, int CBSZ, int BLGP>
__global__ __launch_bounds__(kRingThreads, 2) void grouped_gemm_kernel(GroupedArgs a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int mt = (int)blockIdx.x / a.tiles_n, nt = (int)blockIdx.x % a.tiles_n;
    const GroupSpan s = locate_group<BM, true>(a.sizes, a.E, a.T, mt);
    if (s.e >= a.E) return;
    GemmArgs g;
    g.A = a.A + s.rows_before * a.lda;
    g.B = a.B + (int64_t)s.e * a.b_group_stride;
    g.C = reinterpret_cast<uint8_t*>(a.C) + s.rows_before * a.ldc * (a.c_f32 ? 4 : 2);
    g.c_f32 = a.c_f32;
    g.lda = a.lda;
    g.ldb = a.ldb;
    g.ldc = a.ldc;
    g.M = (int)s.m;
    g.N = a.N;
    g.K = a.K;
    g.sa = a.sa + s.rows_before;
    g.sb = a.sb + (int64_t)s.e * a.sb_group_stride;
    g.sa_vec = 1;
    g.sb_vec = 1;
    g.accumulate = a.accumulate;
    ring_tile<BM, BN, ST, CBSZ, BLGP>(g, (int)(mt - s.units_before) * BM, nt * BN, lds);
}

struct GroupedWgradArgs {
    const uint8_t* At;  // [N, ld_t]
    const uint8_t* Bt;  // [Kl, ld_t]
    int64_t ld_t;
    const int64_t* sizes;
    int E;
    int64_t T;
    int N, Kl;
    const float* sa;  // [E, N]
    const float* sb;  // [E, Kl]
    void* C;          // [E, N, Kl]
    int c_f32;
    int tiles_n, tiles_k;
};

template <int BM, int BN, int ST, int CBSZ, int BLGP, int NW>
__global__ __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) void grouped_wgrad_kernel(GroupedWgradArgs a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int per_group = a.tiles_n * a.tiles_k;
    const int e = (int)blockIdx.x / per_group;
    const int rem = (int)blockIdx.x % per_group;
    const int tn = rem / a.tiles_k, tk = rem % a.tiles_k;
    // segment of group e in the padded token axis: starts at 128 * (tiles of the groups before it)
    const GroupSpan s = locate_group<128, false>(a.sizes, a.E, a.T, e);
    const int64_t seg0 = 128 * s.units_before;
    int64_t seg = 128 * ((s.m + 127) / 128);
    if (seg0 + seg > a.ld_t) seg = 0;
    GemmArgs g;
    g.A = a.At + seg0;
    g.B = a.Bt + seg0;
    g.C = reinterpret_cast<uint8_t*>(a.C) + (int64_t)e * a.N * a.Kl * (a.c_f32 ? 4 : 2);
    g.c_f32 = a.c_f32;
    g.lda = a.ld_t;
    g.ldb = a.ld_t;
    g.ldc = a.Kl;
    g.M = a.N;
    g.N = a.Kl;
    g.K = (int)seg;  // 0 for an empty group: the tile routine then writes zeros
    // an empty group has no scales (nothing was quantised): the raw sums, zeros, are what is wanted
    g.sa = seg ? a.sa + (int64_t)e * a.N : nullptr;
    g.sb = seg ? a.sb + (int64_t)e * a.Kl : nullptr;
    g.sa_vec = seg ? 1 : 0;
    g.sb_vec = seg ? 1 : 0;
    g.accumulate = 0;
    ring_tile<BM, BN, ST, CBSZ, BLGP, false, NW>(g, tn * BM, tk * BN, lds);
}

template <int BM, int BN, int ST, int CBSZ, int BLGP>
int launch_grouped(GroupedArgs& a, hipStream_t st)
{
    auto kern = grouped_gemm_kernel<BM, BN, ST, CBSZ, BLGP>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), kRingLdsBytes<BM, BN, ST>, configured, "mi8_grouped_gemm_fp8"))
        return rc;
    a.tiles_n = (a.N + BN - 1) / BN;
    const int64_t blocks = (ceil_div(a.T, BM) + a.E) * a.tiles_n;  // every group adds at most one partial tile
    MI8_REQUIRE(blocks < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kRingThreads), (kRingLdsBytes<BM, BN, ST>), st, a);
    return launch_status("mi8_grouped_gemm_fp8");
}

// Which kernel a grouped product runs on, by estimated microseconds.  The sizes of the groups are on the device; with
// popularity as skewed as routers make it, T rows in E groups fill about T / BM + E / 2 tiles of BM rows.  Measured, with
// s = K / 128 steps: the persistent kernel has 256 workgroups and takes 3.3 + 1.1 s a round, a ring tile 32, 64 or 128 rows
// high 3.4 + 0.53 s, 2 + s or 3 + 1.38 s for 512 of them, half of that where each has a compute unit to itself; any launch
// 5 more.  64 groups, N 1024, K 2048 (us: persistent, rings of 32, 64 and 128 rows), T = 384: 26, 13.5, 13.5, 17.5;
// 2048: 27, 29, 22, 23; 4096: 29, 46, 38, 30; 8 groups, N 1024, K 1792, T = 1024: 22, 12, 11.5, 15; 4096: 23, 30, 25, 20;
// 8192: 24, 50, 39, 37.  The lines lie where the estimates cross.  All four give the same bits.
enum GroupedKernel { kRing32, kRing64, kRing128, kPersistent };

GroupedKernel choose_grouped(int64_t T, int64_t E, int64_t N, int64_t K, bool persistent_fits)
{
    const double steps = (double)ceil_div(K, 128), columns = (double)ceil_div(N, 128);
    const double rows = (double)T, partial = 0.5 * (double)(E < T ? E : T);
    const auto ring = [&](double round, int bm) {
        const double blocks = (rows / bm + partial) * columns / 512;
        return round * (blocks > 0.5 ? blocks : 0.5);
    };
    const double cost[4] = {ring(3.4 + 0.53 * steps, 32), ring(2.0 + steps, 64), ring(3.0 + 1.38 * steps, 128), [&] {
                                const double tiles = (rows / 256 + partial) * (double)ceil_div(N, 256) / 256;
                                return (3.3 + 1.1 * steps) * (tiles > 1 ? tiles : 1);
                            }()};
    int best = kRing32;
    for (int k = kRing64; k <= (persistent_fits ? kPersistent : kRing128); ++k)
        if (cost[k] < cost[best]) best = k;
    return (GroupedKernel)best;
}

template <int CBSZ, int BLGP>
int launch_grouped_shape(GroupedArgs& a, GroupedKernel k, hipStream_t st)
{
    if (k == kRing32) return launch_grouped<32, 128, 4, CBSZ, BLGP>(a, st);
    if (k == kRing64) return launch_grouped<64, 128, 3, CBSZ, BLGP>(a, st);
    return launch_grouped<128, 128, 2, CBSZ, BLGP>(a, st);
}

template <int BM, int BN, int ST, int CBSZ, int BLGP, int NW = kRingThreads / 64>
int launch_wgrad(GroupedWgradArgs& a, hipStream_t st)
{
    auto kern = grouped_wgrad_kernel<BM, BN, ST, CBSZ, BLGP, NW>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), kRingLdsBytes<BM, BN, ST>, configured, "mi8_grouped_wgrad_fp8"))
        return rc;
    a.tiles_n = (a.N + BM - 1) / BM;
    a.tiles_k = (a.Kl + BN - 1) / BN;
    const int64_t blocks = (int64_t)a.E * a.tiles_n * a.tiles_k;
    MI8_REQUIRE(blocks < ((int64_t)1 << 31), MI8_ERR_UNSUPPORTED, "mi8_grouped_wgrad_fp8: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), (kRingLdsBytes<BM, BN, ST>), st, a);
    return launch_status("mi8_grouped_wgrad_fp8");
}

// Small tiles until the middle ones would put two workgroups on every compute unit; the large ones, eight waves each, where
// they fill the chip four times (groups differ in length, and fewer rounds do not even that out) and do not pad much more
// than the middle ones.  us on middle / large tiles, float32: 131072 rows in 64 groups, 2048 x 1024 555 / 477, 1024 x 2048 531 / 488,
// 512 x 1024 (two rounds) 239 / 380, 264 x 4096 (a third more padding) 342 / 387; 65536 rows in 16 groups, 1800 x 2048 351 / 313.
template <int CBSZ, int BLGP>
int launch_wgrad_shape(GroupedWgradArgs& a, hipStream_t st)
{
    const int64_t middle = (int64_t)a.E * ceil_div(a.N, 128) * ceil_div(a.Kl, 128);
    const int64_t large = (int64_t)a.E * ceil_div(a.N, 256) * ceil_div(a.Kl, 256);
    if (middle < 512) return launch_wgrad<64, 64, 4, CBSZ, BLGP>(a, st);
    if (large < 1024 || 4 * large * 5 > middle * 6) return launch_wgrad<128, 128, 2, CBSZ, BLGP>(a, st);
    return launch_wgrad<256, 256, 2, CBSZ, BLGP, 8>(a, st);
}

bool fp8_code(int v) { return v == MI8_E4M3 || v == MI8_E5M2; }

}  // namespace
}  // namespace mi8

using namespace mi8;

namespace {
int grouped_gemm_entry(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                       int64_t b_group_stride, const int64_t* group_sizes, int32_t num_groups, int64_t T, int64_t N,
                       int64_t K, const float* sa, const float* sb, int64_t sb_group_stride, void* out, int out_dtype,
                       int64_t ldc, bool accumulate, void* stream)
{
    MI8_REQUIRE(a && b && group_sizes && sa && sb && out, MI8_ERR_ARG, "mi8_grouped_gemm_fp8: null pointer");
    MI8_REQUIRE(fp8_code(a_dtype) && fp8_code(b_dtype), MI8_ERR_ARG, "mi8_grouped_gemm_fp8: unknown fp8 dtype");
    MI8_REQUIRE(out_dtype == MI8_BF16 || out_dtype == MI8_F32, MI8_ERR_ARG, "mi8_grouped_gemm_fp8: unknown output dtype");
    MI8_REQUIRE(T > 0 && N > 0 && K > 0 && num_groups > 0, MI8_ERR_ARG, "mi8_grouped_gemm_fp8: empty problem");
    MI8_REQUIRE(K % 16 == 0 && lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K && b_group_stride % 16 == 0,
                MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8: K, lda, ldb and the group stride must be multiples of 16, lda, ldb >= K");
    MI8_REQUIRE(ldc >= N, MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8: ldc < N");
    MI8_REQUIRE(aligned16(a) && aligned16(b), MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8: operands must be 16-byte aligned");
    MI8_REQUIRE(N * ldb < ((int64_t)1 << 32) && T < (1 << 30) && N < (1 << 30) && K < (1 << 30), MI8_ERR_UNSUPPORTED,
                "mi8_grouped_gemm_fp8: operand too large");
    // (a ring tile addresses its rows of A, 128 or, in the smallest, 32, with 32-bit byte offsets)
    const bool whole_a_fits = T <= (((int64_t)1 << 32) - 1) / lda;
    MI8_REQUIRE(whole_a_fits || lda < (1 << 27), MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8: lda (%lld) of 2^27 or more and an operand of 4 GiB or more",
                (long long)lda);
    GroupedArgs g{(const uint8_t*)a, (const uint8_t*)b, out, out_dtype == MI8_F32 ? 1 : 0, lda, ldb, ldc,
                  b_group_stride, sb_group_stride, group_sizes, num_groups, T, (int)N, (int)K, sa, sb, 0,
                  accumulate ? 1 : 0};
    hipStream_t st = (hipStream_t)stream;
    // the persistent kernel takes full-tile shapes with bf16 output (it rewrites the overlap of its shifted last tile
    // column when N is not a multiple of 256: not possible when accumulating)
    const bool fits = out_dtype == MI8_BF16 && T >= 256 && N >= 256 && K % 128 == 0 && N % 8 == 0 && ldc % 8 == 0 && aligned16(out) &&
        sb_group_stride % 4 == 0 && aligned16(sb) && lda < (1 << 23) && ldb < (1 << 23) && ldc < (1 << 22) &&
        (!accumulate || N % 256 == 0);
    const GroupedKernel k = whole_a_fits || lda < (1 << 25) ? choose_grouped(T, num_groups, N, K, fits) : kRing32;
    if (k == kPersistent)
        return launch_m16_grouped((const uint8_t*)a, a_dtype, lda, (const uint8_t*)b, b_dtype, ldb, b_group_stride,
                                   group_sizes, num_groups, T, (int)N, (int)K, sa, sb, sb_group_stride, (uint16_t*)out,
                                   ldc, accumulate, st);
    if (a_dtype == MI8_E4M3)
        return b_dtype == MI8_E4M3 ? launch_grouped_shape<0, 0>(g, k, st) : launch_grouped_shape<0, 1>(g, k, st);
    return b_dtype == MI8_E4M3 ? launch_grouped_shape<1, 0>(g, k, st) : launch_grouped_shape<1, 1>(g, k, st);
}
}  // namespace

extern "C" int mi8_grouped_gemm_fp8(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype, int64_t ldb,
                                    int64_t b_group_stride, const int64_t* group_sizes, int32_t num_groups, int64_t T,
                                    int64_t N, int64_t K, const float* sa, const float* sb, int64_t sb_group_stride,
                                    void* out, int out_dtype, int64_t ldc, void* stream)
{
    return grouped_gemm_entry(a, a_dtype, lda, b, b_dtype, ldb, b_group_stride, group_sizes, num_groups, T, N, K, sa, sb,
                              sb_group_stride, out, out_dtype, ldc, false, stream);
}

extern "C" int mi8_grouped_gemm_fp8_accumulate(const void* a, int a_dtype, int64_t lda, const void* b, int b_dtype,
                                               int64_t ldb, int64_t b_group_stride, const int64_t* group_sizes,
                                               int32_t num_groups, int64_t T, int64_t N, int64_t K, const float* sa,
                                               const float* sb, int64_t sb_group_stride, void* out, int out_dtype,
                                               int64_t ldc, void* stream)
{
    return grouped_gemm_entry(a, a_dtype, lda, b, b_dtype, ldb, b_group_stride, group_sizes, num_groups, T, N, K, sa, sb,
                              sb_group_stride, out, out_dtype, ldc, true, stream);
}

extern "C" int mi8_grouped_gemm_fp8_dual_supported(int64_t T, int64_t N, int64_t K1, int64_t K2)
{
    return (T >= 256 && T < (1 << 30) && N >= 256 && N % 8 == 0 && N < (1 << 30) && K1 >= 256 && K2 >= 256 && K1 % 256 == 0 &&
            K2 % 256 == 0 && K1 < (1 << 30) && K2 < (1 << 30))
               ? 1
               : 0;
}

extern "C" int mi8_grouped_gemm_fp8_dual(const void* a1, const void* a2, int a_dtype, int64_t lda, const void* b1,
                                         const void* b2, int b_dtype, int64_t ldb, int64_t b_group_stride,
                                         const int64_t* group_sizes, int32_t num_groups, int64_t T, int64_t N, int64_t K1,
                                         int64_t K2, const float* sa1, const float* sa2, const float* sb1, const float* sb2,
                                         int64_t sb_group_stride, void* out, int64_t ldc, void* stream)
{
    MI8_REQUIRE(a1 && a2 && b1 && b2 && group_sizes && sa1 && sa2 && sb1 && sb2 && out, MI8_ERR_ARG,
                "mi8_grouped_gemm_fp8_dual: null pointer");
    MI8_REQUIRE(fp8_code(a_dtype) && fp8_code(b_dtype), MI8_ERR_ARG, "mi8_grouped_gemm_fp8_dual: unknown fp8 dtype");
    MI8_REQUIRE(num_groups > 0, MI8_ERR_ARG, "mi8_grouped_gemm_fp8_dual: no groups");
    MI8_REQUIRE(mi8_grouped_gemm_fp8_dual_supported(T, N, K1, K2), MI8_ERR_UNSUPPORTED,
                "mi8_grouped_gemm_fp8_dual: needs T, N >= 256, N %% 8 == 0 and K1, K2 multiples of 256 (got T=%lld N=%lld K1=%lld "
                "K2=%lld); use mi8_grouped_gemm_fp8 and mi8_grouped_gemm_fp8_accumulate",
                (long long)T, (long long)N, (long long)K1, (long long)K2);
    const int64_t kmax = K1 > K2 ? K1 : K2;
    MI8_REQUIRE(lda % 16 == 0 && ldb % 16 == 0 && lda >= kmax && ldb >= kmax && b_group_stride % 16 == 0 && lda < (1 << 23) &&
                    ldb < (1 << 23),
                MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8_dual: lda, ldb and the group stride must be multiples of 16, lda, ldb >= K1, K2 and below 2^23");
    MI8_REQUIRE(ldc >= N && ldc % 8 == 0 && ldc < (1 << 22) && aligned16(out), MI8_ERR_UNSUPPORTED,
                "mi8_grouped_gemm_fp8_dual: the output needs ldc >= N, ldc %% 8 == 0 and 16-byte alignment");
    MI8_REQUIRE(aligned16(a1) && aligned16(a2) && aligned16(b1) && aligned16(b2) && aligned16(sb1) && aligned16(sb2) &&
                    sb_group_stride % 4 == 0,
                MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8_dual: operands and column scales must be 16-byte aligned");
    MI8_REQUIRE(N * ldb < ((int64_t)1 << 32), MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8_dual: operand too large");
    const int64_t m_tiles = ceil_div(T, 256) + num_groups;
    MI8_REQUIRE(m_tiles * ceil_div(N, 256) < ((int64_t)1 << 30), MI8_ERR_UNSUPPORTED, "mi8_grouped_gemm_fp8_dual: grid too large");
    return launch_m16_grouped_dual((const uint8_t*)a1, (const uint8_t*)a2, a_dtype, lda, (const uint8_t*)b1, (const uint8_t*)b2,
                                   b_dtype, ldb, b_group_stride, group_sizes, num_groups, T, (int)N, (int)K1, (int)K2, sa1, sa2,
                                   sb1, sb2, sb_group_stride, (uint16_t*)out, ldc, (hipStream_t)stream);
}

extern "C" int mi8_grouped_wgrad_fp8(const void* a_t, int a_dtype, const void* b_t, int b_dtype, int64_t ld_t,
                                     const int64_t* group_sizes, int32_t num_groups, int64_t T, int64_t N, int64_t Kl,
                                     const float* sa, const float* sb, void* out, int out_dtype, void* stream)
{
    MI8_REQUIRE(a_t && b_t && group_sizes && sa && sb && out, MI8_ERR_ARG, "mi8_grouped_wgrad_fp8: null pointer");
    MI8_REQUIRE(fp8_code(a_dtype) && fp8_code(b_dtype), MI8_ERR_ARG, "mi8_grouped_wgrad_fp8: unknown fp8 dtype");
    MI8_REQUIRE(out_dtype == MI8_BF16 || out_dtype == MI8_F32, MI8_ERR_ARG, "mi8_grouped_wgrad_fp8: unknown output dtype");
    MI8_REQUIRE(T > 0 && N > 0 && Kl > 0 && num_groups > 0, MI8_ERR_ARG, "mi8_grouped_wgrad_fp8: empty problem");
    MI8_REQUIRE(ld_t % 16 == 0 && ld_t >= mi8_grouped_padded_rows(T, num_groups), MI8_ERR_UNSUPPORTED,
                "mi8_grouped_wgrad_fp8: ld_t (%lld) must be a multiple of 16 and at least mi8_grouped_padded_rows()",
                (long long)ld_t);
    MI8_REQUIRE(aligned16(a_t) && aligned16(b_t), MI8_ERR_UNSUPPORTED, "mi8_grouped_wgrad_fp8: operands must be 16-byte aligned");
    MI8_REQUIRE(N * ld_t < ((int64_t)1 << 32) && Kl * ld_t < ((int64_t)1 << 32), MI8_ERR_UNSUPPORTED,
                "mi8_grouped_wgrad_fp8: operand larger than 4 GiB");
    GroupedWgradArgs g{(const uint8_t*)a_t, (const uint8_t*)b_t, ld_t, group_sizes, num_groups, T, (int)N, (int)Kl,
                       sa, sb, out, out_dtype == MI8_F32 ? 1 : 0, 0, 0};
    hipStream_t st = (hipStream_t)stream;
    if (out_dtype == MI8_BF16 && N >= 256 && Kl >= 256 && Kl % 8 == 0 && aligned16(out) && aligned16(sb) &&
        ld_t % 128 == 0 && ld_t < (1 << 23))
        return launch_m16_grouped_wgrad((const uint8_t*)a_t, a_dtype, (const uint8_t*)b_t, b_dtype, ld_t, group_sizes,
                                         num_groups, T, (int)N, (int)Kl, sa, sb, (uint16_t*)out, st);
    if (a_dtype == MI8_E4M3)
        return b_dtype == MI8_E4M3 ? launch_wgrad_shape<0, 0>(g, st) : launch_wgrad_shape<0, 1>(g, st);
    return b_dtype == MI8_E4M3 ? launch_wgrad_shape<1, 0>(g, st) : launch_wgrad_shape<1, 1>(g, st);
}
