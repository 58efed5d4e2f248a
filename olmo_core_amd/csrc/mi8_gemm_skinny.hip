// Scaled float8 GEMM for a few rows of A:  C[M,N] = (A[M,K] . B[N,K]^T) * (1/sa) * (1/sb),  M <= 64.
//
// This is the shape of a generation loop (a handful of tokens against a weight matrix): the arithmetic is
// nothing, the time is reading B once, so the kernel is built to keep HBM busy rather than the matrix cores.
// A tiled kernel does badly here: the few tiles it finds occupy a few compute units, and each walks all of K
// with one memory latency per 128-byte step.
//
// One workgroup owns 16 (M <= 16) or 32 rows of B (columns of C) and all of A; its eight waves each take a
// contiguous eighth of K, so N/16 or N/32 workgroups x 8 waves stream disjoint pieces of B straight from global
// memory into MFMA operand registers (no LDS staging: nothing is reused inside a wave).  v_mfma_f32_16x16x128
// takes 16 rows x 128 bytes per operand, lane l feeding bytes 32*(l/16)..+31 of row l%16 - the B rows go in
// as the first operand, blocks of 16 rows of A as the second, and the 16 x 16 result is C transposed:
// element j of lane l is C[m = l%16][n = 4*(l/16) + j].  Loads of several 128-byte steps are issued before
// the first MFMA of a batch so that every wave has a few KB in flight.  The eight partial results meet in
// LDS and waves 0..MT-1 scale, round and store one block of 16 rows of C each.
//
// A (at most 64 x K bytes) is re-read by every workgroup and stays in L2; with more than 16 rows of A that
// traffic would exceed the read of B, so a workgroup then takes 32 rows of B per pass over A.  Rows of A past M and rows of B past N
// are clamped to the last valid row and their results dropped; K bytes past K (K % 16 == 0) are fed as zeros.
#include "mi8_gemm.h"
#include "mi8_swiglu.h"

namespace mi8 {
namespace gemm {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kSkinnyWaves = 8;  // K slices per workgroup
constexpr int kStep = 128;       // K bytes per MFMA

// 16 bytes of an operand row, or zeros past the end of K
__device__ __forceinline__ v4i load16(const uint8_t* p, bool ok)
{
    return ok ? *reinterpret_cast<const v4i*>(p) : v4i{0, 0, 0, 0};
}

// MT: blocks of 16 rows of A; NB: blocks of 16 rows of B per workgroup (each wave's A fragments serve NB MFMAs,
// which divides the L2 traffic of re-reading A by NB); U: 128-byte steps loaded ahead of their MFMAs; TW / TX:
// MFMA type codes of the B rows (first operand) and the A rows (second operand), 0 = e4m3, 1 = e5m2.
template <int MT, int NB, int U, int TW, int TX>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm_fp8_skinny_kernel(GemmArgs g)
{
    __shared__ v4f red[kSkinnyWaves][MT][64];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int n0 = (int)blockIdx.x * (16 * NB);

    const uint8_t* wp[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int n = n0 + nb * 16 + r16 < g.N ? n0 + nb * 16 + r16 : g.N - 1;
        wp[nb] = g.B + (int64_t)n * g.ldb + kg * 32;
    }
    const uint8_t* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + r16 < g.M ? mt * 16 + r16 : g.M - 1;
        xp[mt] = g.A + (int64_t)m * g.lda + kg * 32;
    }

    const int steps = (g.K + kStep - 1) / kStep;
    const int per_wave = (steps + kSkinnyWaves - 1) / kSkinnyWaves;
    const int s_begin = wave * per_wave;
    const int s_end = s_begin + per_wave < steps ? s_begin + per_wave : steps;

    v4f acc[NB][MT];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = v4f{0, 0, 0, 0};

    for (int s = s_begin; s < s_end; s += U) {
        v4i w[U][NB][2], x[U][MT][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t off = (int64_t)(s + u) * kStep;
            const int k = (s + u) * kStep + kg * 32;  // this lane's first K byte of the step
            const bool in = s + u < s_end;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool ok = in && k + 16 * h < g.K;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) w[u][nb][h] = load16(wp[nb] + off + 16 * h, ok);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[u][mt][h] = load16(xp[mt] + off + 16 * h, ok);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const v8i fx = __builtin_shufflevector(x[u][mt][0], x[u][mt][1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const v8i fw = __builtin_shufflevector(w[u][nb][0], w[u][nb][1], 0, 1, 2, 3, 4, 5, 6, 7);
                    acc[nb][mt] =
                        __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fw, fx, acc[nb][mt], TW, TX, 0, 0, 0, 0);
                }
            }
        }
    }

    // same scale arithmetic as the tiled kernels: IEEE division for single scales, v_rcp_f32 for scale vectors
    const int m = (wave < MT ? wave : 0) * 16 + r16;  // wave mt finishes block mt of the rows of A
    const bool m_ok = wave < MT && m < g.M;
    const float isa = !m_ok ? 0.0f : g.sa_vec ? __builtin_amdgcn_rcpf(g.sa[m]) : 1.0f / g.sa[0];
    const float isb_scalar = g.sb_vec ? 0.0f : 1.0f / g.sb[0];
    const bool both_single = !g.sa_vec && !g.sb_vec;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (nb > 0) __syncthreads();  // the previous block's sums have been read
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red[wave][mt][lane] = acc[nb][mt];
        __syncthreads();
        if (!m_ok) continue;
        v4f sum = red[0][wave][lane];
#pragma unroll
        for (int w2 = 1; w2 < kSkinnyWaves; ++w2) sum += red[w2][wave][lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + nb * 16 + kg * 4 + j;
            if (n >= g.N) continue;
            const float isb = g.sb_vec ? __builtin_amdgcn_rcpf(g.sb[n]) : isb_scalar;
            float v = both_single ? sum[j] * (isa * isb) : sum[j] * isa * isb;
            if (g.c_f32 == 2) v = round_to_bf16(v);
            if (g.c_f32) {
                float* c = reinterpret_cast<float*>(g.C) + (int64_t)m * g.ldc + n;
                *c = g.accumulate ? *c + v : v;
            } else {
                uint16_t* c = reinterpret_cast<uint16_t*>(g.C) + (int64_t)m * g.ldc + n;
                uint16_t h = f32_to_bf16_bits(v);
                if (g.accumulate) h = f32_to_bf16_bits(bits_to_f32((uint32_t)*c << 16) + bits_to_f32((uint32_t)h << 16));
                *c = h;
            }
        }
    }
}

template <int MT, int NB, int U>
int launch_skinny_typed(const GemmArgs& g, int a_dtype, int b_dtype, hipStream_t st)
{
    const dim3 grid((g.N + 16 * NB - 1) / (16 * NB)), block(kSkinnyWaves * 64);
    const bool we5 = b_dtype == MI8_E5M2, xe5 = a_dtype == MI8_E5M2;
    if (!we5 && !xe5) hipLaunchKernelGGL((gemm_fp8_skinny_kernel<MT, NB, U, 0, 0>), grid, block, 0, st, g);
    if (!we5 && xe5) hipLaunchKernelGGL((gemm_fp8_skinny_kernel<MT, NB, U, 0, 1>), grid, block, 0, st, g);
    if (we5 && !xe5) hipLaunchKernelGGL((gemm_fp8_skinny_kernel<MT, NB, U, 1, 0>), grid, block, 0, st, g);
    if (we5 && xe5) hipLaunchKernelGGL((gemm_fp8_skinny_kernel<MT, NB, U, 1, 1>), grid, block, 0, st, g);
    return launch_status("mi8_gemm_fp8");
}

// ---- the same for a generation step of a SwiGLU block: activations quantised by the GEMM that reads them ------------
//
// A step on one token is a chain of launches that each wait for the one before: cast, two projections, SwiGLU, cast,
// projection.  The arithmetic on the activations is so small that every workgroup can repeat it: KIND says how the
// kernel gets its float8 rows of A,
//   kFp8      they are in memory with their scale,
//   kSlots    A is bf16 and partial maxima of |A| are in memory (left by the launch that produced A): every workgroup
//             folds them into the scale and converts A into LDS,
//   kAmax     A is bf16 and small: every workgroup takes the amax itself as well.
// DUAL: 16 rows of B and the same 16 rows of a second matrix B3 per workgroup, x1 = A B^T, x3 = A B3^T; the epilogue
// rounds both to bf16 and stores only h = silu(x1) * x3, with a partial maximum of |h| per workgroup.
// The time is streaming B: a wave's next step is on its way while it works on one, the first while A is quantised, and
// the registers leave room for three workgroups a compute unit, so that the 688 of 11008 rows run in one round (with two
// fitting: 28 us for 90 MB; converting in registers instead of LDS: 17.7 us for 45 MB).
// Bytes, scales and sums are those of the separate launches.
enum FewRowsInput { kFp8, kSlots, kAmax };

struct FewRowsArgs {
    GemmArgs g;  // kSlots, kAmax: A is bf16, lda counts its elements, sa is unused
    const uint8_t* B3;
    const float* sb3;
    const uint32_t* slots_in;  // kSlots
    int n_slots;
    bool pow2;
    uint32_t* slots_out;  // DUAL: one per workgroup
};

constexpr int kFewThreads = kSkinnyWaves * 64;
constexpr int kAmaxVecs = 4;  // 8-element groups of A per lane where every workgroup takes the amax
constexpr int kLdsElems = 65536;  // bytes of LDS for A where partial maxima are given

// eight bf16 values -> eight e4m3 bytes
__device__ __forceinline__ uint2 quantise8(uint4 v, float s)
{
    float f[8];
    unpack8(v, f);
    return make_uint2(quant4<MI8_E4M3, false>(f[0], f[1], f[2], f[3], s, s, s, s),
                      quant4<MI8_E4M3, false>(f[4], f[5], f[6], f[7], s, s, s, s));
}

// WHOLE: a wave's share of K is at most U steps, all of which it requests at the start.
template <int MT, int U, int KIND, bool DUAL, bool WHOLE>
__global__ __launch_bounds__(kFewThreads, WHOLE ? (U > 8 ? 2 : 4) : MT == 1 ? 6 : MT == 2 ? 4 : 2) void few_rows_kernel(FewRowsArgs a)
{
    constexpr int NB = DUAL ? 2 : 1;
    constexpr int UX = WHOLE ? 1 : U;  // steps of A read ahead
    extern __shared__ __attribute__((aligned(16))) uint8_t aq[];  // kSlots, kAmax: A in e4m3, [M][K]
    __shared__ v4f red[kSkinnyWaves][MT][64];
    __shared__ uint32_t smem[kSkinnyWaves];
    const GemmArgs& g = a.g;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int n0 = (int)blockIdx.x * 16;
    const int n_row = n0 + r16 < g.N ? n0 + r16 : g.N - 1;

    const int steps = (g.K + kStep - 1) / kStep;
    const int per_wave = (steps + kSkinnyWaves - 1) / kSkinnyWaves;
    const int s_begin = wave * per_wave;
    const int s_end = s_begin + per_wave < steps ? s_begin + per_wave : steps;

    const uint8_t* wp[NB];
    wp[0] = g.B + (int64_t)n_row * g.ldb + kg * 32;
    if constexpr (DUAL) wp[1] = a.B3 + (int64_t)n_row * g.ldb + kg * 32;
    v4i w[U][NB][2], w_next[WHOLE ? 1 : U][NB][2];
    auto inside = [&](int s, int h) { return s < s_end && s * kStep + kg * 32 + 16 * h < g.K; };
    auto load_w = [&](auto& to, int s) {
#pragma unroll
        for (int u = 0; u < (int)(sizeof(to) / sizeof(to[0])); ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    to[u][nb][h] = load16(wp[nb] + (int64_t)(s + u) * kStep + 16 * h, inside(s + u, h));
    };
    load_w(w, s_begin);

    float scale;
    if constexpr (KIND == kFp8) {
        scale = g.sa[0];
    } else {
        uint32_t m = 0;
        const int per_row = g.K / 8, groups = g.M * per_row;
        uint4 v[KIND == kAmax ? kAmaxVecs : 1];
        if constexpr (KIND == kSlots) {
            for (int i = threadIdx.x; i < a.n_slots; i += kFewThreads) m = umax32(m, a.slots_in[i]);
        } else {  // contiguous, at most kFewThreads * kAmaxVecs groups
#pragma unroll
            for (int i = 0; i < kAmaxVecs; ++i) {
                const int k = (int)threadIdx.x + kFewThreads * i;
                v[i] = k < groups ? reinterpret_cast<const uint4*>(g.A)[k] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < kAmaxVecs; ++i) m = umax32(m, (max_code8(v[i].x, v[i].y, v[i].z, v[i].w) & 0xFFFFu) << 16);
        }
        m = wave_umax(m);
        if (lane == 0) smem[wave] = m;
        __syncthreads();
        m = 0;
#pragma unroll
        for (int i = 0; i < kSkinnyWaves; ++i) m = umax32(m, smem[i]);
        scale = scale_from_amax_bits<MI8_E4M3>(m, a.pow2);
        if constexpr (KIND == kAmax) {
#pragma unroll
            for (int i = 0; i < kAmaxVecs; ++i) {
                const int k = (int)threadIdx.x + kFewThreads * i;
                if (k < groups) reinterpret_cast<uint2*>(aq)[k] = quantise8(v[i], scale);
            }
        } else {
            for (int k = threadIdx.x; k < groups; k += kFewThreads) {
                const int r = k / per_row, c = k - r * per_row;
                const uint16_t* row = reinterpret_cast<const uint16_t*>(g.A) + (int64_t)r * g.lda;
                reinterpret_cast<uint2*>(aq)[k] = quantise8(*reinterpret_cast<const uint4*>(row + 8 * c), scale);
            }
        }
        __syncthreads();
    }

    const uint8_t* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + r16 < g.M ? mt * 16 + r16 : g.M - 1;
        xp[mt] = (KIND == kFp8 ? g.A + (int64_t)m * g.lda : aq + m * g.K) + kg * 32;
    }

    v4f acc[NB][MT];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = v4f{0, 0, 0, 0};

    v4i x[UX][MT][2], x_next[UX][MT][2];
    auto load_x = [&](v4i(&to)[UX][MT][2], int s) {
#pragma unroll
        for (int u = 0; u < UX; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    to[u][mt][h] = load16(xp[mt] + (int64_t)(s + u) * kStep + 16 * h, inside(s + u, h));
    };
    auto step = [&](const v4i(&xs)[MT][2], const v4i(&ws)[NB][2]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const v8i fx = __builtin_shufflevector(xs[mt][0], xs[mt][1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const v8i fw = __builtin_shufflevector(ws[nb][0], ws[nb][1], 0, 1, 2, 3, 4, 5, 6, 7);
                acc[nb][mt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fw, fx, acc[nb][mt], 0, 0, 0, 0, 0, 0);
            }
        }
    };
    load_x(x, s_begin);
    if constexpr (WHOLE) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s_begin + u >= s_end) break;
            load_x(u & 1 ? x : x_next, s_begin + u + 1);
            step(u & 1 ? x_next[0] : x[0], w[u]);
        }
    } else {
        for (int s = s_begin; s < s_end; s += U) {
            load_w(w_next, s + U);
            load_x(x_next, s + U);
#pragma unroll
            for (int u = 0; u < U; ++u) step(x[u], w[u]);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int h = 0; h < 2; ++h) w[u][nb][h] = w_next[u][nb][h];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int h = 0; h < 2; ++h) x[u][mt][h] = x_next[u][mt][h];
        }
    }

    const int m = (wave < MT ? wave : 0) * 16 + r16;  // wave mt finishes block mt of the rows of A
    const int n = n0 + kg * 4;                        // four columns of C per lane (N % 4 == 0)
    const bool ok = wave < MT && m < g.M && n < g.N;
    const float isa = 1.0f / scale;
    uint2 c[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (nb > 0) __syncthreads();  // the previous matrix's sums have been read
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red[wave][mt][lane] = acc[nb][mt];
        __syncthreads();
        c[nb] = make_uint2(0, 0);
        if (!ok) continue;
        v4f sum = red[0][wave][lane];
#pragma unroll
        for (int w2 = 1; w2 < kSkinnyWaves; ++w2) sum += red[w2][wave][lane];
        const float f = isa * (1.0f / (nb ? a.sb3[0] : g.sb[0]));
        c[nb] = make_uint2(pack_bf16x2(sum[0] * f, sum[1] * f), pack_bf16x2(sum[2] * f, sum[3] * f));
    }
    uint2 out = c[0];
    if constexpr (DUAL) out = swiglu_fwd4(c[0], c[NB - 1]);
    if (ok) *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.C) + (int64_t)m * g.ldc + n) = out;
    if constexpr (DUAL) {
        uint32_t hm = ok ? (max_code8(out.x, out.y, out.x, out.y) & 0xFFFFu) << 16 : 0u;
        hm = wave_umax(hm);
        if (lane == 0) smem[wave] = hm;  // (the reads of smem above are two barriers back)
        __syncthreads();
        if (threadIdx.x == 0) {
            hm = 0;
#pragma unroll
            for (int w2 = 0; w2 < MT; ++w2) hm = umax32(hm, smem[w2]);
            a.slots_out[blockIdx.x] = hm;
        }
    }
}

template <int MT, int U, int KIND, bool DUAL, bool WHOLE = false>
int launch_few_rows(const FewRowsArgs& a, hipStream_t st, const char* what)
{
    static std::atomic<uint64_t> configured;
    if constexpr (KIND == kSlots)
        if (int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(few_rows_kernel<MT, U, KIND, DUAL, WHOLE>), kLdsElems, configured, what))
            return rc;
    const int lds = KIND == kFp8 ? 0 : a.g.M * a.g.K;  // (K % 16 == 0)
    hipLaunchKernelGGL((few_rows_kernel<MT, U, KIND, DUAL, WHOLE>), dim3((a.g.N + 15) / 16), dim3(kFewThreads), lds, st, a);
    return launch_status(what);
}

}  // namespace

int launch_skinny(GemmArgs& g, int a_dtype, int b_dtype, hipStream_t st)
{
    if (g.M > kSkinnyMaxM) {
        set_error("mi8_gemm_fp8: the few-rows variant takes M <= %d (M=%d)", kSkinnyMaxM, g.M);
        return MI8_ERR_UNSUPPORTED;
    }
    if (g.M <= 16) return launch_skinny_typed<1, 1, 4>(g, a_dtype, b_dtype, st);
    if (g.M <= 32) return launch_skinny_typed<2, 2, 2>(g, a_dtype, b_dtype, st);
    return launch_skinny_typed<4, 2, 2>(g, a_dtype, b_dtype, st);
}

}  // namespace gemm
}  // namespace mi8

using namespace mi8;
using namespace mi8::gemm;

namespace {
// Whether the float8 rows go to the ring tiles (mi8_gemm.hip), which fetch A once per 32 columns of both products where the
// kernel above reads it from L2 for every 16: more rows, or more bytes of weights, make that the time.  us, above / ring:
// 16 x 8192 x 2048 9.9 / 9.0, 23 x 11008 x 4096 28.5 / 25.3, 48 x 11008 x 4096 43.6 / 27.1, 64 x 8192 x 2048 18.5 / 9.3,
// 4 x 27648 x 5120 66.6 / 56.6, 64 x 27648 x 5120 135 / 70; 8 x 11008 x 4096 24.3 / 24.2, 32 x 2816 x 1024 5.6 / 5.8.
// The line at 200 MB for four rows, below it 20480 x 4096 36.0 / 37.2, 32768 x 2048 28.3 / 30.0, 12288 x 8192 41.1 / 40.2, above
// 20480 x 5120 49.4 / 43.1, 27648 x 4096 46.6 / 45.3, 24576 x 6144 62.5 / 53.5, 22016 x 8192 72.1 / 67.5, 28672 x 8192 86.2 / 85.9.
// Ring tiles address the rows of a tile, all of A and 32 of each matrix, with 32-bit offsets; the kernel above with 64-bit ones.
bool dual_on_ring(int64_t M, int64_t H, int64_t K, int64_t lda, int64_t ldb)
{
    constexpr int64_t most = (int64_t)1 << 32;
    if (lda >= most || ldb >= most || M * lda >= most || 32 * ldb >= most) return false;
    const int64_t bytes = 2 * H * K;
    return M > 32 || (bytes >= 16 << 20 && M > 8) || (bytes >= 200 << 20 && M > 3);
}
}  // namespace

extern "C" int32_t mi8_few_rows_swiglu_slots(int64_t M, int64_t H, int64_t K, int x_is_fp8)
{
    return x_is_fp8 && dual_on_ring(M, H, K, K, K) ? dual_ring_slots(H) : (int32_t)((H + 15) / 16);
}

extern "C" int mi8_few_rows_swiglu(const void* x, int x_is_fp8, int64_t lda, const float* sx, const void* b1, const void* b3,
                                   int64_t ldb, int64_t M, int64_t H, int64_t K, const float* sb1, const float* sb3,
                                   uint32_t flags, void* h, uint32_t* slots_h, int32_t* n_slots_used, void* stream)
{
    MI8_REQUIRE(x && b1 && b3 && sb1 && sb3 && h && slots_h && n_slots_used && (!x_is_fp8 || sx), MI8_ERR_ARG,
                "mi8_few_rows_swiglu: null pointer");
    MI8_REQUIRE(M > 0 && M <= kSkinnyMaxM && H > 0 && H <= 16 * MI8_AMAX_SLOTS && H % 8 == 0 && K > 0 && K % 16 == 0 &&
                    K < (1 << 30),
                MI8_ERR_UNSUPPORTED,
                "mi8_few_rows_swiglu: needs 1..%d rows, H %% 8 == 0 up to %d, K %% 16 == 0 (got %lld x %lld x %lld)", kSkinnyMaxM,
                16 * MI8_AMAX_SLOTS, (long long)M, (long long)H, (long long)K);
    MI8_REQUIRE(x_is_fp8 || (M * K <= (int64_t)kFewThreads * kAmaxVecs * 8 && M <= 16 && lda == K), MI8_ERR_UNSUPPORTED,
                "mi8_few_rows_swiglu: bf16 rows must be contiguous, at most 16 of them and at most %d elements (got %lld x %lld); "
                "use mi8_cast_tensorwise",
                kFewThreads * kAmaxVecs * 8, (long long)M, (long long)K);
    MI8_REQUIRE(lda >= K && ldb >= K && lda % 16 == 0 && ldb % 16 == 0, MI8_ERR_UNSUPPORTED,
                "mi8_few_rows_swiglu: pitches must be multiples of 16 and at least K");
    MI8_REQUIRE(aligned16(x) && aligned16(b1) && aligned16(b3) && aligned16(h), MI8_ERR_UNSUPPORTED,
                "mi8_few_rows_swiglu: pointers must be 16-byte aligned");
    FewRowsArgs a{};
    a.g = GemmArgs{(const uint8_t*)x, (const uint8_t*)b1, h, 0, lda, ldb, H, (int)M, (int)H, (int)K, sx, sb1, 0, 0, 0, 0, 0};
    a.B3 = (const uint8_t*)b3;
    a.sb3 = sb3;
    a.pow2 = (flags & MI8_FLAG_POW2_SCALE) != 0;
    a.slots_out = slots_h;
    const bool on_ring = x_is_fp8 && dual_on_ring(M, H, K, lda, ldb);
    *n_slots_used = on_ring ? dual_ring_slots(H) : (int32_t)((H + 15) / 16);
    hipStream_t st = (hipStream_t)stream;
    if (!x_is_fp8) return launch_few_rows<1, 1, kAmax, true>(a, st, "mi8_few_rows_swiglu");
    if (on_ring) {
        a.g.B3 = a.B3;
        a.g.sb3 = sb3;
        a.g.slots_out = slots_h;
        return launch_dual_ring(a.g, st);
    }
    if (M <= 16) return launch_few_rows<1, 1, kFp8, true>(a, st, "mi8_few_rows_swiglu");
    if (M <= 32) return launch_few_rows<2, 1, kFp8, true>(a, st, "mi8_few_rows_swiglu");
    return launch_few_rows<4, 1, kFp8, true>(a, st, "mi8_few_rows_swiglu");  // (rows too far apart for ring tiles)
}

extern "C" int mi8_few_rows_cast_gemm(const void* x, int64_t lda, const uint32_t* slots, int32_t n_slots, const void* b,
                                      int64_t ldb, int64_t M, int64_t N, int64_t K, const float* sb, uint32_t flags,
                                      void* out, int64_t ldc, void* stream)
{
    MI8_REQUIRE(x && slots && b && sb && out, MI8_ERR_ARG, "mi8_few_rows_cast_gemm: null pointer");
    MI8_REQUIRE(M > 0 && M <= 16 && N > 0 && N < (1 << 30) && N % 8 == 0 && K > 0 && K % 16 == 0 && K < (1 << 30),
                MI8_ERR_UNSUPPORTED, "mi8_few_rows_cast_gemm: needs 1..16 rows, N %% 8 == 0, K %% 16 == 0 (got %lld x %lld x %lld)",
                (long long)M, (long long)N, (long long)K);
    MI8_REQUIRE(M * K <= kLdsElems, MI8_ERR_UNSUPPORTED, "mi8_few_rows_cast_gemm: at most %d elements (got %lld x %lld); use "
                "mi8_cast_tensorwise and mi8_gemm_fp8", kLdsElems, (long long)M, (long long)K);
    MI8_REQUIRE(n_slots > 0 && n_slots <= MI8_AMAX_SLOTS, MI8_ERR_ARG, "mi8_few_rows_cast_gemm: n_slots %d out of range", n_slots);
    MI8_REQUIRE(lda >= K && ldb >= K && lda % 8 == 0 && ldb % 16 == 0 && ldc >= N && ldc % 4 == 0, MI8_ERR_UNSUPPORTED,
                "mi8_few_rows_cast_gemm: lda must be a multiple of 8, ldb of 16 (both at least K), ldc of 4 and at least N");
    MI8_REQUIRE(aligned16(x) && aligned16(b) && aligned16(out), MI8_ERR_UNSUPPORTED,
                "mi8_few_rows_cast_gemm: pointers must be 16-byte aligned");
    FewRowsArgs a{};
    a.g = GemmArgs{(const uint8_t*)x, (const uint8_t*)b, out, 0, lda, ldb, ldc, (int)M, (int)N, (int)K, nullptr, sb, 0, 0, 0, 0, 0};
    a.slots_in = slots;
    a.n_slots = n_slots;
    a.pow2 = (flags & MI8_FLAG_POW2_SCALE) != 0;
    // Where all workgroups fit on the chip at once with the registers for it (one to a compute unit up to N = 4096, two up to
    // 8192 and eight steps), each wave requests its whole share of K before the maxima are folded and A is converted: all of
    // B is under way meanwhile.
    const char* what = "mi8_few_rows_cast_gemm";
    hipStream_t st = (hipStream_t)stream;
    const int share = eighth_steps(K);
    if (N <= 8192 && share <= 4) return launch_few_rows<1, 4, kSlots, false, true>(a, st, what);
    if (N <= 8192 && share <= 8) return launch_few_rows<1, 8, kSlots, false, true>(a, st, what);
    if (N <= 4096 && share <= 12) return launch_few_rows<1, 12, kSlots, false, true>(a, st, what);
    return launch_few_rows<1, 2, kSlots, false>(a, st, what);
}
