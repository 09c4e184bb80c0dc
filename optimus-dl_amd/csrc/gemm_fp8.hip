// FP8 GEMM entry point: argument checks, kernel choice, and the generic kernel.
//
//   C[M,N] = (A[M,K] . B[N,K]^T) * (sa_inv[i] * sb_inv[j]) (+ bias[j])
//
// Both operands are K-contiguous 8-bit codes ("NT").  Kernels:
//   gemm_tiled.hip : BM x BN block tiles through two LDS stages (few 128x128 tiles and a short K: four)
//   gemm_thin.hip  : small tiles, the waves of a block share K: outputs of few tiles (N % 4 == 0, K % 128 == 0)
//   gemm_deep.hip  : 256x128, 128x192 and 128x128 tiles, one block per compute unit, three LDS stages: outputs of about one tile per unit
//   gemm_pipe.hip  : 256x256 tile, one wave per SIMD, explicit software pipeline
//   gemm_stream.hip: the same pipeline running across tile boundaries, epilogue under the
//                    next tile's MFMAs (any M; N, K multiples of 128); with a split over K for
//                    outputs of few tiles, summed by splitk_reduce_kernel below
//   here           : generic one-wave-per-32x32-tile kernel for any M, N, K % 16 == 0
#include "gemm_common.h"

namespace odl {

// ---------------------------------------------------------------- generic kernel
template <int FA, int FB>
__global__ __launch_bounds__(64) void gemm_nt_generic_kernel(const GemmArgs g) {
    const int64_t tile = blockIdx.x;
    const int64_t m0 = (tile % g.tiles_m) * 32, n0 = (tile / g.tiles_m) * 32;
    const int lane = threadIdx.x, lr = lane % 32, lg = lane / 32;
    const uint8_t *pa = g.a + min(m0 + lr, g.M - 1) * g.K;
    const uint8_t *pb = g.b + min(n0 + lr, g.N - 1) * g.K;
    v16f acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    const v4i zero = {0, 0, 0, 0};
    for (int64_t k0 = 0; k0 < g.K; k0 += 64) {
        const int64_t k = k0 + 32 * lg;                         // K % 16 == 0: each 16-byte chunk is wholly in or out
        const v4i a_lo = k < g.K ? *reinterpret_cast<const v4i *>(pa + k) : zero;
        const v4i a_hi = k + 16 < g.K ? *reinterpret_cast<const v4i *>(pa + k + 16) : zero;
        const v4i b_lo = k < g.K ? *reinterpret_cast<const v4i *>(pb + k) : zero;
        const v4i b_hi = k + 16 < g.K ? *reinterpret_cast<const v4i *>(pb + k + 16) : zero;
        const v8i af = {a_lo.x, a_lo.y, a_lo.z, a_lo.w, a_hi.x, a_hi.y, a_hi.z, a_hi.w};
        const v8i bf = {b_lo.x, b_lo.y, b_lo.z, b_lo.w, b_hi.x, b_hi.y, b_hi.z, b_hi.w};
        acc = mfma_32x32x64<FB, FA>(bf, af, acc);
    }
    if (g.out_dtype == ODL_BF16) store_tile<true, false>(g, acc, m0 + lr, n0 + 4 * lg);
    else store_tile<false, false>(g, acc, m0 + lr, n0 + 4 * lg);
}

// ---------------------------------------------------------------- sum of K splits
// out[m, n] = ((p_0 + p_1) + ... + p_{S-1})[m, n] * (sa[m] * sb[n]) (+ bias[n]), fp32 throughout, one
// rounding to the output type; the partial results are added in split order, so the result does not
// depend on how the splits were scheduled.  Four consecutive columns per lane (N % 4 == 0).
template <bool OUT_BF16>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ parts, int splits, int64_t M, int64_t N,
                                                            const float *__restrict__ sa, int sa_vec, const float *__restrict__ sb,
                                                            int sb_vec, const float *__restrict__ bias, void *__restrict__ out,
                                                            int accumulate) {
    const int64_t quads = M * N / 4, slice = M * N;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < quads; q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = q * 4, m = e / N, n = e % N;
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        f32x4 acc = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(parts + e));
        for (int s = 1; s < splits; ++s) {
            const f32x4 p = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(parts + s * slice + e));
            acc.x = acc.x + p.x; acc.y = acc.y + p.y; acc.z = acc.z + p.z; acc.w = acc.w + p.w;
        }
        const float a = sa[m * sa_vec];
        float v[4] = {acc.x * (a * sb[n * sb_vec]), acc.y * (a * sb[(n + 1) * sb_vec]), acc.z * (a * sb[(n + 2) * sb_vec]),
                      acc.w * (a * sb[(n + 3) * sb_vec])};
        if (bias) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = v[j] + bias[n + j];
        }
        if constexpr (OUT_BF16) {
            u32x2 *dst = reinterpret_cast<u32x2 *>(reinterpret_cast<uint16_t *>(out) + e);
            if (accumulate) {                          // out = out + product: the old value joins the fp32 sum, one rounding
                const u32x2 old = *dst;
                v[0] = v[0] + bf16_lo(old.x); v[1] = v[1] + bf16_hi(old.x); v[2] = v[2] + bf16_lo(old.y); v[3] = v[3] + bf16_hi(old.y);
            }
            *dst = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
            float4 *dst = reinterpret_cast<float4 *>(reinterpret_cast<float *>(out) + e);
            if (accumulate) {
                const float4 old = *dst;
                v[0] = v[0] + old.x; v[1] = v[1] + old.y; v[2] = v[2] + old.z; v[3] = v[3] + old.w;
            }
            *dst = float4{v[0], v[1], v[2], v[3]};
        }
    }
}

// ------------------------------------------------------------------- host side
struct Variant {
    const char *name;
    int bm, bn, threads;     // bm == 0: generic kernel
    float eff;               // relative per-tile efficiency used by the automatic choice
};

static const Variant kVariants[] = {
    {"generic 32x32 (1 wave, no LDS)", 0, 0, 64, 0.05f},
    {"256x256x128 4 waves (128x128 per wave)", 256, 256, 256, 0.25f},
    {"256x256x128 8 waves (128x64 per wave)", 256, 256, 512, 1.00f},
    {"256x128x128 4 waves (128x64 per wave)", 256, 128, 256, 0.85f},
    {"128x128x128 4 waves (64x64 per wave)", 128, 128, 256, 0.70f},
    {"256x256x128 4 waves, software-pipelined, persistent (K % 256 == 0)", 256, 256, 256, 1.10f},
    {"256x256x128 4 waves, software-pipelined, one tile per block", 256, 256, 256, 0.50f},
    {"256x256x128 4 waves, streaming across tiles, folded epilogue (N, K multiples of 128)", 256, 256, 256, 1.25f},
    {"thin tiles, 8 waves sharing K (N % 4 == 0, K % 128 == 0)", 64, 64, 512, 0.0f},
    {"256x128x128 4 waves (128x64 per wave), three stages, software-pipelined", 256, 128, 256, 0.0f},
    {"128x128x128 4 waves (64x64 per wave), three stages, software-pipelined", 128, 128, 256, 0.0f},
    {"128x192x128 4 waves (64x96 per wave), three stages, software-pipelined", 128, 192, 256, 0.0f},
};
constexpr int kPipeVariant = 5, kPipeOneTileVariant = 6, kStreamVariant = 7, kThinVariant = 8, kDeepWideVariant = 9, kDeepVariant = 10, kDeep192Variant = 11;
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
// Forced kernel variant of the calling host thread (-1: choose by shape).  Thread-local: a test or a tuning
// sweep that pins a variant cannot change the kernels another thread (e.g. the autograd worker) launches.
static thread_local int t_forced_variant = -1;
// Clock probe of the calling host thread (see odl_fp8_gemm_set_clock_probe): launch i of the streaming kernel writes
// record i % capacity.
static thread_local unsigned long long *t_clock_probe = nullptr;
static thread_local int t_clock_capacity = 0, t_clock_next = 0;

template <int FA, int FB>
static void launch_generic_fmt(const GemmArgs &g, hipStream_t stream) {
    hipLaunchKernelGGL((gemm_nt_generic_kernel<FA, FB>), dim3((unsigned)(g.tiles_m * g.tiles_n)), dim3(64), 0, stream, g);
}

static void launch_gemm_generic(int fa, int fb, const GemmArgs &g, hipStream_t stream) {
    if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E4M3) launch_generic_fmt<ODL_FP8_E4M3, ODL_FP8_E4M3>(g, stream);
    else if (fa == ODL_FP8_E5M2 && fb == ODL_FP8_E4M3) launch_generic_fmt<ODL_FP8_E5M2, ODL_FP8_E4M3>(g, stream);
    else if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E5M2) launch_generic_fmt<ODL_FP8_E4M3, ODL_FP8_E5M2>(g, stream);
    else launch_generic_fmt<ODL_FP8_E5M2, ODL_FP8_E5M2>(g, stream);
}

static int cu_count() { return device_cu_count(); }

// Whether the waves of a block sharing K (gemm_thin.hip) beat one 128 x 128 tile per compute unit.  The line in operand
// rows of the busiest unit lies between what was measured on both sides, thin against 128 x 128: 128 rows (32 x 14336 x
// 4096) 18.6 against 21.1 us, 96 rows (512 x 768 x 3072) 10.1 against 13.8, 48 rows (32 x 4096 x 14336) 19.2 against 53.4;
// 192 rows (768 x 768 x 2048) 13.1 against 10.3, (256 x 4096 x 4096) 22.1 against 17.5, though also (64 x 14336 x 4096) 23.9
// against 25.8.  K under 2048 (fewer than two steps per wave) is left to the tiled kernels: there is no chain to shorten
// (128 x 3072 x 768: 5.6 against 5.9).
static bool thin_ok(int64_t M, int64_t N) { return N % 4 == 0 && ((M + 127) / 128) * ((N + 127) / 128) <= cu_count(); }

static bool thin_pays(int64_t M, int64_t N, int64_t K) {
    const int cus = cu_count();
    return K >= 2048 && thin_ok(M, N) && gemm_thin_rows(M, N, cus) < 145;
}

// The kernel for an output of at most num_cus / 2 tiles of 256 x 256, which the big tiles would leave half the chip idle on
// (kManyTiles: the output has more).  At most one 128 x 128 tile per unit: from 16 K steps on the pipelined kernel of
// gemm_deep.hip; with fewer its longer way to the first MFMA (the second stage has to be there) costs more than its steps
// gain, and the four-stage form of the tiled kernel runs (1024 x 1024, warm and cold operands, deep / four stages: x 512 6.5 / 5.9 and
// 6.1 / 5.4 us, x 1024 7.6 / 7.6 and 7.5 / 7.2, x 1536 8.7 / 9.1 and 9.3 / 8.9, x 2048 9.7 / 10.7 and 10.4 / 10.7).  At most one of
// 128 x 192 and 8 K steps or more: those (against the better of the other two, cold operands: 8192 x 768 x 2048 19.1 -> 17.0 us, x 16384
// 104 -> 93.8; 3072 x 1536 x 4096 fp32 27.0 -> 23.8; 5120 x 1152 x 1024 13.2 -> 12.4; but 3072 x 1920 x 768 9.6 -> 9.8, 8192 x 768 x 512 8.4
// -> 8.7, where two blocks per unit hide each other's ends).  More: 256 x 128 tiles of the same kernel, one per unit, from 24 K steps on (2048 x 4096 x 8192 52.9 us against 60.5 with two 128 x 128
// blocks per unit, x 4096 30.3 against 32.4); with fewer steps the blocks that hide each other's fill and drain win (x 2048:
// 18.0 against 18.4, x 1024 11.6 against 12.7).
FewTiles gemm_few_tiles(int64_t M, int64_t N, int64_t K, int num_cus) { return gemm_few_tiles(TileCounts(M, N), K, num_cus); }

FewTiles gemm_few_tiles(const TileCounts &t, int64_t K, int num_cus) {
    if (t.t128 <= num_cus) return K >= 2048 ? kDeep : kTwoBlocks;
    if (t.t256 * 2 > num_cus) return kManyTiles;
    if (K >= 1024 && t.t192 <= num_cus) return kDeep192;
    return K >= 3072 && t.wide <= num_cus ? kDeepWide : kTwoBlocks;
}

// ... as a variant (kNoVariant: many tiles)
constexpr int kNoVariant = -1;
static int few_tiles_variant(int64_t M, int64_t N, int64_t K, bool lim32) {
    const FewTiles few = gemm_few_tiles(M, N, K, cu_count());
    if (few == kManyTiles) return kNoVariant;
    return few == kTwoBlocks || !lim32 ? 4 : few == kDeep ? kDeepVariant : few == kDeep192 ? kDeep192Variant : kDeepWideVariant;
}

static int choose_variant(int64_t M, int64_t N, int64_t K, bool stream_ok, bool lim32) {
    const int cus = cu_count();
    if (thin_pays(M, N, K)) return kThinVariant;
    if (const int small = few_tiles_variant(M, N, K, lim32); small != kNoVariant) return small;
    int best = 2;
    double best_score = -1.0;
    for (int v = 2; v <= kStreamVariant; ++v) {                       // variant 1 (one wave per SIMD) only by explicit request
        if (v == kStreamVariant && !stream_ok) continue;
        const Variant &cfg = kVariants[v];
        const int64_t tiles = ((M + cfg.bm - 1) / cfg.bm) * ((N + cfg.bn - 1) / cfg.bn);
        const int per_cu = cfg.bm * cfg.bn >= 256 * 256 ? 1 : (cfg.bm * cfg.bn >= 256 * 128 ? 1 : 2);
        const int64_t slots = (int64_t)cus * per_cu;
        const int64_t rounds = (tiles + slots - 1) / slots;
        const double useful = (double)M * N / ((double)rounds * slots * cfg.bm * cfg.bn);
        const double score = useful * cfg.eff;
        if (score > best_score) { best_score = score; best = v; }
    }
    return best;
}

// Rows of A that the streaming kernel should leave to a second launch (0: none).  Its 256 x 256 tiles go round the chip one
// per compute unit, and a last round of few tiles costs as much as a full one.  Those rows in the tiles of few_tiles_variant take
// about half a round with one 128 x 128 tile per unit, 0.6 with more, and 4 us for the launch.  With one tile that pays from 16 K steps on
// (5000 x 4096 x 2048: 47.8 -> 43.4 us, x 14336: 256 -> 216; 4096 x 4864 x 4096: 82.2 -> 68.8), with two from 32
// (11264 x 2048 x 4096: 91.5 -> 86.2, 50304 x 768 x 8192: 290 -> 261; 4016 x 5632 x 2048 would go from 49.1 to 53.7).
// Same K order, same bits.
static int64_t tail_rows(int64_t M, int64_t N, int64_t K) {
    const int cus = cu_count();
    const int64_t tiles_n = (N + 255) / 256, tiles = ((M + 255) / 256) * tiles_n;
    if (K < 2048 || tiles <= cus || tiles_n > cus || tiles % cus == 0) return 0;
    const int64_t rest = M - tiles / cus * cus / tiles_n * 256;
    const int64_t rest_tiles = ((rest + 127) / 128) * ((N + 127) / 128);
    return rest > 0 && rest_tiles <= (K >= 4096 ? 2 : 1) * (int64_t)cus ? rest : 0;
}

}  // namespace odl

using namespace odl;

extern "C" int odl_fp8_gemm_num_variants(void) { return kNumVariants; }

extern "C" const char *odl_fp8_gemm_variant_name(int variant) {
    return (variant >= 0 && variant < kNumVariants) ? kVariants[variant].name : "";
}

void odl::launch_splitk_reduce(const float *workspace, int splits, int64_t M, int64_t N, const float *sa, int sa_vec, const float *sb,
                               int sb_vec, const float *bias, void *c, int out_dtype, int accumulate, hipStream_t stream) {
    const int64_t quads = M * N / 4;
    int64_t blocks = (quads + 255) / 256;
    if (blocks > 4 * (int64_t)cu_count()) blocks = 4 * (int64_t)cu_count();
    if (out_dtype == ODL_BF16)
        hipLaunchKernelGGL((splitk_reduce_kernel<true>), dim3((unsigned)blocks), dim3(256), 0, stream, workspace, splits, M, N, sa, sa_vec, sb,
                           sb_vec, bias, c, accumulate);
    else
        hipLaunchKernelGGL((splitk_reduce_kernel<false>), dim3((unsigned)blocks), dim3(256), 0, stream, workspace, splits, M, N, sa, sa_vec, sb,
                           sb_vec, bias, c, accumulate);
}

void odl::attach_clock_probe(GemmArgs &g) {
    if (!t_clock_probe) return;
    g.clock_out = t_clock_probe + 4 * (size_t)(t_clock_next % t_clock_capacity);
    ++t_clock_next;
}

#ifndef ODL_FP8_NO_BENCH_HOOKS
extern "C" int odl_fp8_gemm_set_clock_probe(uint64_t *records_dev, int capacity) {
    if (records_dev && capacity < 1) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_set_clock_probe: capacity %d", capacity);
    t_clock_probe = reinterpret_cast<unsigned long long *>(records_dev);
    t_clock_capacity = records_dev ? capacity : 0;
    t_clock_next = 0;
    return ODL_OK;
}
#endif

extern "C" int odl_fp8_gemm_set_variant(int variant) {
    if (variant < -1 || variant >= kNumVariants) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_set_variant: %d out of range", variant);
    t_forced_variant = variant;
    return ODL_OK;
}

// Which kernel runs a product of checked arguments, and which one its last rows where they go to a second launch.
struct Route {
    int variant;
    int64_t tail;              // rows of the second launch (0: there is none)
    int tail_variant;
};

// launch_as: the variant to use (-1: the forced one, or the choice by shape)
static Route route_of(int64_t M, int64_t N, int64_t K, int out_dtype, int accumulate, int launch_as) {
    const bool tiled_ok = K >= 128 && K % 128 == 0 && (double)M * (double)K < 4294967296.0 && (double)N * (double)K < 4294967296.0;
    // the pipelined and the streaming kernel address rows with 32-bit byte offsets
    const bool lim32 = (double)(M + 256) * (double)K < 2147483648.0 && (double)(N + 256) * (double)K < 2147483648.0;
    // C = C + product is an epilogue of the kernels whose tiles end in a separate output phase; the streaming kernel
    // stores a tile under the next tile's MFMAs, where nothing can wait for the old values of C
    const bool stream_ok = tiled_ok && lim32 && N % 128 == 0 && K >= 512 && !accumulate;
    int variant = launch_as >= 0 ? launch_as : t_forced_variant >= 0 ? t_forced_variant : (tiled_ok ? choose_variant(M, N, K, stream_ok, lim32) : 0);
    if (variant != 0 && !tiled_ok) variant = 0;
    // the pipelined kernel walks K in pairs of 128-byte steps
    const bool pipe_ok = tiled_ok && K % 256 == 0 && lim32;
    if ((variant == kPipeVariant || variant == kPipeOneTileVariant) && !pipe_ok) variant = 2;

    if (variant == kThinVariant && !thin_ok(M, N)) variant = 4;
    if (variant >= kDeepWideVariant && !lim32) variant = 4;

    if (variant == kStreamVariant && t_forced_variant < 0 && launch_as < 0) {
        // Counted in 256 x 256 tiles those rows can be too many for the kernels of few tiles (half tiles at an edge count
        // whole there): two 128 x 128 blocks per unit then (4224 x 5632 x 4096,
        // rest 1408 rows: 84 us in all).
        const int64_t rest = tail_rows(M, N, K);
        const int small = rest > 0 ? few_tiles_variant(rest, N, K, lim32) : kNoVariant;
        if (rest > 0) return {kStreamVariant, rest, small != kNoVariant ? small : 4};
    }

    GemmArgs g = {};
    g.M = M; g.N = N; g.K = K;
    g.out_dtype = out_dtype;
    g.accumulate = accumulate != 0;
    // the streaming kernel wants N in multiples of 128: next best kernel instead
    if (variant == kStreamVariant && !(stream_ok && gemm_stream_accepts(g))) variant = pipe_ok ? kPipeVariant : 2;
    return {variant, 0, 0};
}

// The launch of checked arguments.
static int gemm_nt_checked(const uint8_t *a, const uint8_t *b, int64_t M, int64_t N, int64_t K, int fmt_a, int fmt_b, const float *sa_inv, int64_t sa_n,
                           const float *sb_inv, int64_t sb_n, const void *bias, void *c, int out_dtype, int accumulate, int launch_as,
                           bool fresh, hipStream_t stream) {
    const Route route = route_of(M, N, K, out_dtype, accumulate, launch_as);
    const int variant = route.variant;
    if (route.tail > 0) {
        const int64_t head = M - route.tail, esz = out_dtype == ODL_BF16 ? 2 : 4;
        const int rc = gemm_nt_checked(a, b, head, N, K, fmt_a, fmt_b, sa_inv, sa_n == 1 ? 1 : head, sb_inv, sb_n, bias, c, out_dtype, accumulate,
                                       kStreamVariant, fresh, stream);
        if (rc != ODL_OK) return rc;
        return gemm_nt_checked(a + head * K, b, route.tail, N, K, fmt_a, fmt_b, sa_n == 1 ? sa_inv : sa_inv + head, sa_n == 1 ? 1 : route.tail, sb_inv,
                               sb_n, bias, reinterpret_cast<uint8_t *>(c) + head * N * esz, out_dtype, accumulate, route.tail_variant,
                               fresh, stream);
    }

    GemmArgs g;
    g.a = a; g.b = b; g.c = c; g.sa = sa_inv; g.sb = sb_inv; g.bias = bias;
    g.M = M; g.N = N; g.K = K;
    g.sa_vec = sa_n == M && M != 1;
    g.sb_vec = sb_n == N && N != 1;
    g.out_dtype = out_dtype;
    g.accumulate = accumulate != 0;
    g.fresh = fresh;
    const int bm = variant == 0 ? 32 : kVariants[variant].bm, bn = variant == 0 ? 32 : kVariants[variant].bn;
    const int64_t tm = (M + bm - 1) / bm, tn = (N + bn - 1) / bn;
    if (tm * tn > 0x7ffffff0LL) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt: too many tiles");
    g.tiles_m = (int)tm; g.tiles_n = (int)tn;

    if (variant == 0) launch_gemm_generic(fmt_a, fmt_b, g, stream);
    else if (variant == kThinVariant) launch_gemm_thin(fmt_a, fmt_b, g, cu_count(), stream);
    else if (variant >= kDeepWideVariant) launch_gemm_deep(bm, bn, fmt_a, fmt_b, g, cu_count(), stream);
    else if (variant == kPipeVariant) launch_gemm_pipe(fmt_a, fmt_b, g, cu_count(), stream);
    else if (variant == kPipeOneTileVariant) launch_gemm_pipe(fmt_a, fmt_b, g, 1 << 30, stream);
    else if (variant == kStreamVariant) { attach_clock_probe(g); launch_gemm_stream(fmt_a, fmt_b, g, cu_count(), stream); }
    else launch_gemm_tiled(variant, fmt_a, fmt_b, g, stream);
    return check_launch("odl_fp8_gemm_nt");
}

extern "C" int odl_fp8_gemm_route(int64_t M, int64_t N, int64_t K, int out_dtype, int accumulate, int64_t *tail_rows_out, int *tail_variant_out) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 16 != 0 || (out_dtype != ODL_BF16 && out_dtype != ODL_F32) || !tail_rows_out || !tail_variant_out) {
        set_error(ODL_ERR_ARG, "odl_fp8_gemm_route: %lld x %lld x %lld, out_dtype %d", (long long)M, (long long)N, (long long)K, out_dtype);
        return -1;
    }
    const Route route = route_of(M, N, K, out_dtype, accumulate, -1);
    *tail_rows_out = route.tail;
    *tail_variant_out = route.tail_variant;
    return route.variant;
}

extern "C" int odl_fp8_gemm_nt_hinted(const uint8_t *a, const uint8_t *b, int64_t M, int64_t N, int64_t K, int fmt_a, int fmt_b,
                                      const float *sa_inv, int64_t sa_n, const float *sb_inv, int64_t sb_n, const void *bias,
                                      int bias_dtype, void *c, int out_dtype, int accumulate, int fresh, odl_stream_t stream_) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (!a || !b || !c || !sa_inv || !sb_inv) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: null pointer");
    if (M < 0 || N < 0 || K < 0) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: negative size");
    if ((fmt_a != ODL_FP8_E4M3 && fmt_a != ODL_FP8_E5M2) || (fmt_b != ODL_FP8_E4M3 && fmt_b != ODL_FP8_E5M2))
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: formats %d, %d", fmt_a, fmt_b);
    if (sa_n != 1 && sa_n != M) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: sa_n=%lld is neither 1 nor M", (long long)sa_n);
    if (sb_n != 1 && sb_n != N) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: sb_n=%lld is neither 1 nor N", (long long)sb_n);
    if (out_dtype != ODL_BF16 && out_dtype != ODL_F32) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: out_dtype %d", out_dtype);
    if (bias && bias_dtype != ODL_F32) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt: bias must be fp32 (bias_dtype %d)", bias_dtype);
    if (K % 16 != 0) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt: K=%lld must be a multiple of 16", (long long)K);
    if ((reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15))
        return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt: operands must be 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(c) & 15) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt: output must be 16-byte aligned");
    if ((sa_n > 1 && (reinterpret_cast<uintptr_t>(sa_inv) & 15)) || (sb_n > 1 && (reinterpret_cast<uintptr_t>(sb_inv) & 15)) ||
        (bias && (reinterpret_cast<uintptr_t>(bias) & 15)))
        return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt: scale vectors and bias must be 16-byte aligned");
    if (M == 0 || N == 0) return ODL_OK;
    return gemm_nt_checked(a, b, M, N, K, fmt_a, fmt_b, sa_inv, sa_n, sb_inv, sb_n, bias, c, out_dtype, accumulate, -1, fresh != 0, stream);
}

extern "C" int odl_fp8_gemm_nt(const uint8_t *a, const uint8_t *b, int64_t M, int64_t N, int64_t K, int fmt_a, int fmt_b,
                               const float *sa_inv, int64_t sa_n, const float *sb_inv, int64_t sb_n, const void *bias,
                               int bias_dtype, void *c, int out_dtype, int accumulate, odl_stream_t stream_) {
    return odl_fp8_gemm_nt_hinted(a, b, M, N, K, fmt_a, fmt_b, sa_inv, sa_n, sb_inv, sb_n, bias, bias_dtype, c, out_dtype, accumulate, 0, stream_);
}

extern "C" int odl_fp8_gemm_nt_sum(int pairs, const uint8_t *const *a, const uint8_t *const *b, const int64_t *K, int64_t M, int64_t N,
                                   int fmt_a, int fmt_b, const float *const *sa_inv, const float *const *sb_inv, void *c,
                                   int out_dtype, odl_stream_t stream_) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (pairs < 1 || pairs > 64) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_sum: %d operand pairs (1 .. 64)", pairs);
    if (!a || !b || !K || !sa_inv || !sb_inv || !c) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_sum: null pointer");
    if (M < 0 || N < 0) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_sum: negative size");
    if ((fmt_a != ODL_FP8_E4M3 && fmt_a != ODL_FP8_E5M2) || (fmt_b != ODL_FP8_E4M3 && fmt_b != ODL_FP8_E5M2))
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_sum: formats %d, %d", fmt_a, fmt_b);
    if (out_dtype != ODL_BF16 && out_dtype != ODL_F32) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_sum: out_dtype %d", out_dtype);
    for (int s = 0; s < pairs; ++s) {
        if (!a[s] || !b[s] || !sa_inv[s] || !sb_inv[s]) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_sum: null pointer in pair %d", s);
        if (K[s] <= 0 || K[s] % 16 != 0)
            return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt_sum: K[%d]=%lld must be a positive multiple of 16", s, (long long)K[s]);
        if ((reinterpret_cast<uintptr_t>(a[s]) & 15) || (reinterpret_cast<uintptr_t>(b[s]) & 15))
            return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt_sum: operands must be 16-byte aligned (pair %d)", s);
    }
    if (reinterpret_cast<uintptr_t>(c) & 15) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt_sum: output must be 16-byte aligned");
    if (M == 0 || N == 0) return ODL_OK;

    // one launch of the streaming kernel when every pair suits it ...
    if (pairs <= 4 && (t_forced_variant < 0 || t_forced_variant == kStreamVariant)) {
        GemmArgs g;
        GemmPairs gp;
        g.a = a[0]; g.b = b[0]; g.c = c; g.sa = sa_inv[0]; g.sb = sb_inv[0]; g.bias = nullptr;
        g.M = M; g.N = N; g.K = K[0];
        g.sa_vec = 0; g.sb_vec = 0;
        g.out_dtype = out_dtype;
        g.tiles_m = (int)((M + 255) / 256); g.tiles_n = (int)((N + 255) / 256);
        gp.count = pairs;
        bool fits = true;
        for (int s = 0; s < pairs; ++s) {
            fits = fits && K[s] < 2147483648LL;
            gp.k[s] = (int)K[s]; gp.a[s] = a[s]; gp.b[s] = b[s]; gp.sa[s] = sa_inv[s]; gp.sb[s] = sb_inv[s];
        }
        if (fits && (pairs > 1 || t_forced_variant == kStreamVariant) && gemm_stream_accepts_pairs(g, gp)) {
            launch_gemm_stream_pairs(fmt_a, fmt_b, g, gp, cu_count(), stream);
            return check_launch("odl_fp8_gemm_nt_sum");
        }
    }
    // ... otherwise a GEMM per pair, the second and later ones adding into C (one rounding to the output type per pair)
    for (int s = 0; s < pairs; ++s) {
        const int rc = odl_fp8_gemm_nt(a[s], b[s], M, N, K[s], fmt_a, fmt_b, sa_inv[s], 1, sb_inv[s], 1, nullptr, ODL_F32, c, out_dtype,
                                       s > 0, stream_);
        if (rc != ODL_OK) return rc;
    }
    return ODL_OK;
}

// the launch of odl_fp8_gemm_layouts and odl_fp8_gemm_wgrad; `who` names the entry, `partial`: A need not be whole tiles
static int gemm_as_stored(const char *who, const uint8_t *a, const uint8_t *b, int64_t M, int64_t N, int64_t K, int fmt_a, int fmt_b, int layout_a,
                          int layout_b, const float *sa_inv, const float *sb_inv, void *c, int out_dtype, bool partial, hipStream_t stream) {
    if (!a || !b || !c || !sa_inv || !sb_inv) return set_error(ODL_ERR_ARG, "%s: null pointer", who);
    if ((fmt_a != ODL_FP8_E4M3 && fmt_a != ODL_FP8_E5M2) || (fmt_b != ODL_FP8_E4M3 && fmt_b != ODL_FP8_E5M2))
        return set_error(ODL_ERR_ARG, "%s: formats %d, %d", who, fmt_a, fmt_b);
    if ((layout_a != ODL_K_FAST && layout_a != ODL_K_SLOW) || (layout_b != ODL_K_FAST && layout_b != ODL_K_SLOW))
        return set_error(ODL_ERR_ARG, "%s: layouts %d, %d", who, layout_a, layout_b);
    if (out_dtype != ODL_BF16 && out_dtype != ODL_F32) return set_error(ODL_ERR_ARG, "%s: out_dtype %d", who, out_dtype);
    if ((reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15) || (reinterpret_cast<uintptr_t>(c) & 15))
        return set_error(ODL_ERR_SHAPE, "%s: operands and output must be 16-byte aligned", who);
    GemmArgs g;
    g.a = a; g.b = b; g.c = c; g.sa = sa_inv; g.sb = sb_inv; g.bias = nullptr;
    g.M = M; g.N = N; g.K = K;
    g.sa_vec = 0; g.sb_vec = 0;
    g.out_dtype = out_dtype;
    g.ta = layout_a == ODL_K_SLOW;
    g.tb = layout_b == ODL_K_SLOW;
    const int mult_m = partial ? 16 : 256, mult_n = partial ? 128 : 256;
    const bool sizes_ok = M >= (partial ? 256 : 1) && N > 0 && K >= 512 && M % mult_m == 0 && N % mult_n == 0 && K % 128 == 0 &&
                          (double)(M + 256) * (double)K < 2147483648.0 && (double)(N + 256) * (double)K < 2147483648.0;
    if (!sizes_ok)
        return set_error(ODL_ERR_SHAPE, "%s: M, N must be multiples of %s, K of 128 (K >= 512) and each operand under 2 GiB; got %lld x %lld x %lld",
                         who, partial ? "16 (256 at least) and 128" : "256", (long long)M, (long long)N, (long long)K);
    g.tiles_m = (int)((M + 255) / 256); g.tiles_n = (int)((N + 255) / 256);
    if (!gemm_stream_accepts(g)) return set_error(ODL_ERR_SHAPE, "%s: shape not taken by the streaming kernel", who);
    attach_clock_probe(g);
    launch_gemm_stream(fmt_a, fmt_b, g, cu_count(), stream);
    return check_launch(who);
}

extern "C" int odl_fp8_gemm_layouts(const uint8_t *a, const uint8_t *b, int64_t M, int64_t N, int64_t K, int fmt_a, int fmt_b,
                                    int layout_a, int layout_b, const float *sa_inv, const float *sb_inv, void *c,
                                    int out_dtype, odl_stream_t stream_) {
    return gemm_as_stored("odl_fp8_gemm_layouts", a, b, M, N, K, fmt_a, fmt_b, layout_a, layout_b, sa_inv, sb_inv, c, out_dtype, false,
                          reinterpret_cast<hipStream_t>(stream_));
}

extern "C" int odl_fp8_gemm_wgrad(const uint8_t *gy, const uint8_t *x_t, int64_t n_out, int64_t n_in, int64_t tokens, int fmt_g, int fmt_x,
                                  const float *sg_inv, const float *sx_inv, void *dw, int out_dtype, odl_stream_t stream_) {
    return gemm_as_stored("odl_fp8_gemm_wgrad", gy, x_t, n_out, n_in, tokens, fmt_g, fmt_x, ODL_K_SLOW, ODL_K_FAST, sg_inv, sx_inv, dw, out_dtype, true,
                          reinterpret_cast<hipStream_t>(stream_));
}

// How many runs to cut K into for an output of few tiles (1 = do not split).  A model in microseconds, fitted to
// measurements on this GPU (outputs 768 x 768 .. 8192 x 1024, K = 8192 .. 151936):
//   one launch, 256 x 256 tiles : 0.92 us per K step of 128 (few compute units busy: high clock) + 3 steps of overhead
//   one launch, smaller tiles   : what odl_fp8_gemm_nt takes for outputs of <= cus / 2 big tiles (few_tiles_variant).
//                                 128 x 128 with a unit each 0.37 us per step + 6 us (3072 x 768 x 16384: 45 - 50 us, in
//                                 six runs 52 and the reduction's launch); 256 x 128 with a unit each 0.70 + 7 (128 x 192 in
//                                 their place: 0.66 + 8; where two runs are proposed instead, odl_fp8_gemm_runs looks
//                                 again); two 128 x 128 blocks per unit 0.62 (it reads every operand panel twice as often)
//   split                       : 0.96 us per step of a run + 9 us (pipeline fill, the fp32 epilogue, the second launch)
//                                 + the partial results, splits x M x N floats written and read back, at 2.7 TB/s in all
//   with operands that outgrow the 256 MB memory-side cache, per step 0.61 (128 x 128: 8192 x 512 x 50304 241 us, in three runs
//                                 234, in four 200), 0.88 (256 x 128: 8192 x 1024 x 151936 1047, in two runs 961), 1.45 (split)
//   each bounded below by its operand traffic (tiles x panel bytes) at about 12 TB/s out of the caches (the kernels of
//   gemm_deep.hip: 18).
//   one launch, thin tiles      : 4 us + 2.7 ns per K step and operand row of the busiest compute unit (how well that
//                                 fits: gemm_thin.hip)
// The runs of a split must fit the compute units at once, and a split must win by 10 %.
// The order of addition is no part of the price: on this hardware the error of a product is that of one MFMA, which aligns its 64
// products before it adds them, however many of them follow each other (fp32 results of random codes E5M2 x E4M3 against 64 bits,
// relative root mean square: 3072 x 768 x 16384 in one chain 1.07889e-5, in six runs 1.07889e-5; 8192 x 768 x 50304 1.08035e-5, in two
// 1.08034e-5; summing in runs inside the one launch was built, gave the same errors, and cost 57.8 -> 63.2 us).
// k_slow: an operand is stored with the contraction index slow (odl_fp8_gemm_layouts), which only the streaming
// kernel reads: the 128 x 128 kernel is then not an alternative.
extern "C" int odl_fp8_gemm_split_count(int64_t M, int64_t N, int64_t K, int k_slow) {
    if (M <= 0 || N <= 0 || M % 128 || N % 128 || K % 128 || K < 2048) return 1;
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
    const int cus = cu_count();
    const int64_t steps = K / 128;
    const bool cold = (double)(M + N) * (double)K > 268435456.0;
    int64_t most = cus / tiles;
    if (most > 16) most = 16;
    const double traffic_us = (double)tiles * 512.0 * (double)K / 12.0e6;
    double whole = 0.92 * ((double)steps + 3.0);
    if (whole < traffic_us) whole = traffic_us;
    if (!k_slow) {
        const int variant = few_tiles_variant(M, N, K, (double)(M + 256) * (double)K < 2147483648.0 && (double)(N + 256) * (double)K < 2147483648.0);
        const double panels = (double)((M + 127) / 128) * (double)((N + 127) / 128) * (double)K;         // of 128 rows, once per tile
        double small = whole, small_traffic_us = 0.0;
        if (variant == kDeepVariant) { small = (cold ? 0.61 : 0.37) * (double)steps + 6.0; small_traffic_us = panels * 256.0 / 18.0e6; }
        else if (variant == kDeepWideVariant || variant == kDeep192Variant) { small = (cold ? 0.88 : 0.70) * (double)steps + 7.0; small_traffic_us = panels * 192.0 / 18.0e6; }
        else if (variant != kNoVariant) { small = 0.62 * ((double)steps + 3.0); small_traffic_us = panels * 256.0 / 12.0e6; }
        if (small < small_traffic_us) small = small_traffic_us;
        if (small < whole) whole = small;
    }
    if (!k_slow && thin_pays(M, N, K)) {
        const double thin = 4.0 + 0.0027 * (double)gemm_thin_rows(M, N, cus) * (double)steps;
        if (thin < whole) whole = thin;
    }
    double best = whole;
    int best_splits = 1;
    for (int64_t splits = 2; splits <= most; ++splits) {
        const int64_t per = ((steps + splits - 1) / splits + 1) & ~(int64_t)1;
        const int64_t last = steps - (splits - 1) * per;
        if (per < 8 || last < 4) continue;
        double run = (cold ? 1.45 : 0.96) * (double)per + 9.0;
        if (run < traffic_us) run = traffic_us;
        const double cost = run + (double)splits * (double)M * (double)N * 4.0 / 2.7e6;
        if (cost < 0.90 * whole && cost < best) { best = cost; best_splits = (int)splits; }
    }
    return best_splits;
}

// One launch of 128 x 192 tiles that gives (nearly) every compute unit one beats two runs of big tiles and the addition behind
// them: 8192 x 768 x 50304 319 -> 283 us, 16384 x 384 x 50304 340 -> 308; with block scales 337 -> 308 and 359 -> 328.  Not three runs
// (3072 x 1536 x 50304 229 against 231, with block scales 236 against 256).
extern "C" int odl_fp8_gemm_runs(int64_t M, int64_t N, int64_t K, int k_slow) {
    const int runs = odl_fp8_gemm_split_count(M, N, K, k_slow);
    return runs == 2 && !k_slow && gemm_few_tiles(M, N, K, cu_count()) == kDeep192 ? 1 : runs;
}

extern "C" int odl_fp8_gemm_splitk(const uint8_t *a, const uint8_t *b, int64_t M, int64_t N, int64_t K, int fmt_a, int fmt_b,
                                   int layout_a, int layout_b, const float *sa_inv, int64_t sa_n, const float *sb_inv,
                                   int64_t sb_n, const float *bias, void *c, int out_dtype, int accumulate, int splits, void *workspace,
                                   int64_t workspace_bytes, odl_stream_t stream_) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (!a || !b || !c || !sa_inv || !sb_inv || !workspace) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: null pointer");
    if ((fmt_a != ODL_FP8_E4M3 && fmt_a != ODL_FP8_E5M2) || (fmt_b != ODL_FP8_E4M3 && fmt_b != ODL_FP8_E5M2))
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: formats %d, %d", fmt_a, fmt_b);
    if ((layout_a != ODL_K_FAST && layout_a != ODL_K_SLOW) || (layout_b != ODL_K_FAST && layout_b != ODL_K_SLOW))
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: layouts %d, %d", layout_a, layout_b);
    if (out_dtype != ODL_BF16 && out_dtype != ODL_F32) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: out_dtype %d", out_dtype);
    if (sa_n != 1 && sa_n != M) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: sa_n=%lld is neither 1 nor M", (long long)sa_n);
    if (sb_n != 1 && sb_n != N) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: sb_n=%lld is neither 1 nor N", (long long)sb_n);
    if ((reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15) || (reinterpret_cast<uintptr_t>(c) & 15) ||
        (reinterpret_cast<uintptr_t>(workspace) & 15))
        return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_splitk: operands, output and workspace must be 16-byte aligned");
    const int ta = layout_a == ODL_K_SLOW, tb = layout_b == ODL_K_SLOW;
    const bool sizes_ok = M > 0 && N > 0 && M % (ta ? 256 : 128) == 0 && N % (tb ? 256 : 128) == 0 && K % 128 == 0 &&
                          (double)(M + 256) * (double)K < 2147483648.0 && (double)(N + 256) * (double)K < 2147483648.0;
    if (!sizes_ok)
        return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_splitk: M, N, K must be multiples of 128 (256 for an operand stored K-slow) and each operand under 2 GiB; got %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
    const int64_t steps = K / 128;
    const int64_t per = ((steps + splits - 1) / (splits > 0 ? splits : 1) + 1) & ~(int64_t)1;
    // what the kernel needs to be correct: every run at least four K steps (its load pipeline is two steps deep and runs
    // in pairs).  odl_fp8_gemm_split_count proposes only runs of eight steps and more, which is where a split pays.
    // one "run" is allowed with accumulate: the way to add a product with an operand stored K-slow into C
    if (splits < (accumulate ? 1 : 2) || splits > 64 || per < 4 || steps - (splits - 1) * per < 4)
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: %d splits of K=%lld leave a run shorter than 512 (or fewer than 2 splits without accumulate)", splits, (long long)K);
    if (workspace_bytes < (int64_t)splits * M * N * 4)
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_splitk: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
                         (long long)splits * M * N * 4);
    GemmArgs g;
    g.a = a; g.b = b; g.c = workspace; g.sa = sa_inv; g.sb = sb_inv; g.bias = nullptr;
    g.M = M; g.N = N; g.K = K;
    g.sa_vec = 0; g.sb_vec = 0;
    g.out_dtype = ODL_F32;
    g.ta = ta; g.tb = tb;
    g.splits = splits; g.split_steps = (int)per;
    g.tiles_m = (int)((M + 255) / 256); g.tiles_n = (int)((N + 255) / 256);
    if (!gemm_stream_accepts(g)) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_splitk: shape not taken by the streaming kernel");
    attach_clock_probe(g);
    launch_gemm_stream(fmt_a, fmt_b, g, cu_count(), stream);
    const int sa_vec = sa_n == M && M != 1, sb_vec = sb_n == N && N != 1;
    if (splits == 1) {
        // a single run is an ordinary launch: the kernel applies the tensor scales itself, the second kernel adds C
        const float *one = unit_scale_for_current_device("odl_fp8_gemm_splitk");
        if (!one) return ODL_ERR_LAUNCH;
        launch_splitk_reduce((const float *)workspace, 1, M, N, one, 0, one, 0, bias, c, out_dtype, accumulate != 0, stream);
        return check_launch("odl_fp8_gemm_splitk");
    }
    launch_splitk_reduce((const float *)workspace, splits, M, N, sa_inv, sa_vec, sb_inv, sb_vec, bias, c, out_dtype, accumulate != 0, stream);
    return check_launch("odl_fp8_gemm_splitk");
}

// ------------------------------------------------------- several products in one launch
// What launches cost, in microseconds: of `variant` over t tiles of its size in all, K in steps of 128.  Fitted to products of 256
// to 14336 rows and columns, K = 768 .. 8192, within 15 % where it decides; the fill of a launch and its last stores are the
// constants.  A last round of 256 x 256 tiles that leaves units idle runs faster than a full one (power, caches): 0.55 of
// one and up.
static double launch_us(int variant, const TileCounts &t, int64_t steps, int cus) {
    const double k = (double)steps;
    if (variant == kStreamVariant) {
        const double rest = (double)(t.t256 % cus) / cus;
        return ((double)(t.t256 / cus) + (rest > 0.0 ? 0.55 + 0.45 * rest : 0.0)) * k * 1.4 + 8.0;
    }
    if (variant == kDeepVariant) return 0.40 * k + 6.0;
    if (variant == kDeep192Variant) return 0.72 * k + 7.0;
    if (variant == kDeepWideVariant) return 0.80 * k + 7.0;
    return t.t128 <= cus ? 0.30 * k + 5.5 : (double)((t.t128 + 2 * cus - 1) / (2 * cus)) * 0.62 * (k + 3.0) + 4.0;
}

static int variant_of(FewTiles few) {
    return few == kManyTiles ? kStreamVariant : few == kTwoBlocks ? 4 : few == kDeep ? kDeepVariant : few == kDeep192 ? kDeep192Variant : kDeepWideVariant;
}

// The kernel that computes several products of one contraction length in one launch, or kNoVariant: one by one.
//
// Products that a Linear's siblings need side by side (q / k / v, gate / up, and their weight gradients) each leave a last round of
// tiles part empty, or are too small to fill the chip at all, and each pays a launch's fill and drain.  Together they are one
// launch of gemm_few_tiles's kernel for all their tiles.  Same K order as alone, so the same bits (fp32 sums of products
// that alone take the thin kernel, few rows of a long K, add in this kernel's order instead, to the same error).  us one by one / in one launch:
//   8192 x (4096, 1024, 1024) x 4096 160.7 / 146.9   2048 x (4096, 1024, 1024) x 4096 64.4 / 44.3   256 x the same 32.1 / 15.7
//   4016 x (5632, 5632) x 2048 93.2 / 76.9           8192 x (3072, 3072) x 1024 59.8 / 49.9        1024 x the same 14.4 / 11.0
//   (3072, 3072) x 1024 x 8192 fp32 61.8 / 51.4      (5632, 5632) x 2048 x 4096 fp32 91.3 / 89.9   (14336 x 2) x 4096 x 4096 395 / 369
//   8192 x (14336, 14336) x 4096 696 / 707: whole rounds either way, and the launches of their own are a little faster
// so the model above has to promise 3 %.  K from 768 on, which is where it was measured.
static int group_variant(int count, const int64_t *M, const int64_t *N, int64_t K, int out_dtype) {
    if (count < 2 || count > 4 || K < 128 || K % 128 != 0) return kNoVariant;
    const int cus = cu_count();
    bool stream_ok = K >= 512;
    TileCounts all;
    double apart = 0.0;
    for (int s = 0; s < count; ++s) {
        if (M[s] <= 0 || N[s] <= 0 || (double)(M[s] + 256) * (double)K >= 2147483648.0 || (double)(N[s] + 256) * (double)K >= 2147483648.0) return kNoVariant;
        GemmArgs g = {};
        g.M = M[s]; g.N = N[s]; g.K = K;
        g.out_dtype = out_dtype;
        stream_ok = stream_ok && gemm_stream_accepts_group(g);
        const TileCounts own(M[s], N[s]);
        all.t128 += own.t128; all.t192 += own.t192; all.wide += own.wide; all.t256 += own.t256;
        if (t_forced_variant >= 0) continue;
        if (K < 768 || odl_fp8_gemm_runs(M[s], N[s], K, 0) > 1) return kNoVariant;         // (K in runs: a workspace, which the caller brings)
        const Route route = route_of(M[s], N[s], K, out_dtype, 0, -1);
        apart += route.variant == kThinVariant ? 4.0 + 0.0027 * gemm_thin_rows(M[s], N[s], cus) * (double)(K / 128)
                 : route.tail > 0 ? launch_us(kStreamVariant, TileCounts(M[s] - route.tail, N[s]), K / 128, cus) +
                                        launch_us(route.tail_variant, TileCounts(route.tail, N[s]), K / 128, cus)
                                  : launch_us(route.variant, own, K / 128, cus);
    }
    if (all.t128 > 0x7ffffff0LL) return kNoVariant;
    const int variant = t_forced_variant >= 0 ? t_forced_variant : variant_of(gemm_few_tiles(all, K, cus));
    if (variant == kStreamVariant ? !stream_ok : variant != 4 && variant < kDeepWideVariant) return kNoVariant;
    return t_forced_variant >= 0 || launch_us(variant, all, K / 128, cus) < 0.97 * apart ? variant : kNoVariant;
}

extern "C" int odl_fp8_gemm_group_route(int count, const int64_t *M, const int64_t *N, int64_t K, int out_dtype) {
    if (!M || !N || (out_dtype != ODL_BF16 && out_dtype != ODL_F32)) {
        set_error(ODL_ERR_ARG, "odl_fp8_gemm_group_route: null pointer, or out_dtype %d", out_dtype);
        return -1;
    }
    return group_variant(count, M, N, K, out_dtype);
}

extern "C" int odl_fp8_gemm_nt_group(int count, const uint8_t *const *a, const uint8_t *const *b, const int64_t *M, const int64_t *N, int64_t K,
                                     int fmt_a, int fmt_b, const float *const *sa_inv, const float *const *sb_inv, void *const *c, int out_dtype,
                                     int fresh, odl_stream_t stream_) {
    if (count < 1 || !a || !b || !M || !N || !sa_inv || !sb_inv || !c) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_group: null pointer, or %d products", count);
    const int variant = group_variant(count, M, N, K, out_dtype);
    // (E4M3 times E5M2 is no product of a Linear: its kernels are not built)
    bool one = variant != kNoVariant && (out_dtype == ODL_BF16 || out_dtype == ODL_F32) &&
               (fmt_b == ODL_FP8_E4M3 ? fmt_a == ODL_FP8_E4M3 || fmt_a == ODL_FP8_E5M2 : fmt_b == ODL_FP8_E5M2 && fmt_a == ODL_FP8_E5M2);
    for (int s = 0; one && s < count; ++s) {
        one = a[s] && b[s] && sa_inv[s] && sb_inv[s] && c[s];
        for (const void *p : {(const void *)a[s], (const void *)b[s], (const void *)c[s]}) one = one && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
    }
    if (!one) {                    // one by one, with the checks of that entry
        for (int s = 0; s < count; ++s) {
            const int rc = odl_fp8_gemm_nt_hinted(a[s], b[s], M[s], N[s], K, fmt_a, fmt_b, sa_inv[s], 1, sb_inv[s], 1, nullptr, ODL_F32, c[s], out_dtype,
                                                  0, fresh, stream_);
            if (rc != ODL_OK) return rc;
        }
        return ODL_OK;
    }
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    const int bm = kVariants[variant].bm, bn = kVariants[variant].bn;
    GemmGroup gg;
    gg.count = count;
    for (int s = 0; s < count; ++s) {
        GemmArgs &g = gg.m[s];
        g.a = a[s]; g.b = b[s]; g.c = c[s]; g.sa = sa_inv[s]; g.sb = sb_inv[s]; g.bias = nullptr;
        g.M = M[s]; g.N = N[s]; g.K = K;
        g.sa_vec = g.sb_vec = 0;
        g.out_dtype = out_dtype;
        g.fresh = fresh != 0;
        const int64_t tm = (M[s] + bm - 1) / bm, tn = (N[s] + bn - 1) / bn;
        g.tiles_m = (int)tm; g.tiles_n = (int)tn;
        gg.first[s] = gg.total;
        gg.total += (int)(tm * tn);
    }
    if (variant == kStreamVariant) launch_gemm_stream_group(fmt_a, fmt_b, gg, cu_count(), stream);
    else if (variant == 4) launch_gemm_tiled_group(fmt_a, fmt_b, gg, stream);
    else launch_gemm_deep_group(bm, bn, fmt_a, fmt_b, gg, cu_count(), stream);
    return check_launch("odl_fp8_gemm_nt_group");
}

// ------------------------------------------------------- products that are added up in one launch
// What a launch costs that adds its product to C in bf16.  C is read once more, in an output phase that nothing overlaps but other
// blocks: charged with 1 us and 0.4 us a MB in the kernels of 128 rows and 256 x 128 tiles (accumulating less plain, C of 16 to 67 MB, two
// 128 x 128 blocks a unit 0.2 - 0.5 us a MB, the deep kernels 0.25 - 0.6 and up to 1 at 8192 x 4096 x 3072; under 10 MB 1 - 6 us in all).  The
// 256 x 256 kernels that have such a phase take 1.5 us a step with cold operands, and 0.8 us a MB.
static double accumulate_us(int variant, const TileCounts &t, int64_t steps, double c_mb, int cus) {
    if (variant == 4 || variant >= kDeepWideVariant) return launch_us(variant, t, steps, cus) + 1.0 + 0.4 * c_mb;
    return (double)((t.t256 + cus - 1) / cus) * (double)steps * 1.5 + 8.0 + 0.8 * c_mb;
}

// The kernel for C = sum of products [M, K_s] . [N, K_s]^T in bf16, or kNoVariant: a launch each.
//
// gemm_deep.h keeps the sum so far in registers and rounds it behind each product, as launches that accumulate do, so the bits are
// theirs (but where one alone takes the thin kernel: see group_variant); us a launch each / together:
//   8192 x 1024 x (3072, 3072) 65.8 / 53.7    4016 x 2048 x (5632, 5632) 98.8 / 86.6    1024 x 1024 x (1024, 512, 512) 20.0 / 14.2
//   5744 x 4096 x (4096, 1024, 1024) 198 / 136 (three rounds of 256 x 128 tiles against the 256 x 256 kernels that accumulate)
//   8192 x 4096 x (14336, 14336) 718 / 804, 256 x 4096 x (14336, 14336) (thin tiles) 64 / 83: launches of their own
// The model: 0.85 us a step of 256 x 128 tiles (operands from memory, the chip full), a last round that leaves units idle faster.
// Where the streaming kernel takes the sum with one rounding (odl_fp8_gemm_nt_sum) callers ask it first.
//
// Block scales have no such launch: their results are rounded one by one and added in bf16, and the streaming kernel, which could
// take them as one contraction (8192 x 2048 x (5632, 5632) 133 us against 172), would round once, other results by 2.9e-3.
static int chain_variant(int pairs, const int64_t *K, int64_t M, int64_t N) {
    if (pairs < 2 || pairs > 4 || M < 32 || N < 128 || N % 128 != 0) return kNoVariant;
    const int cus = cu_count();
    const TileCounts t(M, N);
    const double c_mb = (double)M * (double)N * 2e-6;
    int64_t total = 0;
    double apart = 0.0;
    for (int s = 0; s < pairs; ++s) {
        if (K[s] < 512 || K[s] % 256 != 0 || (double)(M + 256) * (double)K[s] >= 2147483648.0 || (double)(N + 256) * (double)K[s] >= 2147483648.0)
            return kNoVariant;
        total += K[s];
        if (t_forced_variant >= 0) continue;
        if (odl_fp8_gemm_runs(M, N, K[s], 0) > 1) return kNoVariant;
        const int64_t steps = K[s] / 128;
        const Route route = route_of(M, N, K[s], ODL_BF16, s > 0, -1);
        if (route.variant == kThinVariant) apart += 4.0 + 0.0027 * gemm_thin_rows(M, N, cus) * (double)steps + (s > 0 ? 0.4 * c_mb : 0.0);
        else apart += s > 0 ? accumulate_us(route.variant, t, steps, c_mb, cus) : launch_us(route.variant, t, steps, cus);
    }
    if (t.t128 > 0x7ffffff0LL || (double)N * 2.0 * 264.0 >= 2147483648.0) return kNoVariant;
    if (t_forced_variant >= 0) return t_forced_variant >= kDeepWideVariant ? t_forced_variant : kNoVariant;
    const double steps = (double)(total / 128);
    int best = kNoVariant;
    double cost = 0.97 * apart;
    auto offer = [&](int variant, double us) { if (us < cost) { cost = us; best = variant; } };
    if (t.t128 <= cus) offer(kDeepVariant, launch_us(kDeepVariant, t, total / 128, cus));
    if (t.t192 <= cus) offer(kDeep192Variant, launch_us(kDeep192Variant, t, total / 128, cus));
    const double rest = (double)(t.wide % cus) / cus;
    offer(kDeepWideVariant, (t.wide <= cus ? 1.0 : (double)(t.wide / cus) + (rest > 0.0 ? 0.55 + 0.45 * rest : 0.0)) * (0.85 * steps + 7.0));
    return best;
}

extern "C" int odl_fp8_gemm_chain_route(int pairs, const int64_t *K, int64_t M, int64_t N) {
    if (!K) {
        set_error(ODL_ERR_ARG, "odl_fp8_gemm_chain_route: null pointer");
        return -1;
    }
    return chain_variant(pairs, K, M, N);
}

extern "C" int odl_fp8_gemm_nt_chain(int pairs, const uint8_t *const *a, const uint8_t *const *b, const int64_t *K, int64_t M, int64_t N, int fmt_a,
                                     int fmt_b, const float *const *sa_inv, const float *const *sb_inv, void *c, odl_stream_t stream_) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (!a || !b || !K || !c || !sa_inv || !sb_inv) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_chain: null pointer");
    const int variant = chain_variant(pairs, K, M, N);
    if (variant == kNoVariant)
        return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt_chain: %d products of %lld x %lld do not run in one launch (odl_fp8_gemm_chain_route)", pairs, (long long)M, (long long)N);
    if (fmt_b == ODL_FP8_E4M3 ? fmt_a != ODL_FP8_E4M3 && fmt_a != ODL_FP8_E5M2 : fmt_b != ODL_FP8_E5M2 || fmt_a != ODL_FP8_E5M2)
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_chain: formats %d, %d", fmt_a, fmt_b);
    const int bm = kVariants[variant].bm, bn = kVariants[variant].bn;
    GemmChain gc;
    gc.count = pairs;
    if (reinterpret_cast<uintptr_t>(c) & 15) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt_chain: output must be 16-byte aligned");
    for (int s = 0; s < pairs; ++s) {
        if (!a[s] || !b[s] || !sa_inv[s] || !sb_inv[s]) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_nt_chain: null pointer in product %d", s);
        if ((reinterpret_cast<uintptr_t>(a[s]) & 15) || (reinterpret_cast<uintptr_t>(b[s]) & 15))
            return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_nt_chain: operands must be 16-byte aligned (product %d)", s);
        GemmArgs &g = gc.m[s];
        g.a = a[s]; g.b = b[s]; g.c = c; g.sa = sa_inv[s]; g.sb = sb_inv[s]; g.bias = nullptr;
        g.M = M; g.N = N; g.K = K[s];
        g.sa_vec = g.sb_vec = 0;
        g.out_dtype = ODL_BF16;
        g.tiles_m = (int)((M + bm - 1) / bm); g.tiles_n = (int)((N + bn - 1) / bn);
    }
    launch_gemm_deep_chain(bm, bn, fmt_a, fmt_b, gc, cu_count(), stream);
    return check_launch("odl_fp8_gemm_nt_chain");
}
