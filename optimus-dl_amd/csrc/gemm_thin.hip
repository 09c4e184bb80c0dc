// FP8 GEMM for outputs of few tiles: the waves of a block share K instead of the output.
//
// Bound by: the time one compute unit takes to fetch its operands.  A decode step (16 .. 128 rows) or a small data
// gradient has far fewer 128 x 128 tiles than the chip has compute units, and a block of the tiled kernels then walks all
// of K alone: 32 blocks for 32 x 4096 x 14336.  Here a block owns a small tile (16 MT x 16 NT) and its eight waves take
// the 128-byte K steps in turn, so the chip is filled eight times sooner, and neighbouring waves read neighbouring
// 128-byte lines of the same rows.  Lines are fetched whole, eight rows an instruction, and turned into fragments in the
// wave's own part of LDS: with a lane reading the 16-byte chunks of its own row straight into its fragment, every load
// touches a line per lane, and the address unit, not the memory, is what the kernel waits for (32 x 4096 x 14336:
// 24.3 us that way, 19.2 with whole lines, 53.3 with the 128 x 128 kernel).
// Up to two K steps of loads are in flight per wave while a third is multiplied.
// The eight partial tiles are added in wave order through LDS at the end: the result does not depend on scheduling, and
// there is no workspace and no second launch.
#include "gemm_common.h"
#include "swiglu.h"

namespace odl {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kThinWaves = 8;

// D[i][j] += sum_k first[i][k] * second[j][k]: lane l supplies row l % 16 and 32 of the 128 K-bytes of both operands
// (which 32 does not matter as long as both use the same ones); it receives D[4 * (l / 16) + e][l % 16], e = 0..3.
template <int F1, int F2>
__device__ __forceinline__ v4f mfma_16x16x128(v8i first, v8i second, v4f acc) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(first, second, acc, F1, F2, 0, 0, 0, 0);
}

// operand rows of a K step: NT tiles of B, then MT tiles of A; LDS of a block: a stage, later a set of partial tiles, per wave
template <int MT, int NT>
constexpr int thin_lds_bytes() { return kThinWaves * (16 * (MT + NT) * 128 > MT * NT * 1024 ? 16 * (MT + NT) * 128 : MT * NT * 1024); }

// GATED: the first column tile comes from g.b and the second from `up`, 16 columns of each.
template <int MT, int NT, int FA, int FB, bool GATED>
__device__ __forceinline__ void thin_partial_tiles(const GemmArgs &g, const uint8_t *up, int64_t m0, int64_t n0, uint8_t *lds) {
    constexpr int ROWS = 16 * (MT + NT);
    constexpr int LOADS = ROWS / 8;                       // a wave instruction fetches whole 128-byte lines of 8 rows
    constexpr int DEPTH = 3;                              // K steps held in registers
    constexpr int STAGE = ROWS * 128;
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int row = lane % 16, group = lane / 16;

    // Memory -> registers: lane l reads chunk l % 8 of row l / 8 of each group of eight rows (rows past the end are read
    // as the last row; what they give is not stored).  Registers -> the wave's own LDS, chunks swizzled so that the
    // fragment reads of 16 rows spread over the banks.
    uint32_t src[LOADS];                                  // byte offsets: an operand is smaller than 4 GiB
    uint8_t *stage = lds + wave * STAGE;
    int dst[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int r = 8 * j + lane / 8, chunk = lane % 8;
        src[j] = (uint32_t)((j < 2 * NT ? min(n0 + (GATED ? r % 16 : r), g.N - 1) : min(m0 + r - 16 * NT, g.M - 1)) * g.K) + 16 * chunk;
        dst[j] = r * 128 + ((chunk ^ swz(r)) << 4);
    }
    struct Lines { u32x4 v[LOADS]; };
    auto fetch = [&](Lines &f, int64_t k) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) f.v[j] = *reinterpret_cast<const u32x4 *>((j < 2 * NT ? (GATED && j >= 2 ? up : g.b) : g.a) + k + src[j]);
    };
    v4f acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[t][u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto fragment = [&](int first_row) -> v8i {           // the chunks `group` and `group + 4` of this lane's row
        const int r = first_row + row;
        const v4i lo = *reinterpret_cast<const v4i *>(stage + r * 128 + ((group ^ swz(r)) << 4));
        const v4i hi = *reinterpret_cast<const v4i *>(stage + r * 128 + (((group + 4) ^ swz(r)) << 4));
        return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    };
    auto multiply = [&](const Lines &f) {
        // LDS operations of one wave execute in order; the clobbers keep the compiler from moving a lane's reads of what
        // other lanes wrote before its own writes, and the writes of the next step before these reads
#pragma unroll
        for (int j = 0; j < LOADS; ++j) *reinterpret_cast<u32x4 *>(stage + dst[j]) = f.v[j];
        asm volatile("" ::: "memory");
        v8i b[NT];
#pragma unroll
        for (int u = 0; u < NT; ++u) b[u] = fragment(16 * u);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const v8i a = fragment(16 * (NT + t));
#pragma unroll
            for (int u = 0; u < NT; ++u) acc[t][u] = mfma_16x16x128<FB, FA>(b[u], a, acc[t][u]);
        }
        asm volatile("" ::: "memory");
    };

    const int steps = (int)(g.K / 128);
    const int mine = wave < steps ? (steps - 1 - wave) / kThinWaves + 1 : 0;      // K steps wave, wave + 8, ..
    if (mine > 0) {
        // step indexes are clamped, not tested: the loads of the last iterations repeat the last step of this wave
        auto at = [&](int i) { return ((int64_t)min(i, mine - 1) * kThinWaves + wave) * 128; };
        Lines f[DEPTH];
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d) fetch(f[d], at(d));
        for (int i = 0; i < mine; i += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                if (i + d >= mine) break;
                fetch(f[(d + DEPTH - 1) % DEPTH], at(i + d + DEPTH - 1));
                multiply(f[d]);
            }
        }
    }
    __syncthreads();                                      // the partial tiles lie where the operands were
    v4f(*partial)[MT * NT][64] = reinterpret_cast<v4f (*)[MT * NT][64]>(lds);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) partial[wave][t * NT + u][lane] = acc[t][u];
    __syncthreads();
}

// the eight waves' sums of a tile, in wave order
template <int MT, int NT>
__device__ __forceinline__ v4f thin_sum(const uint8_t *lds, int tile) {
    const v4f(*partial)[MT * NT][64] = reinterpret_cast<const v4f (*)[MT * NT][64]>(lds);
    const int lane = threadIdx.x % 64;
    v4f sum = partial[0][tile][lane];
#pragma unroll
    for (int w = 1; w < kThinWaves; ++w) {
        const v4f p = partial[w][tile][lane];
        sum.x = sum.x + p.x; sum.y = sum.y + p.y; sum.z = sum.z + p.z; sum.w = sum.w + p.w;
    }
    return sum;
}

template <int MT, int NT, int FA, int FB>
__global__ __launch_bounds__(64 * kThinWaves) void gemm_nt_thin_kernel(const GemmArgs g) {
    __shared__ __align__(1024) uint8_t lds[thin_lds_bytes<MT, NT>()];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int row = lane % 16, group = lane / 16;
    // the row tiles of one column tile run side by side: they read the same rows of B
    const int64_t m0 = (int64_t)(blockIdx.x % g.tiles_m) * (16 * MT), n0 = (int64_t)(blockIdx.x / g.tiles_m) * (16 * NT);
    thin_partial_tiles<MT, NT, FA, FB, false>(g, nullptr, m0, n0, lds);

    const float *bias = reinterpret_cast<const float *>(g.bias);
    for (int tile = wave; tile < MT * NT; tile += kThinWaves) {
        const v4f sum = thin_sum<MT, NT>(lds, tile);
        const int64_t m = m0 + 16 * (tile / NT) + row, n = n0 + 16 * (tile % NT) + 4 * group;
        if (m >= g.M || n >= g.N) continue;               // N % 4 == 0: the four columns are in or out together
        const float sa = g.sa[m * g.sa_vec];
        float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = v[e] * (sa * g.sb[(n + e) * g.sb_vec]);
            if (bias) v[e] = v[e] + bias[n + e];
        }
        if (g.out_dtype == ODL_BF16) {
            u32x2 *c = reinterpret_cast<u32x2 *>(reinterpret_cast<uint16_t *>(g.c) + m * g.N + n);
            if (g.accumulate) {
                const u32x2 old = *c;
                v[0] = v[0] + bf16_lo(old.x); v[1] = v[1] + bf16_hi(old.x); v[2] = v[2] + bf16_lo(old.y); v[3] = v[3] + bf16_hi(old.y);
            }
            *c = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
            float4 *c = reinterpret_cast<float4 *>(reinterpret_cast<float *>(g.c) + m * g.N + n);
            if (g.accumulate) {
                const float4 old = *c;
                v[0] = v[0] + old.x; v[1] = v[1] + old.y; v[2] = v[2] + old.z; v[3] = v[3] + old.w;
            }
            *c = float4{v[0], v[1], v[2], v[3]};
        }
    }
}

// ---------------------------------------------------------------- gate and up of a SwiGLU MLP, and their product
// h = bf16( silu(bf16(x . gate^T)) * bf16(x . up^T) ) for a few rows, and the partial maxima of |h| that odl_fp8_cast_dynamic
// takes: a block owns 16 columns of both weights.  Bound by reading them (32 x 14336 x 4096 twice: 117 MB).  As two products
// and a third launch for the activation: 16.5 + 15.4 + 6 us, here 33, and two more launches for the host to issue, of the
// seven that a decode step of the MLP took.  At most kParts blocks, each its own entry of `parts`, so that nobody has to
// zero them.  The sums and roundings of those three launches where the products take the thin kernel (K >= 2048); with a shorter K
// they take 128 x 128 tiles, whose one chain of 64 products at a time rounds elsewhere, equally far from 64 bits (relative root
// mean square 1.470e-5 for 32 x 768 -> 2048, 1.489e-5 for 64 x 1024 -> 3072, either way).
template <int MT, int FA, int FB>
__global__ __launch_bounds__(64 * kThinWaves) void gemm_thin_swiglu_kernel(const GemmArgs g, const uint8_t *up, const float *s_up, float *parts) {
    __shared__ __align__(1024) uint8_t lds[thin_lds_bytes<MT, 2>()];
    __shared__ uint32_t red[MT];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int row = lane % 16, group = lane / 16;
    const float sg = g.sa[0] * g.sb[0], su = g.sa[0] * s_up[0];
    uint32_t am = 0;
    const int tiles = g.tiles_m * g.tiles_n;
    for (int p = blockIdx.x; p < tiles; p += gridDim.x) {
        const int64_t m0 = (int64_t)(p % g.tiles_m) * (16 * MT), n0 = (int64_t)(p / g.tiles_m) * 16;
        thin_partial_tiles<MT, 2, FA, FB, true>(g, up, m0, n0, lds);
        if (wave < MT) {
            const v4f a = thin_sum<MT, 2>(lds, 2 * wave), b = thin_sum<MT, 2>(lds, 2 * wave + 1);
            const int64_t m = m0 + 16 * wave + row, n = n0 + 4 * group;
            if (m < g.M && n < g.N) {
                const u32x2 h = {swiglu_fwd_pair(pack_bf16x2(a.x * sg, a.y * sg), pack_bf16x2(b.x * su, b.y * su)),
                                 swiglu_fwd_pair(pack_bf16x2(a.z * sg, a.w * sg), pack_bf16x2(b.z * su, b.w * su))};
                *reinterpret_cast<u32x2 *>(reinterpret_cast<uint16_t *>(g.c) + m * g.N + n) = h;
                am = max_u16x2(am, max_u16x2(abs_bf16x2(h.x), abs_bf16x2(h.y)));
            }
        }
        __syncthreads();                                  // the partial tiles lie where the next tile's operands go
    }
    am = wave_max_u32(fold_u16x2_to_f32bits(am));
    if (wave < MT && lane == 0) red[wave] = am;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < MT; ++w) am = max(am, red[w]);
        parts[blockIdx.x] = bits_to_float(am);
    }
    if (blockIdx.x == 0)
        for (int j = (int)gridDim.x + threadIdx.x; j < ODL_FP8_AMAX_PARTS; j += 64 * kThinWaves) parts[j] = 0.0f;
}

template <int MT, int NT, int FA, int FB>
static void launch_thin(const GemmArgs &args, hipStream_t stream) {
    GemmArgs g = args;
    g.tiles_m = (int)((g.M + 16 * MT - 1) / (16 * MT));
    g.tiles_n = (int)((g.N + 16 * NT - 1) / (16 * NT));
    hipLaunchKernelGGL((gemm_nt_thin_kernel<MT, NT, FA, FB>), dim3((unsigned)(g.tiles_m * g.tiles_n)), dim3(64 * kThinWaves), 0, stream, g);
}

template <int FA, int FB>
static void launch_thin_fmt(int mt, int nt, const GemmArgs &g, hipStream_t stream) {
    if (mt == 1 && nt == 1) launch_thin<1, 1, FA, FB>(g, stream);
    else if (mt == 1) launch_thin<1, 2, FA, FB>(g, stream);
    else if (mt == 2 && nt == 1) launch_thin<2, 1, FA, FB>(g, stream);
    else if (mt == 2) launch_thin<2, 2, FA, FB>(g, stream);
    else launch_thin<4, 2, FA, FB>(g, stream);
}

// The tile with the least operand rows fetched by the busiest compute unit, rows of a tile x rounds of blocks (32 x 4096 x
// 14336 with 16 x 16, 32 x 16, 32 x 32 and 64 x 32 tiles, 64, 48, 64 and 96 rows: 22.3, 19.2, 22.5 and 24.3 us).  With
// the tile picked so and K >= 2048 a launch takes about 4 us + 2.7 ns per such row and K step: over 16 measured shapes
// within 14 % but for 32 x 14336 x 4096 (15.1 by the rule, 18.6 measured), 128 x 4096 x 14336 (33.0, 28.5) and 32 x 768 x
// 50304 (38.0, 29.3).  It says nothing of tiles that are not picked (up to 65 % too much: one round of large tiles) nor of
// several rounds over a short K (half of what they take).  At all 16 shapes the picked tile was the fastest of the five, or tied.
static int thin_tile(int64_t M, int64_t N, int num_cus, int *mt_out, int *nt_out) {
    static const int tiles[][2] = {{4, 2}, {2, 2}, {2, 1}, {1, 2}, {1, 1}};
    int64_t best = INT32_MAX;
    for (const auto &tile : tiles) {
        const int64_t blocks = ((M + 16 * tile[0] - 1) / (16 * tile[0])) * ((N + 16 * tile[1] - 1) / (16 * tile[1]));
        const int64_t rows = 16 * (tile[0] + tile[1]) * ((blocks + num_cus - 1) / num_cus);
        if (rows < best) { best = rows; *mt_out = tile[0]; *nt_out = tile[1]; }
    }
    return (int)best;
}

int gemm_thin_rows(int64_t M, int64_t N, int num_cus) {
    int mt, nt;
    return thin_tile(M, N, num_cus, &mt, &nt);
}

void launch_gemm_thin(int fa, int fb, const GemmArgs &g, int num_cus, hipStream_t stream) {
    int mt = 1, nt = 1;
    thin_tile(g.M, g.N, num_cus, &mt, &nt);
    if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E4M3) launch_thin_fmt<ODL_FP8_E4M3, ODL_FP8_E4M3>(mt, nt, g, stream);
    else if (fa == ODL_FP8_E5M2 && fb == ODL_FP8_E4M3) launch_thin_fmt<ODL_FP8_E5M2, ODL_FP8_E4M3>(mt, nt, g, stream);
    else if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E5M2) launch_thin_fmt<ODL_FP8_E4M3, ODL_FP8_E5M2>(mt, nt, g, stream);
    else launch_thin_fmt<ODL_FP8_E5M2, ODL_FP8_E5M2>(mt, nt, g, stream);
}

template <int FA, int FB>
static void launch_thin_swiglu(const GemmArgs &args, const uint8_t *up, const float *s_up, float *parts, hipStream_t stream) {
    GemmArgs g = args;
    const int mt = g.M <= 16 ? 1 : g.M <= 32 ? 2 : 4;
    g.tiles_m = (int)((g.M + 16 * mt - 1) / (16 * mt));
    g.tiles_n = (int)((g.N + 15) / 16);
    const int tiles = g.tiles_m * g.tiles_n;
    const dim3 grid((unsigned)(tiles < ODL_FP8_AMAX_PARTS ? tiles : ODL_FP8_AMAX_PARTS)), block(64 * kThinWaves);
    if (mt == 1) hipLaunchKernelGGL((gemm_thin_swiglu_kernel<1, FA, FB>), grid, block, 0, stream, g, up, s_up, parts);
    else if (mt == 2) hipLaunchKernelGGL((gemm_thin_swiglu_kernel<2, FA, FB>), grid, block, 0, stream, g, up, s_up, parts);
    else hipLaunchKernelGGL((gemm_thin_swiglu_kernel<4, FA, FB>), grid, block, 0, stream, g, up, s_up, parts);
}

}  // namespace odl

using namespace odl;

extern "C" int odl_fp8_gemm_swiglu(const uint8_t *x, const uint8_t *gate, const uint8_t *up, int64_t M, int64_t N, int64_t K, int fmt_x, int fmt_w,
                                   const float *sx_inv, const float *sg_inv, const float *su_inv, void *h, float *parts, odl_stream_t stream_) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (!x || !gate || !up || !sx_inv || !sg_inv || !su_inv || !h || !parts) return set_error(ODL_ERR_ARG, "odl_fp8_gemm_swiglu: null pointer");
    if ((fmt_x != ODL_FP8_E4M3 && fmt_x != ODL_FP8_E5M2) || (fmt_w != ODL_FP8_E4M3 && fmt_w != ODL_FP8_E5M2))
        return set_error(ODL_ERR_ARG, "odl_fp8_gemm_swiglu: formats %d, %d", fmt_x, fmt_w);
    if (M <= 0 || N <= 0 || K <= 0 || M > 64 || N % 4 != 0 || K % 128 != 0 || (double)N * (double)K >= 4294967296.0 || (double)M * (double)K >= 4294967296.0)
        return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_swiglu: at most 64 rows, N %% 4 == 0, K %% 128 == 0, operands under 4 GiB; got %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
    for (const void *p : {(const void *)x, (const void *)gate, (const void *)up, (const void *)h})
        if (reinterpret_cast<uintptr_t>(p) & 15) return set_error(ODL_ERR_SHAPE, "odl_fp8_gemm_swiglu: operands and output must be 16-byte aligned");
    GemmArgs g;
    g.a = x; g.b = gate; g.c = h; g.sa = sx_inv; g.sb = sg_inv; g.bias = nullptr;
    g.M = M; g.N = N; g.K = K;
    g.sa_vec = g.sb_vec = 0;
    g.out_dtype = ODL_BF16;
    if (fmt_x == ODL_FP8_E4M3 && fmt_w == ODL_FP8_E4M3) launch_thin_swiglu<ODL_FP8_E4M3, ODL_FP8_E4M3>(g, up, su_inv, parts, stream);
    else if (fmt_x == ODL_FP8_E5M2 && fmt_w == ODL_FP8_E4M3) launch_thin_swiglu<ODL_FP8_E5M2, ODL_FP8_E4M3>(g, up, su_inv, parts, stream);
    else if (fmt_x == ODL_FP8_E4M3 && fmt_w == ODL_FP8_E5M2) launch_thin_swiglu<ODL_FP8_E4M3, ODL_FP8_E5M2>(g, up, su_inv, parts, stream);
    else launch_thin_swiglu<ODL_FP8_E5M2, ODL_FP8_E5M2>(g, up, su_inv, parts, stream);
    return check_launch("odl_fp8_gemm_swiglu");
}
