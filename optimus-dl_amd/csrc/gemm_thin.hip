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
// One K step of loads is in flight per wave while another is multiplied.  (Two, with the steps past a wave's last requested
// like the others, fetched half as much again where a wave has four steps: 32 x 14336 x 4096 19.3 us against 17.7, 32 x 4096 x
// 14336 13.1 against 12.1, 128 x 768 x 3072 5.3 against 4.8.)
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

template <int MT, int NT, int FA, int FB>
__device__ __forceinline__ void thin_partial_tiles(const GemmArgs &g, int64_t m0, int64_t n0, uint8_t *lds) {
    constexpr int ROWS = 16 * (MT + NT);
    constexpr int LOADS = ROWS / 8;                       // a wave instruction fetches whole 128-byte lines of 8 rows
    constexpr int DEPTH = 2;                              // K steps held in registers
    constexpr int STAGE = ROWS * 128;
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int row = lane % 16, group = lane / 16;

    // Memory -> registers: lane l reads chunk l % 8 of row l / 8 of each group of eight rows (rows past the end are read
    // as the last row; what they give is not stored).  Registers -> the wave's own LDS, chunks swizzled so that the
    // fragment reads of 16 rows spread over the banks.
    uint8_t *stage = lds + wave * STAGE;
    uint32_t src[LOADS];                                  // byte offsets: an operand is smaller than 4 GiB
    int dst[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int r = 8 * j + lane / 8, chunk = lane % 8;
        src[j] = (uint32_t)((j < 2 * NT ? min(n0 + r, g.N - 1) : min(m0 + r - 16 * NT, g.M - 1)) * g.K) + 16 * chunk;
        dst[j] = r * 128 + ((chunk ^ swz(r)) << 4);
    }
    struct Lines { u32x4 v[LOADS]; };
    auto fetch = [&](Lines &f, int64_t k) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) f.v[j] = *reinterpret_cast<const u32x4 *>((j < 2 * NT ? g.b : g.a) + k + src[j]);
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
__device__ __forceinline__ v4f thin_sum(const uint8_t *lds, int tile, int lane) {
    const v4f(*partial)[MT * NT][64] = reinterpret_cast<const v4f (*)[MT * NT][64]>(lds);
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
    thin_partial_tiles<MT, NT, FA, FB>(g, m0, n0, lds);

    const float *bias = reinterpret_cast<const float *>(g.bias);
    for (int tile = wave; tile < MT * NT; tile += kThinWaves) {
        const v4f sum = thin_sum<MT, NT>(lds, tile, lane);
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
// takes.  As two products and a third launch for the activation: 16.5 + 15.4 + 6 us, and two more launches for the host to issue.
// Bound by what a compute unit can fetch, 60 - 70 bytes a nanosecond: the rows of both weights once (32 x 14336 x 4096 twice: 117
// MB, 459 KB a unit), and x again for every tile.  So a block owns as many columns as give every unit one block, in units of
// eight of gate and eight of up (56 of each there, 144 operand rows in place of four tiles of 64): 30.3 -> 21.8 us with the
// weights in the memory-side cache, 37.6 -> 28.3 from memory; 32 x 5632 x 2048 11.4 -> 7.4, 64 x 3072 x 1024 11.1 -> 5.6.
// At most kParts blocks, each its own entry of `parts`, so that nobody has to
// zero them.  The sums and roundings of those three launches where the products take the thin kernel (K >= 2048); with a shorter K
// they take 128 x 128 tiles, whose one chain of 64 products at a time rounds elsewhere, equally far from 64 bits (relative root
// mean square 1.470e-5 for 32 x 768 -> 2048, 1.489e-5 for 64 x 1024 -> 3072, either way).

// The first of a tile's eight columns: where the matrix ends inside them, its last eight (computed twice, the same), all of them
// where there are fewer.
__device__ __forceinline__ int64_t gated_column(int64_t n, int64_t N) { return max(min(n, N - 8), (int64_t)0); }

// The eight waves' partial tiles, in LDS.  16 operand rows are eight columns of gate and the same eight of up.  A step goes straight
// to the wave's own stage in LDS (144 rows of it would take 72 registers, and the two steps that a pipeline in registers needs do
// not fit); while a wave waits for its step, the other seven have theirs under way, 18 KB each.
template <int MT, int NT, int FA, int FB>
__device__ __forceinline__ void gated_partial_tiles(const GemmArgs &g, const uint8_t *up, int64_t m0, int64_t n0, uint8_t *lds) {
    constexpr int ROWS = 16 * (MT + NT), LOADS = ROWS / 8, STAGE = ROWS * 128;
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int row = lane % 16, group = lane / 16;
    const int K = (int)g.K, steps = K / 128;

    // load j brings rows 8 j + lane / 8, chunk lane % 8 of the stage holding chunk (lane % 8) ^ swz(row) of the row; swz(8 j + r) =
    // r ^ (j & 7).  The eight rows of a load of gate or up are reached through the scalar offset, those of x through the lane's
    // (rows past its end are read as its last one).
    const uint32_t row_b = (uint32_t)min((int64_t)(lane / 8), g.N - 1) * (uint32_t)K;
    uint32_t row_a[2 * MT];
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) row_a[j] = (uint32_t)min(m0 + 8 * j + lane / 8, g.M - 1) * (uint32_t)K;
    const int chunk = (lane % 8) ^ (lane / 8);
    auto window = [](const uint8_t *base, int64_t bytes) -> v4i {
        const uint64_t addr = reinterpret_cast<uint64_t>(base);
        return v4i{(int)(uint32_t)addr, (int)(uint32_t)(addr >> 32), (int)(uint32_t)bytes, 0x00020000};
    };
    const v4i wa = window(g.a, g.M * g.K), wg = window(g.b, g.N * g.K), wu = window(up, g.N * g.K);
    uint32_t base_b[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) base_b[u] = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)gated_column(n0 + 8 * u, g.N) * (uint32_t)K));
    uint8_t *stage = lds + wave * STAGE;
    const uint32_t stage_at = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)lds + wave * STAGE;
    auto request = [&](int step) {
        const uint32_t k = (uint32_t)step * 128;
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const bool of_a = j >= 2 * NT;
            const uint32_t at = (of_a ? row_a[of_a ? j - 2 * NT : 0] : row_b) + ((chunk ^ (j & 7)) << 4);
            const uint32_t so = of_a ? k : base_b[of_a ? 0 : j / 2] + k;
            // s_nop 4: the scalars may come from vector instructions (the build checks the distance)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         ::"s"(stage_at + j * 1024), "v"(at), "s"(of_a ? wa : j % 2 ? wu : wg), "s"(so));
        }
    };
    auto fragment = [&](int first_row) -> v8i {           // the chunks `group` and `group + 4` of this lane's row
        const int r = first_row + row;
        const v4i lo = *reinterpret_cast<const v4i *>(stage + r * 128 + ((group ^ swz(r)) << 4));
        const v4i hi = *reinterpret_cast<const v4i *>(stage + r * 128 + (((group + 4) ^ swz(r)) << 4));
        return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    };
    v4f acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[t][u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if (wave < steps) request(wave);
    for (int step = wave; step < steps; step += kThinWaves) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        v8i a[MT], b[NT];
#pragma unroll
        for (int t = 0; t < MT; ++t) a[t] = fragment(16 * (NT + t));
#pragma unroll
        for (int u = 0; u < NT; ++u) b[u] = fragment(16 * u);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // the stage has been read ...
        __builtin_amdgcn_sched_barrier(0);
        if (step + kThinWaves < steps) request(step + kThinWaves);    // ... and may be written again
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u) acc[t][u] = mfma_16x16x128<FB, FA>(b[u], a[t], acc[t][u]);
    }
    __syncthreads();                                      // the partial tiles lie where the operands were
    v4f(*partial)[MT * NT][64] = reinterpret_cast<v4f (*)[MT * NT][64]>(lds);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) partial[wave][t * NT + u][lane] = acc[t][u];
    __syncthreads();
}

template <int MT, int NT, int FA, int FB>
__global__ __launch_bounds__(64 * kThinWaves) void gemm_thin_swiglu_kernel(const GemmArgs g, const uint8_t *up, const float *s_up, float *parts) {
    constexpr int TILES = MT * NT;
    __shared__ __align__(1024) uint8_t lds[thin_lds_bytes<MT, NT>()];
    __shared__ uint32_t red[kThinWaves];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const float sg = g.sa[0] * g.sb[0], su = g.sa[0] * s_up[0];
    uint32_t am = 0;
    const int tiles = g.tiles_m * g.tiles_n;
    for (int p = blockIdx.x; p < tiles; p += gridDim.x) {
        const int64_t m0 = (int64_t)(p % g.tiles_m) * (16 * MT), n0 = (int64_t)(p / g.tiles_m) * (8 * NT);
        gated_partial_tiles<MT, NT, FA, FB>(g, up, m0, n0, lds);
        // half a wave per tile: its lanes 0 .. 31 hold gate, 32 .. 63 up, lane l row l % 16 and columns 4 (l / 16) .. of the eight
        for (int first = 2 * wave; first < TILES; first += 2 * kThinWaves) {
            const int tile = first + lane / 32, half = lane % 32;
            if (tile >= TILES) continue;
            const v4f a = thin_sum<MT, NT>(lds, tile, half), b = thin_sum<MT, NT>(lds, tile, half + 32);
            const int64_t m = m0 + 16 * (tile / NT) + half % 16, n = gated_column(n0 + 8 * (tile % NT), g.N) + 4 * (half / 16);
            if (m >= g.M || n >= g.N || n0 + 8 * (tile % NT) >= g.N) continue;
            const u32x2 h = {swiglu_fwd_pair(pack_bf16x2(a.x * sg, a.y * sg), pack_bf16x2(b.x * su, b.y * su)),
                             swiglu_fwd_pair(pack_bf16x2(a.z * sg, a.w * sg), pack_bf16x2(b.z * su, b.w * su))};
            *reinterpret_cast<u32x2 *>(reinterpret_cast<uint16_t *>(g.c) + m * g.N + n) = h;
            am = max_u16x2(am, max_u16x2(abs_bf16x2(h.x), abs_bf16x2(h.y)));
        }
        __syncthreads();                                  // the partial tiles lie where the next tile's operands go
    }
    am = wave_max_u32(fold_u16x2_to_f32bits(am));
    if (lane == 0) red[wave] = am;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kThinWaves; ++w) am = max(am, red[w]);
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

// The columns of a block (eight times nt) with the least operand rows fetched by the busiest compute unit.  The choices are what the
// widths it was measured at want (3072, 5632, 14336) and steps between; six is not built, though 12288 columns would fill 256 units with
// it (they take seven: 144 operand rows a step in 220 blocks in place of 128).
static int swiglu_nt(int mt, int64_t M, int64_t N, int num_cus) {
    static const int choices[] = {1, 2, 3, 4, 5, 7};
    int64_t best = INT64_MAX;
    int best_nt = 1;
    for (const int nt : choices) {
        if (mt == 4 && nt > 4) break;                     // (a stage per wave: 8 x 128 (16 mt + 16 nt) bytes of LDS)
        const int64_t blocks = ((M + 16 * mt - 1) / (16 * mt)) * ((N + 8 * nt - 1) / (8 * nt));
        const int64_t rows = 16 * (mt + nt) * ((blocks + num_cus - 1) / num_cus);
        if (rows < best) { best = rows; best_nt = nt; }
    }
    return best_nt;
}

template <int MT, int NT, int FA, int FB>
static void launch_thin_swiglu_tile(const GemmArgs &args, const uint8_t *up, const float *s_up, float *parts, hipStream_t stream) {
    GemmArgs g = args;
    g.tiles_m = (int)((g.M + 16 * MT - 1) / (16 * MT));
    g.tiles_n = (int)((g.N + 8 * NT - 1) / (8 * NT));
    const int tiles = g.tiles_m * g.tiles_n;
    const dim3 grid((unsigned)(tiles < ODL_FP8_AMAX_PARTS ? tiles : ODL_FP8_AMAX_PARTS)), block(64 * kThinWaves);
    hipLaunchKernelGGL((gemm_thin_swiglu_kernel<MT, NT, FA, FB>), grid, block, 0, stream, g, up, s_up, parts);
}

template <int MT, int FA, int FB>
static void launch_thin_swiglu_rows(int nt, const GemmArgs &g, const uint8_t *up, const float *s_up, float *parts, hipStream_t stream) {
    if (nt == 1) launch_thin_swiglu_tile<MT, 1, FA, FB>(g, up, s_up, parts, stream);
    else if (nt == 2) launch_thin_swiglu_tile<MT, 2, FA, FB>(g, up, s_up, parts, stream);
    else if (nt == 3) launch_thin_swiglu_tile<MT, 3, FA, FB>(g, up, s_up, parts, stream);
    else if (nt == 4 || MT == 4) launch_thin_swiglu_tile<MT, 4, FA, FB>(g, up, s_up, parts, stream);
    else if constexpr (MT < 4) {
        if (nt == 5) launch_thin_swiglu_tile<MT, 5, FA, FB>(g, up, s_up, parts, stream);
        else launch_thin_swiglu_tile<MT, 7, FA, FB>(g, up, s_up, parts, stream);
    }
}

template <int FA, int FB>
static void launch_thin_swiglu(const GemmArgs &g, const uint8_t *up, const float *s_up, float *parts, hipStream_t stream) {
    const int mt = g.M <= 16 ? 1 : g.M <= 32 ? 2 : 4, nt = swiglu_nt(mt, g.M, g.N, device_cu_count());
    if (mt == 1) launch_thin_swiglu_rows<1, FA, FB>(nt, g, up, s_up, parts, stream);
    else if (mt == 2) launch_thin_swiglu_rows<2, FA, FB>(nt, g, up, s_up, parts, stream);
    else launch_thin_swiglu_rows<4, FA, FB>(nt, g, up, s_up, parts, stream);
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
