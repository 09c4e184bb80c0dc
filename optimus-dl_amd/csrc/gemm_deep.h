// FP8 GEMM for outputs of about one tile per compute unit: 256 x 128, 128 x 192 or 128 x 128 tiles, four waves, three LDS stages,
// explicit software pipeline.  Both operands K-contiguous, K % 128 == 0, any M and N, every scale form (block scales
// K-step-major), `accumulate`.
//
// Bound by: what LDS delivers.  A K step of a 128 x 128 tile reads 64 KB of LDS and writes 32 KB of it, 768 cycles at 128
// bytes a cycle, for 512 cycles of MFMA; of a 256 x 128 tile 96 + 48 KB, 1152 cycles for 1024.  With the whole chip busy
// the caches come into it: 18 - 20 TB/s of operand panels is the most they were seen to deliver.  Measured per K step
// (slope over K = 2048 .. 8192): 128 x 128 0.29 us (705 cycles) with 24 units busy, 0.35 with 192, 0.40 with 256; 256 x 128
// 0.52 and 0.71.  A launch costs 5.5 - 7 us beside its steps.  128 x 192 tiles lie between: 0.66 us with 256 units busy and
// operands from HBM, which is what 40 KB a step take there (see warm_operands; nobody is left to warm).  They fill the
// chip where 256 x 128 tiles leave a quarter of it idle: 8192 x 768 x 3072 26.1 -> 24.4 us, x 50304 327 -> 285.  (256 x 192 in two
// stages does not fit the registers: 2.7 us a step.)
//
// A block that has a compute unit to itself has nobody to hide its waits behind, so nothing here waits for what was
// asked for recently:
//   * a wave tile is 64 x 64, 64 x 96 or 128 x 64, four waves: with eight waves of 64 x 32 LDS would deliver half as much again;
//   * the fragments of step kt + 1 (both halves) stream from LDS into one set of registers while the MFMAs of step kt
//     work on the other.  Half a step ahead, as the 256 x 256 kernels do it, is 256 cycles of MFMA here and less than
//     LDS takes (0.39 us a step instead of 0.29);
//   * the loads of step kt + 3 go into the stage that step kt lay in, two whole steps ahead of their use;
//   * one barrier per step.  Behind it everybody has read stage kt into registers and everybody's loads of stage kt + 1
//     have landed: a wave's loads complete in order, so that is "at most one step's loads outstanding".
// Against the four-stage tiled kernel (eight waves, fragments read as they are needed), which keeps the contractions of less
// than 16 steps (gemm_few_tiles), bf16 outputs in us: 2048 x 2048 x 2048 12.1 -> 11.6, x 4096 20.8 -> 18.6, x 8192 36.4 -> 31.2; 3072 x 1024 x 8192 fp32
// 35.3 -> 28.3; 1024 x 4096 x 14336 65.3 -> 52.5 (operands in the memory-side cache).  Four or five stages: the same but for
// 0.2 us a launch and stage.
//
// Rows past the end of a matrix, and steps past the end of K, are requested through descriptors that end there: they
// read as zero.  Loads, waits and barriers of the K loop are inline asm (the compiler would wait for every load in front
// of every LDS read).
#pragma once

#include "gemm_common.h"

namespace odl {

namespace {

constexpr int NW = 4, STAGES = 3;

// MX: block scales (g.mx_sa / g.mx_sb, K-step-major: dword [step][row] = the four scale bytes of a row in that step).  A wave
// brings 64 dwords of A and B rows to LDS beside its operand loads; a lane reads the dwords of its rows with the fragments
// and shifts them so that byte 0 / byte 2 are what it supplies in the first / second half (lanes 32 .. 63 hold the odd
// blocks).  The instruction takes registers 0 .. 3 / 4 .. 7 as K 16 g .. / 32 + 16 g .., so the chunks of a fragment are lg and
// 2 + lg; without scales any 32 of the 64 bytes do.
//
// Args: one product, several side by side (GemmGroup), or several that are added up (GemmChain).  Of a chain a block stays on its
// tile through all products; the loads go on from one to the next three steps ahead, as they do from step to step, with other
// descriptors and another row pitch.  Behind a product that is not the last its value, the old one added, is rounded to bf16 and waits
// in registers (two to a register) instead of in memory: the roundings of a launch per product with `accumulate`.
template <int TM, int TN, int FA, int FB, bool MX, class Args>
__global__ __launch_bounds__(256) void gemm_nt_deep_kernel(const Args args) {
    constexpr int BM = 64 * TM, BN = 64 * TN, WM = 32 * TM, WN = 32 * TN;
    constexpr int A_BYTES = BM * 128, CODES = (BM + BN) * 128, STAGE = CODES + (MX ? (BM + BN + 255) / 256 * 1024 : 0);
    constexpr int LA = BM / 32, LB = BN / 32, SC = MX ? (BM + BN + 255) / 256 : 0, PER = LA + LB + SC;         // direct-to-LDS loads per wave and step
    constexpr int MFMAS = TM * TN, TNS = TN % 2 ? 1 : TN;             // TNS: sub-tiles of a row staged together
    constexpr int GM = BM == 256 ? 4 : 8;                             // tile rows walked together
    static_assert(PER * (STAGES - 1) <= 63, "the counter holds 63 loads");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * STAGE];

    const int total = tile_count(args);
    const int per_xcd = (total + 7) / 8;
    int pid = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if ((int)blockIdx.x >= 8 * per_xcd) {
        const int spare = (int)blockIdx.x - 8 * per_xcd, spares = (int)gridDim.x - 8 * per_xcd;
        if constexpr (std::is_same_v<Args, GemmArgs>) warm_operands(args, spare, spares, 10);
        else if constexpr (std::is_same_v<Args, GemmGroup>) warm_operands(args.m[spare % args.count], spare / args.count, spares / args.count, 10);
        else
            for (int p = 0; p < args.count; ++p) warm_operands(args.m[p], spare, spares, 10);
        return;
    }
    if (pid >= total) return;
    const GemmArgs &g = product_of(args, pid);
    const int in_group = GM * g.tiles_n;
    const int first_m = (pid / in_group) * GM;
    const int group_rows = min(g.tiles_m - first_m, GM);
    const int m0 = __builtin_amdgcn_readfirstlane((first_m + (pid % in_group) % group_rows) * BM);
    const int n0 = __builtin_amdgcn_readfirstlane(((pid % in_group) / group_rows) * BN);

    const int lane = threadIdx.x % 64;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int wm0 = (wave / 2) * WM, wn0 = (wave % 2) * WN;
    const int lr = lane % 32, lg = lane / 32;
    constexpr bool CHAIN = std::is_same_v<Args, GemmChain>;
    static_assert(!CHAIN || !MX, "a chain has one scale per operand");
    const int KT = (int)(g.K / 128);

    auto rsrc_for = [&](const uint8_t *base, int row0, int rows, int nk) -> v4i {
        const uint64_t addr = reinterpret_cast<uint64_t>(base + (int64_t)row0 * nk);
        return v4i{(int)(uint32_t)addr, (int)(uint32_t)(addr >> 32), rows * nk, 0x00020000};
    };
    v4i rsrc_a, rsrc_b;
    int voff[LA > LB ? LA : LB];
    auto aim_loads = [&](const GemmArgs &p) {             // (CHAIN: once per product)
        rsrc_a = rsrc_for(p.a, m0, (int)min(g.M - m0, (int64_t)BM), (int)p.K);
        rsrc_b = rsrc_for(p.b, n0, (int)min(g.N - n0, (int64_t)BN), (int)p.K);
#pragma unroll
        for (int j = 0; j < (LA > LB ? LA : LB); ++j) {
            const int row = (wave + j * NW) * 8 + lane / 8;
            voff[j] = row * (int)p.K + (((lane % 8) ^ swz(row)) << 4);
        }
    };
    aim_loads(g);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)lds;
    auto dma = [&](const v4i &rsrc, uint32_t lds_addr, int vo, int so) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     ::"s"(lds_addr), "v"(vo), "s"(rsrc), "s"(so));
    };
    // scale dwords 256 q + 64 wave + lane of a stage: the rows of A, then the rows of B, then nothing
    v4i rsrc_s[SC > 0 ? SC : 1];
    int step_s[SC > 0 ? SC : 1];
    if constexpr (MX) {
#pragma unroll
        for (int q = 0; q < SC; ++q) {
            const int first = 256 * q + 64 * wave;
            const bool is_a = first < BM;
            const int row = is_a ? m0 + first : n0 + first - BM, rows = (int)(is_a ? g.M : g.N) - row;
            const uint64_t addr = reinterpret_cast<uint64_t>(is_a ? g.mx_sa : g.mx_sb) + (int64_t)row * 4;
            step_s[q] = (int)(is_a ? g.M : g.N) * 4;
            // up to the end of the whole array (the scalar offset counts in the bounds check); rows past the last one of a
            // group of 64 get the next step's dwords, and what they scale is zero and not stored
            rsrc_s[q] = v4i{(int)(uint32_t)addr, (int)(uint32_t)(addr >> 32), first < BM + BN && rows > 0 ? KT * step_s[q] - row * 4 : 0, 0x00020000};
        }
    }
    // load j of a step (`live` false: a step past the end of K, of which nothing is read)
    auto issue_one = [&](uint32_t stage, const v4i &da, const v4i &db, bool live, int kt, int j) {
        if (j < LA) dma(da, stage + (wave + j * NW) * 1024, voff[j], kt * 128);
        else if (j < LA + LB) dma(db, stage + A_BYTES + (wave + (j - LA) * NW) * 1024, voff[j - LA], kt * 128);
        else {
            v4i d = rsrc_s[j - LA - LB];
            d.z = live ? d.z : 0;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                         ::"s"(stage + CODES + (j - LA - LB) * 1024 + wave * 256), "v"(4 * lane), "s"(d), "s"(kt * step_s[j - LA - LB]));
        }
    };

    int ra[2][2], rb[2][2];                       // [e][h ^ (t & 1)] byte offsets inside a stage (fragment 0)
    {
        const int rowa = wm0 + lr, rowb = wn0 + lr;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int chunk = MX ? lg + 2 * e : 2 * lg + e;
                ra[e][p] = rowa * 128 + (((chunk ^ swz(rowa)) ^ (4 * p)) << 4);
                rb[e][p] = A_BYTES + rowb * 128 + (((chunk ^ swz(rowb)) ^ (4 * p)) << 4);
            }
    }
    auto read = [&](const uint8_t *stage, const int (&r)[2][2], int t, int h) -> v8i {
        const v4i lo = *reinterpret_cast<const v4i *>(stage + r[0][h ^ (t & 1)] + t * 4096);
        const v4i hi = *reinterpret_cast<const v4i *>(stage + r[1][h ^ (t & 1)] + t * 4096);
        return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    };

    v16f acc[TM][TN];
    struct Frags { v8i a[2][TM], b[2][TN]; int ea[TM], eb[TN]; };     // a step's fragments, both halves, and their scale dwords
    Frags fx, fy;
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][u][e] = 0.0f;

    auto request = [&](int s) {
        v4i da = rsrc_a, db = rsrc_b;
        da.z = s < KT ? da.z : 0;
        db.z = s < KT ? db.z : 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) issue_one(lds0 + s * STAGE, da, db, s < KT, s, j);
    };
#pragma unroll
    for (int s = 0; s < STAGES; ++s) request(s);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PER * (STAGES - 1)) : "memory");
    constexpr int FR = 2 * (TM + TN), N2 = 2 * MFMAS;
    auto read_frag = [&](Frags &f, const uint8_t *stage, int i) {
        const int h = i / (TM + TN), k = i % (TM + TN);
        if (k < TN) f.b[h][k] = read(stage, rb, k, h);
        else f.a[h][k - TN] = read(stage, ra, k - TN, h);
    };
    auto read_scales = [&](Frags &f, const uint8_t *stage) {
        const int *d = reinterpret_cast<const int *>(stage + CODES);
#pragma unroll
        for (int t = 0; t < TM; ++t) f.ea[t] = d[wm0 + 32 * t + lr];
#pragma unroll
        for (int u = 0; u < TN; ++u) f.eb[u] = d[BM + wn0 + 32 * u + lr];
    };
    if constexpr (MX) read_scales(fx, lds);
#pragma unroll
    for (int i = 0; i < FR; ++i) read_frag(fx, lds, i);

    constexpr int PF = (FR + N2 / 2 - 1) / (N2 / 2);     // fragments requested behind an MFMA: all behind the first half
    constexpr int PD = (PER + N2 - 1) / N2;
    int cur = 0;                                   // byte offset of the stage that step kt lies in
    // CHAIN: the step that is requested next, of product `ahead`, which has `ahead_steps` (at least four, an even number)
    int ahead = 0, ahead_kt = STAGES, ahead_steps = KT;
    bool live = true;
    auto step = [&](Frags &now, Frags &then, int kt) {
        const int nxt = cur + STAGE == STAGES * STAGE ? 0 : cur + STAGE;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PER * (STAGES - 2)) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        v4i da = rsrc_a, db = rsrc_b;
        const int want = CHAIN ? ahead_kt : kt + STAGES;
        const bool there = CHAIN ? live : want < KT;
        da.z = there ? da.z : 0;
        db.z = there ? db.z : 0;
        int ea[TM], eb[TN];
        if constexpr (MX) {
#pragma unroll
            for (int t = 0; t < TM; ++t) ea[t] = (int)((uint32_t)now.ea[t] >> (8 * lg));
#pragma unroll
            for (int u = 0; u < TN; ++u) eb[u] = (int)((uint32_t)now.eb[u] >> (8 * lg));
        }
#pragma unroll
        for (int i = 0; i < N2; ++i) {
            const int h = i / MFMAS, t = i % MFMAS / TN, u = i % TN;
            if constexpr (!MX) acc[t][u] = mfma_32x32x64<FB, FA>(now.b[h][u], now.a[h][t], acc[t][u]);
            else if (h == 0) acc[t][u] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(now.b[0][u], now.a[0][t], acc[t][u], FB, FA, 0, eb[u], 0, ea[t]);
            else acc[t][u] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(now.b[1][u], now.a[1][t], acc[t][u], FB, FA, 2, eb[u], 2, ea[t]);
            if (MX && i == 0) read_scales(then, lds + nxt);
#pragma unroll
            for (int f = PF * i; f < PF * (i + 1) && f < FR; ++f) read_frag(then, lds + nxt, f);
#pragma unroll
            for (int j = PD * i; j < PD * (i + 1) && j < PER; ++j) issue_one(lds0 + cur, da, db, there, want, j);
            __builtin_amdgcn_sched_barrier(0);
        }
        cur = nxt;
        if constexpr (CHAIN) {
            if (++ahead_kt == ahead_steps) {
                ahead_kt = 0;
                live = ++ahead < args.count;
                if (live) {
                    ahead_steps = (int)(args.m[ahead].K / 128);
                    aim_loads(args.m[ahead]);
                }
            }
        }
    };
    if constexpr (CHAIN) {
        uint32_t carry[TM][TN][8];
        for (int p = 0; p < args.count; ++p) {
            const GemmArgs &product = args.m[p];
            const int steps = (int)(product.K / 128);
            for (int kt = 0; kt < steps; kt += 2) {
                step(fx, fy, kt);
                step(fy, fx, kt + 1);
            }
            const float scale = product.sa[0] * product.sb[0];
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
                for (int u = 0; u < TN; ++u)
#pragma unroll
                    for (int e = 0; e < 16; e += 2) {
                        float lo = acc[t][u][e] * scale, hi = acc[t][u][e + 1] * scale;
                        if (p > 0) {
                            lo = lo + bf16_lo(carry[t][u][e / 2]);
                            hi = hi + bf16_hi(carry[t][u][e / 2]);
                        }
                        const bool last = p + 1 == args.count;        // (the epilogue rounds it)
                        if (!last) carry[t][u][e / 2] = pack_bf16x2(lo, hi);
                        acc[t][u][e] = last ? lo : 0.0f;
                        acc[t][u][e + 1] = last ? hi : 0.0f;
                    }
        }
    } else {
        for (int kt = 0; kt < KT; kt += 2) {
            step(fx, fy, kt);
            if (kt + 1 < KT) step(fy, fx, kt + 1);
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    constexpr int EPI_BYTES = 32 * (TN * 32 * 4 + 16);
    static_assert(NW * EPI_BYTES <= STAGES * STAGE, "epilogue staging must fit in the operand stages");
    // Staged also where the matrix ends between two slabs of the wave tile: 5632 and 2048 columns leave a third or two thirds of
    // the last 128 x 192 tile, and with direct stores for it 1024 x 5632 x 2048 took 20.4 us instead of 14.7 (two 128 x 128 blocks
    // per unit: 16.7), 2304 x 2048 x 1024 13.0 instead of 10.5.
    if (g.N % 8 == 0 && (n0 + wn0 + WN <= g.N || g.N % (32 * TNS) == 0)) {
        uint8_t *wave_lds = lds + wave * EPI_BYTES;
        if constexpr (CHAIN) epilogue_staged<true, TM, TN, TNS, true, true>(g, acc, wave_lds, m0 + wm0, n0 + wn0, lane);
        else if (g.accumulate) {
            if (g.out_dtype == ODL_BF16) epilogue_staged_accumulate<true, TM, TN, 1, true>(g, acc, wave_lds, m0 + wm0, n0 + wn0, lane);
            else epilogue_staged_accumulate<false, TM, TN, 1, true>(g, acc, wave_lds, m0 + wm0, n0 + wn0, lane);
        } else if (g.out_dtype == ODL_BF16) epilogue_staged<true, TM, TN, TNS, true>(g, acc, wave_lds, m0 + wm0, n0 + wn0, lane);
        else epilogue_staged<false, TM, TN, TNS, true>(g, acc, wave_lds, m0 + wm0, n0 + wn0, lane);
    } else if constexpr (!CHAIN) {               // (the columns of a chain are whole slabs)
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int u = 0; u < TN; ++u) {
                if (g.out_dtype == ODL_BF16) store_tile<true, false>(g, acc[t][u], m0 + wm0 + 32 * t + lr, n0 + wn0 + 32 * u + 4 * lg);
                else store_tile<false, false>(g, acc[t][u], m0 + wm0 + 32 * t + lr, n0 + wn0 + 32 * u + 4 * lg);
            }
    }
}

}  // namespace

}  // namespace odl
