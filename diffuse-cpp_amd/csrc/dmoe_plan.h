// dmoe_plan.h — which kernels a projection, an LM head, a dense MLP or a routed
// layer's Q4_K experts take: pure host functions of the sizes, the weights' type and the context's
// switches.  A call decides once, from all of its tokens, and plans its
// workspace and launches its kernels from that one decision.  No HIP here:
// tests/test_plan.py compiles this file for the CPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace dmoe {

// Alternative kernels kept selectable for measurement, read from the
// environment by dmoe_create into its context (never in a forward):
//   DMOE_Q4K_COLUMN_BLOCKS = 1, 2, 4  column blocks of the Q4_K items (0: by tokens per expert)
//   DMOE_DOWN_FUSED = 1               few-token Q4_K down products as the single fused launch
//   DMOE_GATEUP_LDS = 1               the LDS-ring gate/up kernel instead of the register ring
//   DMOE_EXPERT_TILE = 0 / 1          the tile kernels (k_expert_tile.hip) off / on for every N
//   DMOE_EXPERT_GEMM = 0 / 1          the Q4_K grouped GEMM (k_expert_gemm.hip) off / on for every N
//   DMOE_PROJ_GEMM = 0 / 1            Q4_K, Q6_K and Q8_0 projections (attention, LM head; Q4_K and Q6_K dense MLP)
//                                     past the few-token kernels on that GEMM off / on for every N
struct KernelSwitches {
    int q4k_column_blocks = 0;
    int expert_tile = -1;                // -1: by tokens per expert
    int expert_gemm = -1;                // -1: by tokens per expert
    int proj_gemm = -1;                  // -1: by tokens
    int attn_waves = 0;                  // 0: by grid size, else 4 or 8 per workgroup
    bool down_fused = false;
    bool gateup_lds = false;
    int n_cu = 256;                      // compute units of the context's device (not a switch)
};

// Kernel family of a matrix, by its type and shape (dense_path, head_path).
enum WeightPath { DP_GEMV = 0, DP_Q4K, DP_Q80, DP_F16, DP_Q6K };

// The few-token kernel (k_proj.hip): Q4_K and Q6_K, up to 32 tokens a launch.
constexpr int PROJ_MAX_TOKENS = 32;
constexpr int PROJ_WAVES = 8, PROJ_TMAX = 6;     // wavefronts of a workgroup, 16-row tiles of a wavefront at most
constexpr int PROJ_STEP_BYTES = 4672;            // activations of 8 tokens and a super-block

inline bool proj_ok(int R, int K, int N)
{
    return R > 0 && R % 16 == 0 && K > 0 && K % 256 == 0 && N > 0 && N <= PROJ_MAX_TOKENS;
}

// Tiles per wavefront (T) and reduction slices (KS, a divisor of K / 256)
// for a shape, by a cost model fitted to measured launches on the 256-CU
// part this is built for (at 32 tokens): a launch takes about 8 us plus
// 1.9 us per tile step of a wavefront (T S) and round of workgroups over the
// CUs, and the slices' sums, when there are several, about 2 us plus 0.6 us
// per MB to add (k_proj_reduce / k_proj_swiglu); the activation steps every
// workgroup reads from L2 (4.7 KB per 8 tokens and super-block) count 0.1 us
// per MB.  Ties go to more tiles per wavefront.
struct ProjPlan {
    int T;                   // 16-row tiles per wavefront
    int KS;                  // reduction slices
    double us;               // the model's estimate
};

inline ProjPlan proj_plan(int R, int K, int M, int N)
{
    const int tiles = R / 16, nsb = K / 256;
    const int nb = (N + 7) / 8;
    ProjPlan best{1, nsb, -1.0};
    for (int t = PROJ_TMAX; t >= 1; t--)
        for (int ks = 1; ks <= nsb; ks++) {
            if (nsb % ks) continue;
            const long wgs = (long)((tiles + PROJ_WAVES * t - 1) / (PROJ_WAVES * t)) * M * ks;
            const long rounds = (wgs + 255) / 256;
            double us = 8.0 + 1.9 * t * (nsb / ks) * rounds;
            if (ks > 1) us += 2.0 + 0.6 * ((double)M * ks * N * R * 4 / 1e6);
            us += 0.1 * ((double)wgs * (nsb / ks) * nb * PROJ_STEP_BYTES / 1e6);
            if (best.us < 0.0 || us < best.us) best = ProjPlan{t, ks, us};
        }
    return best;
}

// Q6_K past 32 tokens in chunks of 32 of that kernel, by the model: a
// launch and its share of the conversions take 1.1 times its estimate and 1 us.
inline double proj_chunks_us(int R, int K, int M, int N)
{
    auto chunk_us = [&](int n) { return 1.1 * proj_plan(R, K, M, n).us + 1.0; };
    const int whole = N / PROJ_MAX_TOKENS, rest = N % PROJ_MAX_TOKENS;
    return (whole ? whole * chunk_us(PROJ_MAX_TOKENS) : 0.0) + (rest ? chunk_us(rest) : 0.0);
}

// Output rows up to which a few-token Q4_K projection runs one workgroup per
// 16 rows (k_down_rows); above it (the LM head) the expert kernel's items.
constexpr int PROJ_ROWS_MAX = 32768;

// The grouped GEMM (k_expert_gemm.hip): rows of a gate/up and of a down item.
constexpr int EXPERT_GEMM_GU_ROWS = 128, EXPERT_GEMM_DN_ROWS = 256;

inline bool expert_gemm_q4k_ok(int H, int FF, int SF, bool shared)
{
    if (H % EXPERT_GEMM_DN_ROWS || FF % EXPERT_GEMM_GU_ROWS || H < 512 || FF < 512 || H % 256 || FF % 256) return false;
    if (shared && SF != FF) return false;
    return true;
}

// Whether the routed Q4_K experts of N tokens take the GEMM (units of up to 128
// pairs) rather than the tile kernels (units of up to 32).  From 64 pairs per
// expert on, averaged over all experts, always.  From 32 on it depends on
// whether its larger items still fill the chip and whether the pairs fill its
// blocks of 32: block routing gathers a block's pairs on few experts, plain
// top-k leaves each with about the average.  Items below are the gate/up
// launch's, one unit per expert.  Measured (tile kernels against GEMM, us):
//   4,096 x 1,024, 256 experts, top 8 (2,176 items): 1,024 tokens 666 / 591, 1,025 752 / 727
//   2,048 x 512, 256 experts, top 8 (1,088): 1,024 tokens 245 / 233, 1,025 280 / 282, 1,409 322 / 314
//   2,048 x 512, 128 experts, top 8 (544): 512 tokens 148 / 124, 513 158 / 167
//   2,048 x 1,024, 16 experts, top 2 (160): 256 tokens 88 / 98; 480 92 / 101
//   1,024 x 512, 32 experts, top 4 (144): 256 tokens 58 / 74; 480 70 / 77
// Where the tile kernels do not take the shape (moe_ff 2,048), the GEMM is
// ahead of the item kernels from 32 on: 4,096 x 2,048, 8 experts, top 2, 128
// tokens 172 / 152.
constexpr long GEMM_Q4K_MIN_AVG = 32, GEMM_Q4K_MIN_AVG_PLAIN = 40, GEMM_Q4K_ANY_AVG = 64;

inline bool moe_gemm_pays(int N, int top_k, int E, int FF, bool shared, bool block_routing, bool tile_ok, int n_cu)
{
    const long avg = (long)N * top_k / (E > 0 ? E : 1);
    if (avg >= GEMM_Q4K_ANY_AVG || avg < GEMM_Q4K_MIN_AVG) return avg >= GEMM_Q4K_ANY_AVG;
    if (!tile_ok) return true;
    const long items = (long)(E + (shared ? (N + 63) / 64 : 0)) * (FF / EXPERT_GEMM_GU_ROWS);
    return block_routing ? items >= 2L * n_cu : avg >= GEMM_Q4K_MIN_AVG_PLAIN && items >= 3L * n_cu;
}

// Q4_K, Q6_K and Q8_0 projections of proj_gemm_min_tokens or more tokens run on the
// grouped GEMM's down launch (k_expert_gemm.hip) with shared units only: 64 tokens
// (128 digit rows) per unit, 256 output rows per item, the reduction split
// into slices of 2 or more super-blocks, as many as minimise the static
// schedule's rounds x steps plus the slices' own traffic.  ks is the slice
// count, 0 where the GEMM does not take the shape; rounds the workgroups' items
// one after another, us the estimate.
struct ProjGemm {
    int ks;
    long rounds;
    double us;
};

constexpr int PROJ_GEMM_MIN_TOKENS = 33;

// Q6_K matrices of an LM head's rows take the GEMM (in units of 32 tokens)
// from 17 tokens on where q6k_head_gemm_pays says so, from 25 on always: the
// few-token kernel's work per weight grows by the eight tokens, the GEMM's not.
// Few-token kernel against GEMM at 25 / 32 tokens, us: 157,184 x 4,096 220 / 224 against
// 177 / 182, 157,184 x 2,048 121 / 123 against 107 / 103, 33,024 x 2,048 51 / 54
// against 46 / 48.
constexpr int PROJ_GEMM_MIN_TOKENS_Q6K_HEAD = 17, PROJ_GEMM_ANY_TOKENS_Q6K_HEAD = 25;

// Q8_0 projections have no few-token kernel of their own: against the expert
// kernel's items of 8 tokens the GEMM takes the attention half of 1 / 8 / 20
// tokens from 95 / 98 / 99 us to 46 / 49 / 53, and an LM head of 16 / 32 tokens
// from 233 / 468 us to 160 / 194; one item of the expert kernel covers a head
// of up to 8 tokens (128 / 133 us at 1 / 8 tokens against 137 / 148).  Between
// these q80_gemm_pays weighs the two.
constexpr int PROJ_GEMM_MIN_TOKENS_Q80 = 1, PROJ_GEMM_MIN_TOKENS_Q80_HEAD = 9;

inline int proj_gemm_min_tokens(int path, int rows)
{
    if (path == DP_Q80) return rows > PROJ_ROWS_MAX ? PROJ_GEMM_MIN_TOKENS_Q80_HEAD : PROJ_GEMM_MIN_TOKENS_Q80;
    return path == DP_Q6K && rows > PROJ_ROWS_MAX ? PROJ_GEMM_MIN_TOKENS_Q6K_HEAD : PROJ_GEMM_MIN_TOKENS;
}

inline ProjGemm proj_gemm(const KernelSwitches &sw, int path, int rows, int K, int N)
{
    ProjGemm g{0, 0, 0.0};
    if ((path != DP_Q4K && path != DP_Q6K && path != DP_Q80) || sw.proj_gemm == 0 ||
        (sw.proj_gemm < 0 && N < proj_gemm_min_tokens(path, rows)) ||
        !expert_gemm_q4k_ok(rows, K, K, true) || 2L * N * K >= (1L << 31))
        return g;
    const long items = (long)((N + 63) / 64) * (rows / 256);
    const int nsb = K / 256;
    const long grid = (sw.n_cu + 7) / 8 * 8;
    // rounds of the static schedule x super-blocks per item at ~4.5 us per
    // step, plus the slices written and read again at ~4 TB/s.  (A step of a
    // full unit measures 3.5 us of Q4_K, 4.4 of Q6_K, 5 of Q8_0, less of part
    // units and 5.4 of Q6_K in large heads at their lower clock; one figure
    // serves the slice count, the rules below take their own.)
    for (int ks = 1; ks <= 16; ks *= 2) {
        if (nsb % ks || (ks > 1 && nsb / ks < 2)) continue;
        const long rounds = (items * ks + grid - 1) / grid;
        double us = 4.5 * (double)(rounds * (nsb / ks));
        if (ks > 1) us += (double)ks * N * rows * 8 / 4e6;
        if (ks == 1 || us < g.us) g = ProjGemm{ks, rounds, us};
    }
    return g;
}

// Q8_0: the GEMM g against the expert kernel's items of 8 tokens x 256 rows,
// which spread few rows over more compute units and take an item's whole
// reduction at about 2.2 us per super-block.  A step of the GEMM lasts 2 / 3 /
// 4 / 5 us with up to 16 / 32 / 48 / 64 tokens in a unit; slices cost a few us
// and their traffic, the item kernel a conversion launch (1 us).  A head of
// 405 shapes (512 to 16,384 rows x 512 to 4,096, 1 to 512 tokens) measured on
// both, items / GEMM: 2,048 x 512 at 16 tokens 22 / 20 us, at 64 22 / 27; 4,096 x
// 1,024 at 32 tokens 26 / 25, at 48 26 / 27; 4,096 x 2,816 (a prime number of
// super-blocks: one slice) at 16 tokens 39 / 36, at 32 39 / 46, at 128 41 / 71;
// 16,384 x 2,816 at 64 tokens 63 / 72, at 96 86 / 72.
inline bool q80_gemm_pays(const ProjGemm &g, int rows, int K, int N, int n_cu)
{
    const long grid = (n_cu + 7) / 8 * 8, items = (long)((N + 7) / 8) * (rows / 256);
    const int nsb = K / 256;
    double gemm_us = (1.0 + std::min(4, (N + 15) / 16)) * (double)(g.rounds * (nsb / g.ks));
    if (g.ks > 1) gemm_us += 3.0 + (double)g.ks * N * rows * 8 / 4e6;
    return gemm_us <= 2.2 * nsb * (double)((items + grid - 1) / grid) + 1.0;
}

// A Q6_K head of 17 to 24 tokens: a step of the GEMM's units of 32 tokens
// lasts about 3.55 us, its slices an own launch and their traffic; the few-token
// kernel takes nine tenths of its estimate.  Over 135 measured heads (33,024 to 157,184 rows x
// 1,024 to 5,120) never the slower by more than 1 percent.  Few-token kernel against
// GEMM at 20 tokens, us: 65,536 x 4,096 85 against 71, 100,352 x 2,048 81 against
// 70 (the GEMM); 157,184 x 2,048 101 against 104, 81,920 x 1,024 43 against 47 (row groups that
// leave its last round half empty, or the slices' launch on a short
// reduction).
inline bool q6k_head_gemm_pays(const ProjGemm &g, int rows, int K, int N)
{
    double gemm_us = 3.55 * (double)(g.rounds * (K / 256 / g.ks));
    if (g.ks > 1) gemm_us += 6.0 + (double)g.ks * N * rows * 8 / 4e6;
    return gemm_us <= 0.9 * proj_plan(rows, K, 1, N).us;
}

// Q6_K past the few-token kernel: the GEMM (gemm_us) against chunks of 32 tokens
// of that kernel.  They read the matrix again for every chunk but split a
// reduction by any divisor, the GEMM by powers of two: with an odd number of
// super-blocks a workgroup walks all of them (4.5 us each) however few rows
// there are.  Over 270 projections (512 to 16,384 rows x 512 to 4,096, 33 to
// 160 tokens) the rule never picks the slower; chunks against GEMM, us:
// 1,024 x 2,816 at 33 / 65 / 160 tokens 37 / 52 / 84 against 54 / 58 / 59, 8,192 x 2,816 at
// 33 / 64 52 / 63 against 55 / 58, 1,024 x 4,096 at 33 40 against 28.  Dense
// MLPs, 175 shapes, nowhere more than 3 percent behind the chunks: 4,096 x 11,008 at
// 33 tokens 181 against 215, 1,024 x 2,816 at 64 56 against 73, 4,096 x 9,216 at 33 140
// against 107 (six shapes, mostly n_ff 11,008 at 65 to 192 tokens, keep the chunks where the
// GEMM would be 10 to 30 percent ahead).
template <class ChunksUs>
bool q6k_gemm_pays(double gemm_us, int N, ChunksUs &&chunks_us)
{
    // (the model is asked only when it can matter: no chunk's estimate is below 11.8 us)
    const int chunks = (N + PROJ_MAX_TOKENS - 1) / PROJ_MAX_TOKENS;
    return gemm_us <= 11.8 * chunks || gemm_us <= chunks_us();
}

// What a projection y [N][rows] = W x, or a dense MLP, runs on:
//   few          the few-token kernel, `chunk` tokens a launch (Q6_K of any N:
//                it has no item kernel; Q4_K in one launch)
//   gemm_ks > 0  the grouped GEMM over all tokens, the (down) reduction in
//                gemm_ks slices
//   neither      the item kernels over all tokens
// `chunk` is the tokens whose converted activations are held at once.
struct ProjRoute {
    bool few;
    int gemm_ks;
    int chunk;
};

inline ProjRoute proj_route(const KernelSwitches &sw, int path, int rows, int K, int N)
{
    const ProjGemm g = proj_gemm(sw, path, rows, K, N);
    ProjRoute r{false, g.ks, N};
    if (path == DP_Q80 && g.ks && sw.proj_gemm < 0 && !q80_gemm_pays(g, rows, K, N, sw.n_cu)) r.gemm_ks = 0;
    if (path == DP_Q6K && g.ks && sw.proj_gemm < 0 && N > PROJ_MAX_TOKENS &&
        !q6k_gemm_pays(g.us + (g.ks > 1 ? 2.0 : 0.0), N, [&] { return proj_chunks_us(rows, K, 1, N); }))
        r.gemm_ks = 0;
    if (path == DP_Q6K && g.ks && sw.proj_gemm < 0 && N < PROJ_GEMM_ANY_TOKENS_Q6K_HEAD &&
        !q6k_head_gemm_pays(g, rows, K, N))
        r.gemm_ks = 0;
    const bool int4_6 = path == DP_Q4K || path == DP_Q6K;
    if (int4_6 && proj_ok(rows, K, N) && (N < proj_gemm_min_tokens(path, rows) || !r.gemm_ks))
        return ProjRoute{true, 0, N};
    if (path == DP_Q6K && !r.gemm_ks) return ProjRoute{true, 0, std::min(N, PROJ_MAX_TOKENS)};
    return r;
}

// The dense MLP: gate and up as one two-matrix projection and down as
// another, both on the few-token kernel (Q6_K past it in chunks, where the
// GEMM does not take the shape or is slower), or the GEMM's gate/up and down launches.
inline ProjRoute dense_route(const KernelSwitches &sw, int path, int H, int FF, int N)
{
    const ProjGemm g = proj_gemm(sw, path, H, FF, N);
    int ks = path == DP_Q80 || 2L * N * H >= (1L << 31) ? 0 : g.ks;
    if (path == DP_Q6K && ks && sw.proj_gemm < 0 && N > PROJ_MAX_TOKENS) {
        const long grid = (sw.n_cu + 7) / 8 * 8, items = (long)((N + 63) / 64) * (FF / EXPERT_GEMM_GU_ROWS);
        const double gu_us = 4.5 * (double)((items + grid - 1) / grid * (H / 256));
        if (!q6k_gemm_pays(gu_us + g.us + (ks > 1 ? 2.0 : 0.0), N,
                           [&] { return proj_chunks_us(FF, H, 2, N) + proj_chunks_us(H, FF, 1, N); }))
            ks = 0;
    }
    const int chunk = path == DP_Q6K && !ks ? std::min(N, PROJ_MAX_TOKENS) : N;
    const bool int4_6 = path == DP_Q4K || path == DP_Q6K;
    if (int4_6 && proj_ok(FF, H, chunk) && proj_ok(H, FF, chunk)) return ProjRoute{true, 0, chunk};
    return ProjRoute{false, ks, N};
}

} // namespace dmoe
