// k_expert_gemm.hip — Q4_K and, in projections, Q6_K and Q8_0 products as a
// grouped int8-MFMA GEMM when many rows share each weight (prompt prefill and the sampler's large windows,
// N = 32 (blk + 1) of a thousand tokens and more):
// src/diffuse-moe-graph.cpp:264-269 (ggml's mul_mat_id over Q4_K weights
// with Q8_K activations), the shared expert of :280-286 (F32 activations
// as two int8 digits) and, with shared units only, projections of more than a
// few tokens.
//
// Units: work-list entries of up to 128 pairs of one expert (eight 16-row
// blocks) and chunks of 64 tokens of the shared expert (two int8 digit rows
// each, eight blocks again).  Items: (unit, row group); an item is 256 weight
// rows, 32 per wavefront: gate/up items 128 h rows (wavefront w: the gate and
// the up tile of rows 16 w .. + 15), down items 256 n_embd rows (wavefront
// w: rows 32 w .. + 31).  One workgroup per CU walks its items
// (schedule_item): with row groups a multiple of 8 per unit, one row group of
// every unit runs on one XCD (workgroup b is placed on XCD b % 8) and
// consecutive units together, so chunks of one expert next to each other read
// its weights once from HBM and then from that XCD's L2 (four row groups, the
// gate/up units of moe_ff 512, alternate between two XCDs, so such a row group
// is read twice).  The units go out by falling size, the shared ones first,
// then the work list (by_size): at 2,048 tokens a CU runs about seven units of
// one to eight blocks, and in expert order a wavefront was busy for 0.76
// (gate/up) of the launch.  That order costs the combine launch after it,
// which finds less of the products in the last-level cache.  2,048 tokens, each
// pass alone, us, expert order and shared units last / by size, shared last /
// by size, shared first: gate/up 556 / 501 / 502, down 311 / 305 / 303, combine
// 61 / 66 / 70, the layer 1,058 / 1,033 / 1,040; 1,024 tokens 613 / 599 / 589.
//
// Pipeline: one step per 256-value super-block of the reduction.  A
// wavefront's 32 weight rows are private to it: one LDS buffer of their own
// (the tiled layout's runs as they lie), read to registers at the start of a
// step and refilled for the next step right after, so it needs no second
// stage.  The step's 128 activation rows lie in a ring of three stages shared
// by the workgroup, filled two steps ahead.  Both by LDS-direct loads, across
// items; the waits count the loads issued since, so the younger activation
// stage stays in flight.
//
// Products: v_mfma_i32_32x32x32_i8 on 32 activation rows x 32 weight rows.
// The sub-block scales are folded into the int8 weight operand once per step
// (sc = 8 sh + sl, sh and sl below 8: sh q and sl q are int8) and applied to
// all the unit's rows.  What bounds a step is the SIMD's issue and, in large
// calls that run on end, the clock that issue leaves (below): per 32 x 32 output
// tile and super-block 16 int8 MFMAs of 32 cycles (twice the useful products:
// the two scale digits), 80 VALU instructions of scale
// epilogue (five per output) and the fold's ~150 shared by up to four tiles.
// Launches with shared units only (MERGE) keep a token's two digit rows in
// separate blocks of 32, so that both digits of an output lie in one lane and
// take one epilogue (8 instructions per token against 10).
//
// Measured (calls on end, against 16 x 16 MFMA tiles with one epilogue per
// digit row, the weights and activations of a step in one of two shared stages,
// units in expert order): Q4_K MoE layer of 2,048 tokens 1,073 -> 1,012 us, of
// 1,024 tokens 646 -> 582; dense MLP of 160 tokens 129 -> 110 us, of 512 314 ->
// 286; attention half of 777 tokens 268 -> 247, of 2,048 612 -> 603 us.  In
// calls on end the card lowers its clock under the large ones: MoE layer of
// 2,048 tokens 2,146 MHz (2,398 with the former tiles), attention half of 2,048
// 2,312 (2,400), Q6_K head of 256 tokens 1,968; the dense MLP of 160 tokens stays at
// 2,398.  The launches around the GEMM slow down with it, so the layer gains less than
// the launches do in short runs (620 -> 497 and 314 -> 300 us at 2,048 tokens).
//
// Arithmetic: the integer sums of every super-block are compute_sb's exactly
// (8 sum (sh q) a + sum (sl q) a = sum_j sc_j S_j), then one f32 epilogue per
// super-block in super-block order rounded by q4k_epi, so the outputs of routed
// launches equal the tile and column-block kernels' bit for bit.  MERGE
// launches round a token's two digits together, in a full block of 32 tokens
// also the min term's sum (past 2^24, in the MFMA's accumulation), in a half
// block that sum's two parts by one fused multiply-add: a token's last bits depend on
// the block it falls in, as on the reduction's slices.  h goes to HBM as f32
// ([pair][moe_ff], [token][shared_ff]) and one conversion launch writes the
// down products' int8 layout; the down products go to ye [pair][n_embd] /
// ys [token][n_embd] for the combine launch, as with the tile kernels.
#include "dmoe_q4k.h"
#include "dmoe_q80.h"

#include <type_traits>

namespace dmoe {

typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int XG_WAVES = 8;
constexpr int XG_NC = 8;                                     // 16-row blocks of a unit
constexpr int XG_CHUNK = EXPERT_CHUNK * XG_NC;               // routed pairs of a unit (128)
constexpr int XG_SCHUNK = SHARED_CHUNK * XG_NC;              // shared tokens of a unit (64)
constexpr int XG_GU_ROWS = XG_WAVES * 16;                    // h rows of a gate/up item
constexpr int XG_DN_ROWS = XG_WAVES * 32;                    // n_embd rows of a down item

// A stage of the activation ring: four blocks of 32 rows.  A block's int8
// values lie in eight chunks of four rows (1 KB each, as one LDS-direct load
// writes them): row r of the block at 1024 (r / 4) + 64 (r / 8) + 256 (r % 4),
// its 16-byte unit 8 gp + 4 h + c (values as the ActI8 layout orders them) at
// slot 8 gp + 4 h + (c ^ (r % 4)).  An operand read (lane: row l % 32, h =
// l / 32, one (gp, c)) takes four rows' units from 64 bytes of each chunk, and
// the 64-byte step between chunk pairs puts the four lane quads that are
// served together on different banks.  Then the 32 rows' sums of 16 (f16) and
// scales.
constexpr int XG_ABS = 8 * 1024 + 3 * 64;                    // sums of 16: [32][16] f16
constexpr int XG_AD = XG_ABS + 1024;                         // scales: [32] f32
constexpr int XG_ABLK = XG_AD + 128;                         // one block (9,344)
constexpr int XG_AHEAD = 4;                                  // operand reads ahead of their MFMAs (divides 8)
static_assert(XG_ABLK % 16 == 0, "16-byte pieces");
static_assert(XG_GU_ROWS == EXPERT_GEMM_GU_ROWS && XG_DN_ROWS == EXPERT_GEMM_DN_ROWS, "the dispatch's item rows");

// Item k is row group k % rg_n of unit k / rg_n; a unit is shared chunk
// u < nch, else work-list entry u - nch.  Every field is wave-uniform.
struct XgItem {
    int rg, e, t_first, nt, nblk;
    bool shared, valid;
};

template <bool MERGE, int SCHUNK = XG_SCHUNK>
__device__ __forceinline__ XgItem xg_decode(const MoeJob &job, int k, int rg_n, int n_ec, int nch)
{
    XgItem I{};
    const int unit = k / rg_n;
    I.rg = k - unit * rg_n;
    I.valid = unit < n_ec + nch;
    if (!I.valid) return I;
    I.shared = unit < nch;
    if (!I.shared) {
        I.e = ldc(job.wl.ec_expert, unit - nch);
        const int c0 = ldc(job.wl.ec_chunk, unit - nch) * XG_CHUNK;
        I.t_first = ldc(job.offsets, I.e) + c0;
        I.nt = min(XG_CHUNK, ldc(job.counts, I.e) - c0);
        I.nblk = (I.nt + EXPERT_CHUNK - 1) / EXPERT_CHUNK;
    } else {
        I.e = 0;
        I.t_first = unit * SCHUNK;
        I.nt = min(SCHUNK, job.n_tokens - I.t_first);
        // MERGE: 32-token blocks (four 16-row blocks), the last one a half
        // block (two) when it holds up to 16 tokens
        I.nblk = MERGE ? 2 * ((I.nt + 15) / 16) : (I.nt + SHARED_CHUNK - 1) / SHARED_CHUNK;
    }
    return I;
}

// Activation row of row r (0..15) of 16-row block c: routed rows from the
// item's pair ids (x by token, pid / K, for gate/up; h by pair for down);
// shared items interleave the a1 / a0 digit rows (a0 rows start at N), or
// (MERGE) hold the a1 rows of 32 tokens in blocks 4 b, 4 b + 1 and their a0
// rows in blocks 4 b + 2, 4 b + 3, a last half block of up to 16 tokens the a1
// rows in block 4 b and the a0 rows in 4 b + 1.  Rows past the item's last
// repeat it.
template <bool DOWN, bool MERGE>
__device__ __forceinline__ int xg_arow(const XgItem &I, const int32_t *s_pids, int N, int K, int c, int r)
{
    if (MERGE) {
        const bool half = (c | 3) >= I.nblk;
        const int t = 32 * (c >> 2) + (half ? 0 : 16 * (c & 1)) + r, a0 = half ? c & 1 : (c >> 1) & 1;
        return I.t_first + min(t, I.nt - 1) + a0 * N;
    }
    if (I.shared) return I.t_first + min(SHARED_CHUNK * c + (r >> 1), I.nt - 1) + (r & 1) * N;
    const int p = s_pids[min(EXPERT_CHUNK * c + r, I.nt - 1)];
    return DOWN ? p : p / K;
}

// LDS-direct load of 16 bytes per active lane from a wave-uniform base plus a
// per-lane offset (lane l's bytes to LDS address lds + 16 l).  No non-temporal hint: the
// chunks of one expert read its weights through L2.
__device__ __forceinline__ void xg_lds16(const void *base, uint32_t voff, uint32_t lds)
{
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint64_t sb = (uint64_t)lo | ((uint64_t)hi << 32);
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sb), "s"(m0) : "memory", "m0");
}

// The same for 4 bytes per active lane (to lds + 4 l).
__device__ __forceinline__ void xg_lds4(const void *base, uint32_t voff, uint32_t lds)
{
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint64_t sb = (uint64_t)lo | ((uint64_t)hi << 32);
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(sb), "s"(m0) : "memory", "m0");
}

// Weight formats.  A lane holds weight row l % 32 (16-row tile (l / 16) % 2 of
// the wavefront's two) and the values of lane groups g = h and 2 + h (h = l /
// 32) of a super-block.  Each gives:
//   TILE, TLDS, WLOADS   bytes of a 16-row tile's super-block in HBM, its
//                        stride in LDS
//   ASTAGES, ALOADS      activation stages; loads of a 16-row block
//   MIN                  a min term on the sums of 16
//   PER32                scales per 32 values (the products are XgQ80's)
//   Raw, read, pin       the lane's bytes of a super-block, from LDS; in
//                        registers from there on
//   Ops, fold            the int8 operands: hi and lo digits of scale x quant,
//                        chunk c of lane group 2 gp + h at [4 gp + c]
struct XgQ4K {
    static constexpr int TILE = TILE_BYTES, TLDS = TILE_BYTES, ASTAGES = 3, ALOADS = 6;
    static constexpr bool MIN = true, PER32 = false;
    struct Raw {
        uint4 h, q[4];
    };
    // bm: the min-term operand (m of the lane's eight sums of 16: sub-blocks
    // 4 h .. 4 h + 3, twice each); d, dmin: the row's scales
    struct Ops {
        v4i hi[8], lo[8];
        h8 bm;
        float d, dmin;
    };
    __device__ static void read(Raw &t, const uint8_t *tile, int r16, int h)
    {
        const uint4 *p = reinterpret_cast<const uint4 *>(tile);
        t.h = p[r16];
#pragma unroll
        for (int gp = 0; gp < 2; gp++) {
            t.q[2 * gp] = p[(1 + 2 * (2 * gp + h)) * 16 + r16];
            t.q[2 * gp + 1] = p[(2 + 2 * (2 * gp + h)) * 16 + r16];
        }
    }
    __device__ static void pin(Raw &t)
    {
        asm volatile("" : "+v"(t.h.x), "+v"(t.h.y), "+v"(t.h.z), "+v"(t.h.w));
#pragma unroll
        for (int i = 0; i < 4; i++)
            asm volatile("" : "+v"(t.q[i].x), "+v"(t.q[i].y), "+v"(t.q[i].z), "+v"(t.q[i].w));
    }
    // sc = 8 sh + sl: hi = sh q, lo = sl q
    __device__ static void fold(const Raw &t, int h, Ops &f)
    {
        typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
        // scale j: 6 bits at 6j of dword y (j < 5), at 6 (j - 5) of dword z
        uint32_t sh[8], sl[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t src = j < 5 ? t.h.y : t.h.z;
            const uint32_t off = j < 5 ? 6u * j : 6u * (j - 5);
            sl[j] = bfe(src, off, 3);
            sh[j] = bfe(src, off + 3, 3);
        }
        // byte-wise products by a scale below 8: each byte stays below 128, so
        // a 16-bit lane product carries nothing across its two bytes
        auto mul = [](uint32_t v, uint32_t s) -> int {
            const u16x2 a = __builtin_bit_cast(u16x2, v);
            const u16x2 b = {(unsigned short)s, (unsigned short)s};
            return __builtin_bit_cast(int, (u16x2)(a * b));
        };
#pragma unroll
        for (int gp = 0; gp < 2; gp++) {
            const uint4 q0 = t.q[2 * gp], q1 = t.q[2 * gp + 1];
            const uint32_t w[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t l0 = w[2 * c] & 0x0F0F0F0Fu, l1 = w[2 * c + 1] & 0x0F0F0F0Fu;
                const uint32_t h0 = (w[2 * c] >> 4) & 0x0F0F0F0Fu, h1 = (w[2 * c + 1] >> 4) & 0x0F0F0F0Fu;
                f.hi[4 * gp + c] =
                    (v4i){mul(l0, sh[2 * c]), mul(l1, sh[2 * c]), mul(h0, sh[2 * c + 1]), mul(h1, sh[2 * c + 1])};
                f.lo[4 * gp + c] =
                    (v4i){mul(l0, sl[2 * c]), mul(l1, sl[2 * c]), mul(h0, sl[2 * c + 1]), mul(h1, sl[2 * c + 1])};
            }
        }
        // mins: m0 m1 at 18, 24 of dword z, m2 .. m6 at 0, 6, .. of dword w, m7 in
        // bits 30..31 of the three dwords
        const uint32_t m7 = (t.h.y >> 30) | ((t.h.z >> 30) << 2) | ((t.h.w >> 30) << 4);
        const uint32_t mm[4] = {h ? bfe(t.h.w, 12, 6) : bfe(t.h.z, 18, 6), h ? bfe(t.h.w, 18, 6) : bfe(t.h.z, 24, 6),
                                h ? bfe(t.h.w, 24, 6) : bfe(t.h.w, 0, 6), h ? m7 : bfe(t.h.w, 6, 6)};
#pragma unroll
        for (int i = 0; i < 4; i++) f.bm[2 * i] = f.bm[2 * i + 1] = (_Float16)(float)mm[i];
        f.d = h16f(t.h.x & 0xffffu);
        f.dmin = h16f(t.h.x >> 16);
        // (as an f32 operand: folded into v_fma_mix_f32 the epilogue's min term
        // issues at half the rate of v_fmac_f32)
        asm volatile("" : "+v"(f.dmin));
    }
};

// Q6_K (tiled by k_tile_q6k): p = sc (q - 32), |p| <= 4096, as two digits p =
// 256 hi + lo, lo in [-128, 127]; no min term, so no sums of 16.  With 256 the
// ratio of both the weight's and the activation's digits, the two middle
// products share one sum.  The fold (16-bit products, their bytes gathered by
// v_perm) is 450 instructions, what the 64 MFMAs of 64 tokens leave room for.
// Measured against the few-token kernel in chunks of 32 tokens, which reads
// and unpacks the matrix once per chunk: LM head of 157,184 rows at 256 tokens
// 1,679 -> 884 us, at 40 tokens 316 -> 218; dense MLP of 200 tokens 494 -> 150
// us, of 40 tokens 120 -> 109.
struct XgQ6K {
    static constexpr int TILE = 16 * Q6K_BYTES, TLDS = 14 * 256, ASTAGES = 2, ALOADS = 5;
    static constexpr bool MIN = false, PER32 = false;
    struct Raw {
        uint4 q[6], sc;                  // L[0..3], L[4..7], H[0..3] of both lane groups; scales
        uint32_t d;
    };
    struct Ops {
        v4i hi[8], lo[8];
        float d;
    };
    __device__ static void read(Raw &t, const uint8_t *tile, int r16, int h)
    {
        const uint4 *p = reinterpret_cast<const uint4 *>(tile);
#pragma unroll
        for (int gp = 0; gp < 2; gp++)
#pragma unroll
            for (int k = 0; k < 3; k++) t.q[3 * gp + k] = p[64 * k + 16 * (2 * gp + h) + r16];
        t.sc = p[192 + r16];
        t.d = reinterpret_cast<const uint16_t *>(tile + 208 * 16)[r16];
    }
    __device__ static void pin(Raw &t)
    {
        asm volatile("" : "+v"(t.sc.x), "+v"(t.sc.y), "+v"(t.sc.z), "+v"(t.sc.w), "+v"(t.d));
#pragma unroll
        for (int i = 0; i < 6; i++)
            asm volatile("" : "+v"(t.q[i].x), "+v"(t.q[i].y), "+v"(t.q[i].z), "+v"(t.q[i].w));
    }
    __device__ static void fold(const Raw &t, int, Ops &f)
    {
        typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
        const uint32_t scw[4] = {t.sc.x, t.sc.y, t.sc.z, t.sc.w};
        f.d = h16f(t.d);
#pragma unroll
        for (int gp = 0; gp < 2; gp++) {
            const uint4 la = t.q[3 * gp], lb = t.q[3 * gp + 1], hh = t.q[3 * gp + 2];
            const uint32_t L[8] = {la.x, la.y, la.z, la.w, lb.x, lb.y, lb.z, lb.w};
            const uint32_t Hb[4] = {hh.x, hh.y, hh.z, hh.w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                // four dwords of four quants 0..63: sub-block 2c, then 2c + 1
                const uint32_t e[4] = {(L[2 * c] & 0x0F0F0F0Fu) | ((Hb[c] << 4) & 0x30303030u),
                                       ((L[2 * c] >> 4) & 0x0F0F0F0Fu) | ((Hb[c] << 2) & 0x30303030u),
                                       (L[2 * c + 1] & 0x0F0F0F0Fu) | (Hb[c] & 0x30303030u),
                                       ((L[2 * c + 1] >> 4) & 0x0F0F0F0Fu) | ((Hb[c] >> 2) & 0x30303030u)};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    // 32 j + 8 g .. lies in the sub-block of 16 number 2 j + g / 2
                    const int k = 2 * (2 * c + (i >> 1)) + gp;
                    const int sc = (int)(scw[k >> 2] << (24 - 8 * (k & 3))) >> 24;
                    const u16x2 s2 = {(unsigned short)sc, (unsigned short)sc};
                    const unsigned short m = (unsigned short)(128 - 32 * sc);
                    const u16x2 m2 = {m, m};
                    // p + 128 of bytes 0, 2 and of bytes 1, 3 in 16-bit lanes
                    const uint32_t pe = __builtin_bit_cast(
                        uint32_t, (u16x2)(__builtin_bit_cast(u16x2, e[i] & 0x00FF00FFu) * s2 + m2));
                    const uint32_t po = __builtin_bit_cast(
                        uint32_t, (u16x2)(__builtin_bit_cast(u16x2, (e[i] >> 8) & 0x00FF00FFu) * s2 + m2));
                    f.hi[4 * gp + c][i] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
                    f.lo[4 * gp + c][i] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
                }
            }
        }
    }
};

// Q8_0 (tiled by launch_tile_q80, ACT_SPLIT32 activations), projections only:
// the quants are the int8 operands as they lie, and a v_mfma_i32_32x32x32_i8 is
// one 32-value block, so a token's output takes, per block, S = 256 S1 + S0 of
// its two digit rows and one fused multiply-add of S by d_w d_x: four VALU
// instructions per output and block, which bound it (64 MFMAs of 32 cycles
// against 1,024 VALU instructions per wavefront and 64 tokens).  The block's
// operand of a lane is the eight bytes of lane groups 2 h and 2 h + 1.
// Measured against the expert kernel's items of 8 tokens (each tile read and
// its three instructions per digit row and block repeated for every 8):
// attention half of 200 tokens 180 -> 113 us, of 2,048 tokens 1,386 -> 668.
struct XgQ80 {
    static constexpr int TILE = Q80_TILE, TLDS = Q80_TILE, ASTAGES = 2, ALOADS = 6;
    static constexpr bool MIN = false, PER32 = true;
    struct Raw {
        v4i w[8];
        uint4 d;                         // the row's eight f16 scales
    };
    struct Ops {
        v4i w[8];
        float d[8];
    };
    __device__ static void read(Raw &t, const uint8_t *tile, int r16, int h)
    {
        const uint8_t *p = tile + r16 * 16;
        t.d = *reinterpret_cast<const uint4 *>(p);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint8_t *q = p + (1 + 8 * h + (j >> 1)) * 256 + 8 * (j & 1);
            const uint2 a = *reinterpret_cast<const uint2 *>(q), b = *reinterpret_cast<const uint2 *>(q + 1024);
            t.w[j] = (v4i){(int)a.x, (int)a.y, (int)b.x, (int)b.y};
        }
    }
    __device__ static void pin(Raw &t)
    {
        asm volatile("" : "+v"(t.d.x), "+v"(t.d.y), "+v"(t.d.z), "+v"(t.d.w));
#pragma unroll
        for (int j = 0; j < 8; j++) asm volatile("" : "+v"(t.w[j]));
    }
    __device__ static void fold(const Raw &t, int, Ops &f)
    {
        const uint32_t dw[4] = {t.d.x, t.d.y, t.d.z, t.d.w};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            f.w[j] = t.w[j];
            f.d[j] = h16f(j & 1 ? dw[j >> 1] >> 16 : dw[j >> 1] & 0xffffu);
        }
    }
};

// FEW: units of 32 tokens (MERGE), whose smaller activation stages leave room
// for two stages of weights: with few tokens a step lasts no longer than a CU's
// weights take to arrive, and one stage, refilled only while a step's products
// run, stalls it (LM head of Q6_K, 157,184 x 4,096, at 32 tokens: 190 us with
// one stage, 177 with two; the fold is the larger part of what is left).
// (Measured and not kept: the same for the routed Q4_K experts, units of 64
// pairs, from 256 tokens: 292 us against 269 on the tile kernels.)
template <class F, bool DOWN, bool MERGE, bool FEW = false>
__global__ __launch_bounds__(XG_WAVES * 64) void k_gemm_q(MoeJob job)
{
    static_assert(!FEW || (MERGE && F::ASTAGES == 2), "weight stages beside two activation stages");
    constexpr int NC = FEW ? XG_NC / 2 : XG_NC, SCHUNK = FEW ? XG_SCHUNK / 2 : XG_SCHUNK;
    constexpr int NBMAX = MERGE ? NC / 4 : NC / 2;         // 32-row (MERGE: 32-token) blocks of a unit
    constexpr int XG_ASTAGE = (NC / 2) * XG_ABLK;          // bytes of an activation stage
    constexpr int WST = FEW ? 2 : 1;                       // weight stages
    constexpr int WLOADS = 2 * ((F::TILE + 1023) / 1024);  // loads of a weight stage
    __shared__ __align__(16) uint8_t SA[F::ASTAGES][XG_ASTAGE];
    __shared__ __align__(16) uint8_t SW[XG_WAVES][WST][2 * F::TLDS];
    // pair ids of the routed items i, i + 1 (its activations load during
    // item i) and i + 2 (read from perm during item i, written at its end)
    __shared__ int32_t s_pids[3][XG_CHUNK];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, r32 = lane & 31, h = lane >> 5;
    const int H = job.H, FF = job.FF, N = job.n_tokens, K = job.top_k;
    const int n_ec = job.wl.n_ec ? ldc(job.wl.n_ec, 0) : 0;   // none: shared units only
    const int nch = job.has_shared ? (N + SCHUNK - 1) / SCHUNK : 0;
    const int rg_n = DOWN ? H / XG_DN_ROWS : FF / XG_GU_ROWS;
    const int Kin = DOWN ? FF : H;
    // down launches of a projection split the reduction into KS slices of
    // `steps` super-blocks (item k: slice k % KS of item k / KS)
    const int KS = DOWN && job.ks > 1 ? job.ks : 1;
    const int nsb = Kin / 256, steps = nsb / KS;     // >= 2
    const int G = gridDim.x;

    int k = schedule_item(blockIdx.x, G, 0), round = 0;
    XgItem I = xg_decode<MERGE, SCHUNK>(job, k / KS, rg_n, n_ec, nch);
    if (!I.valid) return;
    int slice = k % KS;
    k = schedule_item(blockIdx.x, G, 1);
    XgItem NI = xg_decode<MERGE, SCHUNK>(job, k / KS, rg_n, n_ec, nch);
    int nslice = k % KS;
    if (tid < XG_CHUNK && !I.shared) s_pids[0][tid] = job.perm[I.t_first + min(tid, I.nt - 1)];
    if (tid < XG_CHUNK && NI.valid && !NI.shared) s_pids[1][tid] = job.perm[NI.t_first + min(tid, NI.nt - 1)];
    __syncthreads();

    // Load cursors, across items: the weights run one step ahead of the
    // products, the activations two.  Wave-uniform bases; wavefront w loads
    // 16-row block w of the items that have it, by this lane's byte offsets
    // (32-bit: the host keeps every activation array below 2 GiB).
    const uint32_t sw0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&SW[wave][0][0];
    const uint32_t sa = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&SA[0][0];
    const uint8_t *wb0 = nullptr, *wb1 = nullptr;
    const uint8_t *aqb = nullptr, *absb = nullptr, *adb = nullptr;
    uint32_t aqo[4] = {0, 0, 0, 0}, abso = 0, ado = 0;
    bool act_on = false;
    // (slice cs of an item starts at super-block cs * steps of every row)
    auto weights_of = [&](const XgItem &C, int cs) {
        if (!DOWN) {
            const WTensor &a = C.shared ? job.sg : job.eg;
            const WTensor &b = C.shared ? job.su : job.eu;
            const int t16 = C.rg * (XG_GU_ROWS / 16) + wave;
            wb0 = a.data + (size_t)C.e * a.nb2 + (size_t)t16 * nsb * F::TILE;
            wb1 = b.data + (size_t)C.e * b.nb2 + (size_t)t16 * nsb * F::TILE;
        } else {
            const WTensor &W = C.shared ? job.sd : job.ed;
            const int t16 = C.rg * (XG_DN_ROWS / 16) + 2 * wave;
            wb0 = W.data + (size_t)C.e * W.nb2 + ((size_t)t16 * nsb + cs * steps) * F::TILE;
            wb1 = wb0 + (size_t)nsb * F::TILE;
        }
    };
    auto acts_of = [&](const XgItem &C, int cs, const int32_t *pids) {
        act_on = wave < C.nblk;
        if (!act_on) return;
        const int sb0 = cs * steps;
        const ActI8 &A = DOWN ? (C.shared ? job.ahs : job.ah) : (C.shared ? job.axs : job.ax);
        aqb = reinterpret_cast<const uint8_t *>(A.q) + (size_t)sb0 * 256;
        absb = reinterpret_cast<const uint8_t *>(A.bs) + (size_t)sb0 * 32;
        adb = reinterpret_cast<const uint8_t *>(A.d) + (size_t)sb0 * (F::PER32 ? 32 : 4);
        // (the lane through an empty asm: its rows and units are formed here,
        // once per item, and not held in registers across the steps)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int u = ((ln & 15) ^ (ln >> 4)) * 16;
#pragma unroll
        for (int j = 0; j < 4; j++)
            aqo[j] = (uint32_t)xg_arow<DOWN, MERGE>(C, pids, N, K, wave, 4 * j + (ln >> 4)) * (uint32_t)Kin + u;
        abso = ((uint32_t)xg_arow<DOWN, MERGE>(C, pids, N, K, wave, (ln >> 1) & 15) * (uint32_t)(Kin / 16) + (ln & 1) * 8) * 2;
        ado = (uint32_t)xg_arow<DOWN, MERGE>(C, pids, N, K, wave, ln & 15) * (uint32_t)(Kin / 256);
        ado = F::PER32 ? (8 * ado + (ln >> 4)) * 4 : 4 * ado;
    };
    // the weight cursor's super-block to the wavefront's stage ws; on to the next
    auto issue_w = [&](int ws) {
        constexpr int FULL = F::TILE / 1024, REST = (F::TILE % 1024) / 16;
        const uint32_t vo = (uint32_t)lane * 16, sw = sw0 + ws * (2 * F::TLDS);
#pragma unroll
        for (int i = 0; i < FULL; i++) {
            xg_lds16(wb0, vo + 1024 * i, sw + 1024 * i);
            xg_lds16(wb1, vo + 1024 * i, sw + F::TLDS + 1024 * i);
        }
        if (lane < REST) {
            xg_lds16(wb0, vo + 1024 * FULL, sw + 1024 * FULL);
            xg_lds16(wb1, vo + 1024 * FULL, sw + F::TLDS + 1024 * FULL);
        }
        wb0 += F::TILE;
        wb1 += F::TILE;
    };
    // the activation cursor's super-block to ring stage st (F::ALOADS loads of
    // a wavefront that has a block); on to the next
    auto issue_a = [&](int st) {
        if (!act_on) return;
        const uint32_t blk = sa + st * XG_ASTAGE + (wave >> 1) * XG_ABLK;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int q = 4 * (wave & 1) + j;         // chunk of four rows
            xg_lds16(aqb, aqo[j], blk + 1024 * q + 64 * (q >> 1));
        }
        if (F::MIN && lane < 32) xg_lds16(absb, abso, blk + XG_ABS + 512 * (wave & 1));
        if (F::PER32) {
            // scales [8 blocks][16 rows], four blocks a load, in place of the sums
            xg_lds4(adb, ado, blk + XG_ABS + 512 * (wave & 1));
            xg_lds4(adb + 16, ado, blk + XG_ABS + 512 * (wave & 1) + 256);
        } else if (lane < 16) {
            xg_lds4(adb, ado, blk + XG_AD + 64 * (wave & 1));
        }
        aqb += 256;
        absb += 32;
        adb += F::PER32 ? 32 : 4;
    };
    // this lane's operand addresses in a stage: row r32, unit 8 gp + 4 h + c
    // (c's swizzle in the address, gp 128 bytes on); PER32: units 8 h + c and,
    // 64 bytes on, 8 h + 4 + c
    uint32_t ao[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        ao[c] = 1024 * (r32 >> 2) + 64 * (r32 >> 3) + 256 * (r32 & 3) + (F::PER32 ? 128 : 64) * h + 16 * (c ^ (r32 & 3));
    const uint8_t *wrd = &SW[wave][0][((lane >> 4) & 1) * F::TLDS];

    weights_of(I, slice);
    acts_of(I, slice, s_pids[0]);
    issue_w(0);
    issue_a(0);
    if (F::ASTAGES == 3) issue_a(1);                  // steps >= 2
    if (FEW) issue_w(1);
    int wst = 0;                                      // the weight stage the step reads
    bool w_ahead = FEW;                               // weight loads issued after this step's activations
    int stg = 0;                                      // the stage the products read
    bool ahead = act_on;                              // activation loads issued after this step's weights
    int pb = 0;                                       // pair list of item I (of 3)

    for (;;) {
        const int pb1 = pb == 2 ? 0 : pb + 1, pb2 = pb1 == 2 ? 0 : pb1 + 1;
        k = schedule_item(blockIdx.x, G, round + 2);
        const XgItem NNI = xg_decode<MERGE, SCHUNK>(job, k / KS, rg_n, n_ec, nch);
        int npid = 0;
        if (tid < XG_CHUNK && NNI.valid && !NNI.shared) npid = job.perm[NNI.t_first + min(tid, NNI.nt - 1)];

        v16f acc[NBMAX];
#pragma unroll
        for (int c = 0; c < NBMAX; c++) acc[c] = (v16f)(0.0f);

        // NB: the item's 32-row (MERGE: 32-token) blocks; HALF: a half block
        // after them
        auto run = [&](auto nb_c, auto half_c) __attribute__((always_inline)) {
            constexpr int NB = decltype(nb_c)::value;
            constexpr bool HALF = decltype(half_c)::value;
            static_assert(NB + HALF <= NBMAX, "the accumulators of a unit");
            for (int s = 0; s < steps; s++) {
                // this step's weights (this wavefront's) and activations
                // (every wavefront's) have landed, the stage two steps on has
                // been read by all
                if (FEW && w_ahead)
                    EXPERT_WAIT_VM(WLOADS);
                else if (F::ASTAGES == 3 && ahead)
                    EXPERT_WAIT_VM(F::ALOADS);
                else
                    EXPERT_WAIT_VM(0);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                typename F::Raw t;
                F::read(t, wrd + wst * (2 * F::TLDS), r16, h);
                F::pin(t);                            // the stage may be refilled
                // the stage the activations of step s + LEAD go to
                constexpr int LEAD = F::ASTAGES - 1;
                const int st2 = stg == 0 ? LEAD : stg - 1;
                auto next_w = [&]() {
                    w_ahead = s + WST < steps || NI.valid;
                    if (!w_ahead) return;
                    if (s + WST == steps) weights_of(NI, nslice);
                    issue_w(wst);
                };
                auto next_a = [&]() {
                    ahead = false;
                    if (s + LEAD >= steps && !NI.valid) return;
                    if (s + LEAD == steps) acts_of(NI, nslice, s_pids[pb1]);
                    issue_a(st2);
                    ahead = act_on;
                };
                // (the loads a wait leaves in flight are the last issued)
                if (FEW) next_a();
                next_w();
                if (!FEW) next_a();
                if (FEW) wst ^= 1;
                typename F::Ops f;
                F::fold(t, h, f);
                // The blocks' products.  The operand reads run XG_AHEAD ahead
                // of their MFMAs (the next block's first ones go out before
                // this block's epilogue); the scheduling barriers keep that
                // order, which the compiler otherwise undoes to save registers.
                const uint8_t *st = &SA[0][0] + stg * XG_ASTAGE;
                auto read_a = [&](int b, int i) __attribute__((always_inline)) -> v4i {
                    return *reinterpret_cast<const v4i *>(st + b * XG_ABLK + ao[i & 3] + 128 * (i >> 2));
                };
                if constexpr (F::PER32) {
                    static_assert(!F::PER32 || (MERGE && DOWN), "Q8_0: projections");
                    // block b's operand of 32-value block j
                    auto read_q = [&](int b, int j) __attribute__((always_inline)) -> v4i {
                        const uint8_t *q = st + b * XG_ABLK + ao[j >> 1] + 8 * (j & 1);
                        const uint2 u = *reinterpret_cast<const uint2 *>(q), v = *reinterpret_cast<const uint2 *>(q + 64);
                        return (v4i){(int)u.x, (int)u.y, (int)v.x, (int)v.y};
                    };
                    // scales of block j, activation rows 8 i + 4 h .. + 3
                    auto read_dx = [&](int b, int j, int i) __attribute__((always_inline)) -> f4 {
                        return *reinterpret_cast<const f4 *>(st + b * XG_ABLK + XG_ABS + 512 * (i >> 1) + 64 * j +
                                                             32 * (i & 1) + 16 * h);
                    };
                    // (token block, 32-value block) n = 8 c + j: the next pair's
                    // MFMAs go out before this pair's scale products
                    constexpr int T = 8 * NB;
                    if constexpr (NB > 0) {
                        v4i x1[2], x0[2];
                        v16i p1[2], p0[2];
                        x1[0] = read_q(0, 0);
                        x0[0] = read_q(1, 0);
                        x1[1] = read_q(0, 1);
                        x0[1] = read_q(1, 1);
                        p1[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x1[0], f.w[0], (v16i)(0), 0, 0, 0);
                        p0[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0[0], f.w[0], (v16i)(0), 0, 0, 0);
#pragma unroll
                        for (int n = 0; n < T; n++) {
                            const int c = n >> 3, j = n & 7, u = n & 1;
                            __builtin_amdgcn_sched_barrier(0);
                            f4 dx[4];
#pragma unroll
                            for (int i = 0; i < 4; i++) dx[i] = read_dx(2 * c + 1, j, i);
                            if (n + 2 < T) {
                                x1[u] = read_q(2 * ((n + 2) >> 3), (n + 2) & 7);
                                x0[u] = read_q(2 * ((n + 2) >> 3) + 1, (n + 2) & 7);
                            }
                            if (n + 1 < T) {
                                p1[u ^ 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x1[u ^ 1], f.w[(n + 1) & 7], (v16i)(0), 0, 0, 0);
                                p0[u ^ 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0[u ^ 1], f.w[(n + 1) & 7], (v16i)(0), 0, 0, 0);
                            }
#pragma unroll
                            for (int i = 0; i < 16; i++)
                                acc[c][i] = __builtin_fmaf((float)(256 * p1[u][i] + p0[u][i]), f.d[j] * dx[i >> 2][i & 3], acc[c][i]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if constexpr (HALF) {
                        v4i x[2];
                        v16i p[2];
                        x[0] = read_q(2 * NB, 0);
                        x[1] = read_q(2 * NB, 1);
                        p[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[0], f.w[0], (v16i)(0), 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const int u = j & 1;
                            __builtin_amdgcn_sched_barrier(0);
                            const f4 dx[2] = {read_dx(2 * NB, j, 2), read_dx(2 * NB, j, 3)};
                            if (j + 2 < 8) x[u] = read_q(2 * NB, j + 2);
                            if (j + 1 < 8)
                                p[u ^ 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[u ^ 1], f.w[(j + 1) & 7], (v16i)(0), 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 8; i++)
                                acc[NB][i] = __builtin_fmaf((float)(256 * p[u][i] + p[u][i + 8]), f.d[j] * dx[i >> 2][i & 3], acc[NB][i]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else if constexpr (MERGE) {
                    // block c: 32 tokens, their a1 rows in stage block 2 c, a0
                    // rows in 2 c + 1; the four digit products of a chunk, then
                    // one epilogue per token
                    v4i a1[XG_AHEAD / 2], a0[XG_AHEAD / 2];
                    if (NB)
#pragma unroll
                        for (int i = 0; i < XG_AHEAD / 2; i++) {
                            a1[i] = read_a(0, i);
                            a0[i] = read_a(1, i);
                        }
#pragma unroll
                    for (int c = 0; c < NB; c++) {
                        const uint8_t *ab1 = st + 2 * c * XG_ABLK, *ab0 = ab1 + XG_ABLK;
                        v16i p11 = (v16i)(0), p10 = (v16i)(0), p01 = (v16i)(0), p00 = (v16i)(0);
                        v16f s2 = (v16f)(0.0f);
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            __builtin_amdgcn_sched_barrier(0);
                            const v4i x1 = a1[i % (XG_AHEAD / 2)], x0 = a0[i % (XG_AHEAD / 2)];
                            p11 = __builtin_amdgcn_mfma_i32_32x32x32_i8(x1, f.hi[i], p11, 0, 0, 0);
                            p10 = __builtin_amdgcn_mfma_i32_32x32x32_i8(x1, f.lo[i], p10, 0, 0, 0);
                            p00 = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0, f.lo[i], p00, 0, 0, 0);
                            if (F::MIN)
                                p01 = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0, f.hi[i], p01, 0, 0, 0);
                            else                      // both weigh 256
                                p10 = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0, f.hi[i], p10, 0, 0, 0);
                            const int n = 8 * c + i + XG_AHEAD / 2;
                            if (n < 8 * NB) {
                                a1[i % (XG_AHEAD / 2)] = read_a(2 * (n >> 3), n & 7);
                                a0[i % (XG_AHEAD / 2)] = read_a(2 * (n >> 3) + 1, n & 7);
                            }
                            if constexpr (F::MIN)
                                if (i == 6) {
                                    // sums of 16: 256 (a1 sums) + (a0 sums), the
                                    // factor on the operand (m <= 63: exact
                                    // there; the f32 sum may round)
                                    const h8 s1 = *reinterpret_cast<const h8 *>(ab1 + XG_ABS + r32 * 32 + 16 * h);
                                    const h8 s0 = *reinterpret_cast<const h8 *>(ab0 + XG_ABS + r32 * 32 + 16 * h);
                                    s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(s1, f.bm * (_Float16)256.0f, s2, 0, 0, 0);
                                    s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(s0, f.bm, s2, 0, 0, 0);
                                }
                        }
                        // (the a0 row's scale; the a1 row's is 256 times it)
                        f4 dx = *reinterpret_cast<const f4 *>(ab0 + XG_AD + 16 * h);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            f4 nx = dx;
                            __builtin_amdgcn_sched_barrier(0);
                            if (j < 3) nx = *reinterpret_cast<const f4 *>(ab0 + XG_AD + 32 * (j + 1) + 16 * h);
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                const int i = 4 * j + k;
                                if constexpr (F::MIN) {
                                    const int t1 = 8 * p11[i] + p10[i], t0 = 8 * p01[i] + p00[i];
                                    const float S = __builtin_fmaf((float)t1, 256.0f, (float)t0);
                                    acc[c][i] = q4k_epi(acc[c][i], dx[k], f.d, S, f.dmin, s2[i]);
                                } else {
                                    const float S = __builtin_fmaf((float)(256 * p11[i] + p10[i]), 256.0f, (float)p00[i]);
                                    acc[c][i] = __builtin_fmaf(dx[k], f.d * S, acc[c][i]);
                                }
                            }
                            dx = nx;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if constexpr (HALF) {
                        // stage block 2 NB: a1 rows 0..15, a0 rows 16..31 of up to
                        // 16 tokens; a lane's rows i and i + 8 are the two digits
                        // of one token
                        const uint8_t *ab = st + 2 * NB * XG_ABLK;
                        v4i ah[XG_AHEAD];
#pragma unroll
                        for (int i = 0; i < XG_AHEAD; i++) ah[i] = read_a(2 * NB, i);
                        v16i ph = (v16i)(0), pl = (v16i)(0);
                        v16f s2 = (v16f)(0.0f);
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            __builtin_amdgcn_sched_barrier(0);
                            const v4i x = ah[i % XG_AHEAD];
                            ph = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, f.hi[i], ph, 0, 0, 0);
                            pl = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, f.lo[i], pl, 0, 0, 0);
                            if (i + XG_AHEAD < 8) ah[i % XG_AHEAD] = read_a(2 * NB, i + XG_AHEAD);
                            if constexpr (F::MIN)
                                if (i == 6) {
                                    const h8 sm = *reinterpret_cast<const h8 *>(ab + XG_ABS + r32 * 32 + 16 * h);
                                    s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm, f.bm, s2, 0, 0, 0);
                                }
                        }
                        const f4 dx[2] = {*reinterpret_cast<const f4 *>(ab + XG_AD + 64 + 16 * h),
                                          *reinterpret_cast<const f4 *>(ab + XG_AD + 96 + 16 * h)};
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            float o = acc[NB][i];
                            if constexpr (F::MIN) {
                                const int t1 = 8 * ph[i] + pl[i], t0 = 8 * ph[i + 8] + pl[i + 8];
                                const float S = __builtin_fmaf((float)t1, 256.0f, (float)t0);
                                o = q4k_epi(o, dx[i >> 2][i & 3], f.d, S, f.dmin,
                                            __builtin_fmaf(s2[i], 256.0f, s2[i + 8]));
                            } else {
                                const int t1 = 256 * ph[i] + pl[i] + ph[i + 8];
                                const float S = __builtin_fmaf((float)t1, 256.0f, (float)pl[i + 8]);
                                o = __builtin_fmaf(dx[i >> 2][i & 3], f.d * S, o);
                            }
                            acc[NB][i] = o;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    v4i a[XG_AHEAD];
#pragma unroll
                    for (int i = 0; i < XG_AHEAD; i++) a[i] = read_a(i >> 3, i & 7);
#pragma unroll
                    for (int c = 0; c < NB; c++) {
                        const uint8_t *ab = st + c * XG_ABLK;
                        const h8 as = *reinterpret_cast<const h8 *>(ab + XG_ABS + r32 * 32 + 16 * h);
                        v16i sh = (v16i)(0), sl = (v16i)(0);
                        v16f s2;
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            __builtin_amdgcn_sched_barrier(0);
                            const v4i ai = a[i % XG_AHEAD];
                            sh = __builtin_amdgcn_mfma_i32_32x32x32_i8(ai, f.hi[i], sh, 0, 0, 0);
                            sl = __builtin_amdgcn_mfma_i32_32x32x32_i8(ai, f.lo[i], sl, 0, 0, 0);
                            const int n = 8 * c + i + XG_AHEAD;
                            if (n < 8 * NB) a[i % XG_AHEAD] = read_a(n >> 3, n & 7);
                            if (i == 6) s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(as, f.bm, (v16f)(0.0f), 0, 0, 0);
                        }
                        // lane: weight row r32, activation rows 8 j + 4 h + i
                        f4 dx = *reinterpret_cast<const f4 *>(ab + XG_AD + 16 * h);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            f4 nx = dx;
                            __builtin_amdgcn_sched_barrier(0);
                            if (j < 3) nx = *reinterpret_cast<const f4 *>(ab + XG_AD + 32 * (j + 1) + 16 * h);
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                const int isum = 8 * sh[4 * j + i] + sl[4 * j + i];
                                acc[c][4 * j + i] = q4k_epi(acc[c][4 * j + i], dx[i], f.d, (float)isum, f.dmin, s2[4 * j + i]);
                            }
                            dx = nx;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                stg = stg == LEAD ? 0 : stg + 1;
            }
        };
        typedef std::integral_constant<int, 0> zero;
        typedef std::integral_constant<int, 1> one;
        if constexpr (FEW) {
            // (32 tokens at most: half a block or a whole one)
            if (I.nblk >> 1 == 1)
                run(zero(), one());
            else
                run(one(), zero());
        } else if constexpr (MERGE) {
            switch (I.nblk >> 1) {
            case 1: run(zero(), one()); break;
            case 2: run(one(), zero()); break;
            case 3: run(one(), one()); break;
            default: run(std::integral_constant<int, 2>(), zero()); break;
            }
        } else {
            switch ((I.nblk + 1) >> 1) {
            case 1: run(one(), zero()); break;
            case 2: run(std::integral_constant<int, 2>(), zero()); break;
            case 3: run(std::integral_constant<int, 3>(), zero()); break;
            default: run(std::integral_constant<int, 4>(), zero()); break;
            }
        }

        // Results.  Lane: weight row r32; activation rows (MERGE: tokens) 32 c +
        // 8 j + 4 h + i, i < 4 (shared: the digits of token 16 c + 4 j + 2 h + i / 2).
        // (the lane's row goes through an empty asm, so that the compiler does
        // not hold every row's index in registers across the steps)
        const int32_t *pids = s_pids[pb];
        int hr = h, odd = (lane >> 4) & 1;
        asm volatile("" : "+v"(hr), "+v"(odd));
        if (!DOWN) {
            // h = silu(gate) * up, f32.  Lanes 0..15 of each 32 hold gate row
            // r16, lanes 16..31 up row r16: v_permlane16_swap of rows (a, b)
            // leaves gate of a (lanes 0..15) and of b (16..31) in the first,
            // up of both in the second
            const int col = I.rg * XG_GU_ROWS + 16 * wave + r16;
            auto swap = [](float &a, float &b) {
                const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a),
                                                                __builtin_bit_cast(unsigned, b), false, false);
                const unsigned r0 = r[0], r1 = r[1];
                a = __builtin_bit_cast(float, r0);
                b = __builtin_bit_cast(float, r1);
            };
#pragma unroll
            for (int c = 0; c < NBMAX; c++) {
                if ((MERGE ? 4 : 2) * c >= I.nblk) continue;
                if (MERGE || !I.shared) {
#pragma unroll
                    for (int i = 0; i < 16; i += 2) {
                        float a = acc[c][i], b = acc[c][i + 1];
                        swap(a, b);
                        const int q = 32 * c + 8 * (i >> 2) + 4 * hr + (i & 3) + odd;
                        if (q >= I.nt) continue;
                        float *o = MERGE ? job.hs + (size_t)(I.t_first + q) * job.SF : job.h + (size_t)pids[q] * FF;
                        o[col] = silu(a) * b;
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 16; i += 4) {
                        float a = acc[c][i] + acc[c][i + 1], b = acc[c][i + 2] + acc[c][i + 3];
                        swap(a, b);
                        const int q = 16 * c + i + 2 * hr + odd;
                        if (q < I.nt) job.hs[(size_t)(I.t_first + q) * job.SF + col] = silu(a) * b;
                    }
                }
            }
        } else {
            const int row = I.rg * XG_DN_ROWS + 32 * wave + r32;
            float *out = I.shared ? job.ys + (size_t)slice * N * H : job.ye;
#pragma unroll
            for (int c = 0; c < NBMAX; c++) {
                if ((MERGE ? 4 : 2) * c >= I.nblk) continue;
                if (MERGE || !I.shared) {
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int q = 32 * c + 8 * (i >> 2) + 4 * hr + (i & 3);
                        if (q < I.nt) out[(size_t)(MERGE ? I.t_first + q : pids[q]) * H + row] = acc[c][i];
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 16; i += 2) {
                        const int q = 16 * c + 4 * (i >> 2) + 2 * hr + ((i >> 1) & 1);
                        if (q < I.nt) out[(size_t)(I.t_first + q) * H + row] = acc[c][i] + acc[c][i + 1];
                    }
                }
            }
        }
        if (!NI.valid) break;
        // (every wavefront has passed this item's first barrier: none reads
        // the list of the item before it any more)
        if (tid < XG_CHUNK) s_pids[pb2][tid] = npid;
        I = NI;
        NI = NNI;
        slice = nslice;
        round++;
        nslice = k % KS;
        pb = pb1;
    }
    // every wavefront leaves with no loads in flight
    EXPERT_WAIT_VM(0);
}

// ---------------------------------------------------------------------------
// One workgroup per CU (the activation ring and the weight buffers fill the LDS), a multiple of 8 (one
// row group per XCD); each runs its items until the schedule's units end.
hipError_t launch_expert_gemm_q4k(int phase, const MoeJob &job, hipStream_t s)
{
    // routed experts (eg / eu / ed), the shared one (sg / su / sd) or both;
    // a projection is a down launch of shared units only (no routed weights;
    // the work list's count may be null there), optionally in ks reduction
    // slices
    const bool routed = job.eg.data || job.ed.data;
    const WTensor &wr = phase == 0 ? job.eg : job.ed, &ws = phase == 0 ? job.sg : job.sd;
    if ((routed && wr.type != DMOE_TYPE_Q4_K) || (!routed && !job.has_shared) ||
        (job.has_shared && ws.type != DMOE_TYPE_Q4_K && (routed || (ws.type != DMOE_TYPE_Q6_K && ws.type != DMOE_TYPE_Q8_0))))
        return hipErrorInvalidValue;
    if (!expert_gemm_q4k_ok(job.H, job.FF, job.SF, job.has_shared) || job.wl.chunk != XG_CHUNK ||
        (routed && !job.wl.n_ec))
        return hipErrorInvalidValue;
    if (phase == 0 ? ((routed && job.ax.K != job.H) || (job.has_shared && job.axs.K != job.H))
                   : ((routed && job.ah.K != job.FF) || (job.has_shared && job.ahs.K != job.SF)))
        return hipErrorInvalidValue;
    // slices (read by the down launch only): shared units only, each slice
    // two or more super-blocks
    if (phase == 1 && job.ks > 1 && (routed || (job.FF / 256) % job.ks || job.FF / 256 / job.ks < 2))
        return hipErrorInvalidValue;
    // the activation arrays' byte offsets are 32-bit: x (N rows, two digit
    // rows per token for the shared expert) and h (N k and 2 N rows)
    const long N = job.n_tokens;
    if (phase == 0 ? 2L * N * job.H >= (1L << 31)
                   : N * job.top_k * job.FF >= (1L << 31) || 2L * N * job.SF >= (1L << 31))
        return hipErrorInvalidValue;
    if (phase == 0 ? ((routed && !job.h) || (job.has_shared && !job.hs))
                   : ((routed && !job.ye) || (job.has_shared && !job.ys)))
        return hipErrorInvalidValue;
    int n_cu = 0;
    const hipError_t e = device_cu_count(&n_cu);
    if (e != hipSuccess) return e;
    const int grid = ((n_cu + 7) / 8) * 8;
    const dim3 gd(grid), bd(XG_WAVES * 64);
    if (ws.type == DMOE_TYPE_Q8_0) {
        if (routed || phase == 0) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_gemm_q<XgQ80, true, true>), gd, bd, 0, s, job);
        return hipGetLastError();
    }
    if (ws.type == DMOE_TYPE_Q6_K && !routed && phase == 1 && N <= XG_SCHUNK / 2) {
        hipLaunchKernelGGL((k_gemm_q<XgQ6K, true, true, true>), gd, bd, 0, s, job);
    } else if (ws.type == DMOE_TYPE_Q6_K && !routed) {
        if (phase == 0)
            hipLaunchKernelGGL((k_gemm_q<XgQ6K, false, true>), gd, bd, 0, s, job);
        else
            hipLaunchKernelGGL((k_gemm_q<XgQ6K, true, true>), gd, bd, 0, s, job);
    } else if (!routed) {
        if (phase == 0)
            hipLaunchKernelGGL((k_gemm_q<XgQ4K, false, true>), gd, bd, 0, s, job);
        else
            hipLaunchKernelGGL((k_gemm_q<XgQ4K, true, true>), gd, bd, 0, s, job);
    } else {
        if (phase == 0)
            hipLaunchKernelGGL((k_gemm_q<XgQ4K, false, false>), gd, bd, 0, s, job);
        else
            hipLaunchKernelGGL((k_gemm_q<XgQ4K, true, false>), gd, bd, 0, s, job);
    }
    return hipGetLastError();
}

} // namespace dmoe
