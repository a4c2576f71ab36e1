// gemm.hip -- grouped dequant-fused GEMM for gfx950: many-row problems
// (prefill chunks, verification batches, dense matrices of many rows), y[b, o]
// = sum_g scale[o, g] * sum_{k in g} x[b, k] w[o, k], the same arithmetic as
// the GEMV (c/quant.h fmt=4 and fmt=7) with the weights read once per 128 rows
// instead of once per 16.
//
// Work item = (problem, 128-row tile (64: moe_tile_rows, moe.hip), output block of COLI_GM_BLOCK_TILES row
// tiles, K split). Tiles of more than 64 rows run gemm_tall below (their
// bound is the matrix cores and the issue slots); shorter ones, whose bound is
// the weight stream, the loop described here. A K split (only where the host
// knows the work list: gemm_plan, expert.hip) leaves raw partial sums that
// coli_gemm_reduce adds in split order. A workgroup of COLI_GM_W waves gives
// each wave R = COLI_GM_BLOCK_TILES / COLI_GM_W weight tiles (DUAL: gate/up
// pairs of the same 16 output rows, SwiGLU in the epilogue) over its K, one
// 128-column quad per step:
//  * every load of the main loop is an LDS DMA into a ring of PD stages: each
//    wave's weight tiles and their scales (private to the wave), and the
//    quad's activation fragments of the tile's rows (fp16 hi + lo of x * 2^-E,
//    built by coli_prep_frag; shared by the workgroup, each wave fetching a
//    number of the 1 KiB chunks that depends on the live subtiles). No load of the loop writes a
//    register, so the compiler inserts no wait of its own: the loop waits with
//    exact s_waitcnt vmcnt(N) for its oldest stage and synchronizes with a
//    bare s_barrier (the fence of __syncthreads() would drain the ring). The
//    activations ride in the same ring as the weights, as deep: loads retire
//    in order, so a shallower activation ring would retire the weights with it;
//  * an activation chunk is 4 rows x 256 B, whole cache lines (16 rows x 64 B, and
//    as many DMAs for dead subtiles as for live ones, before: the 384-expert
//    MXFP4 layer at 512 rows 1086 -> 1051 us),
//    its 16 B pieces XOR-swizzled so the operand reads are free of bank
//    conflicts;
//  * the loop is specialized per (lo parts present, folded scales, live
//    16-row subtiles NM): the stage holds only NM subtiles' activations, so
//    short tiles (the common prefill case of a few rows per expert) stream
//    through a deeper ring, and the MFMA schedule is straight-line code;
//  * each 32-column group is one v_mfma_f32_16x16x32_f16 per (weight tile,
//    live 16-row subtile) -- two with the lo fragments -- its result scaled by
//    the group scale and accumulated in f32. The unpacked B operand of a group
//    is reused by the row subtiles. MXFP4 matrices whose e8m0 scales keep
//    every e2m1 value times its scale a normal fp16 (fold) take the scale into
//    the unpack instead (exact) and accumulate inside the MFMA: no per-group
//    VALU work beyond the conversion.
// Measured limits: the LDS carries the DMA writes and every wave's operand
// reads, and its capacity bounds the ring depth; more tiles per wave (fewer
// activation reads) costs ring depth and occupancy and was slower.
#include <type_traits>

// waves per workgroup; each owns COLI_GM_BLOCK_TILES / COLI_GM_W weight tiles
#ifndef COLI_GM_W
#define COLI_GM_W 8
#endif

#include "coli_device.h"

// deepest ring a short tile gets
#ifndef COLI_GM_PDMAX
#define COLI_GM_PDMAX 6
#endif

// Ring geometry. A stage holds the activation chunks of the tile's live
// 16-row subtiles (NM of them, 4 KiB each for the hi half, as much again for
// lo) and each wave's weight tiles + scales; the ring takes as many stages as
// the LDS of a CU holds (at most 6), so short tiles stream deeper. One 1 KiB
// trash slot takes the DMAs past a stage's last chunk (their count per wave
// depends on NM alone).
template <int KIND>
struct GmGeom {
    static constexpr int kMt = COLI_GM_ROWS / 16;                 // 16-row subtiles per tile
    static constexpr int kW = COLI_GM_W, kR = COLI_GM_BLOCK_TILES / COLI_GM_W;   // waves, tiles per wave
    static constexpr int scale_inst(int rn) { return (rn + ScaleGeom<KIND>::kPerInst - 1) / ScaleGeom<KIND>::kPerInst; }
    static constexpr int wslot(int rn) { return rn * COLI_TILE_BYTES + scale_inst(rn) * 256; }
    static constexpr int kTrash = 0;                               // the trash slot, then the ring
    static constexpr int kRing = 1024;
    static constexpr int kLds = 159 * 1024;
    static constexpr int act(int nm, bool lo) { return nm * 4096 * (lo ? 2 : 1); }
    static constexpr int stage(int nm, bool lo, int rn) { return act(nm, lo) + kW * wslot(rn); }
    static constexpr int pd(int nm, bool lo, int rn) {
        return (kLds - kRing) / stage(nm, lo, rn) > COLI_GM_PDMAX ? COLI_GM_PDMAX : (kLds - kRing) / stage(nm, lo, rn);
    }
    // tiles per pass: all of the wave's tiles when three stages fit, else two
    // passes over K of half as many (the activations are staged twice)
    static constexpr int passes(int nm, bool lo) { return pd(nm, lo, kR) >= 3 ? 1 : 2; }
};
static_assert(GmGeom<COLI_KIND_I4_F>::pd(COLI_GM_ROWS / 16, true, GmGeom<COLI_KIND_I4_F>::kR / 2) >= 3,
              "the ring needs three stages");

// Ring geometry of a tall tile (65-128 rows). Activations are staged per half
// quad (2 groups x 8 subtiles), weights and scales per quad; the weights of
// quad q are fetched with the activations of quad q - 1.
template <int KIND>
struct GtGeom {
    static constexpr int kSub = COLI_GM_TILE / 16;
    static constexpr int kHalf = 2 * kSub * 1024;                                       // one half quad, hi or lo
    static constexpr int act(bool lo) { return kHalf * (lo ? 2 : 1); }
    static constexpr int kWSlot = COLI_GM_BLOCK_TILES * (COLI_TILE_BYTES + ScaleGeom<KIND>::kBytes);
    static constexpr int pd(bool lo) { return lo ? 3 : 5; }                             // activation stages
    static constexpr int nw(bool lo) { return lo ? 2 : 3; }                             // weight slots
    static constexpr int kScInst = COLI_GM_BLOCK_TILES * ScaleGeom<KIND>::kBytes / 1024;  // 1 KiB scale DMAs a quad
    static constexpr int kExp = GmGeom<KIND>::kLds - 4096;   // the rows' exponents, 8 copies each
    static_assert(act(true) * pd(true) + nw(true) * kWSlot <= kExp && act(false) * pd(false) + nw(false) * kWSlot <= kExp,
                  "the rings must fit the LDS");
};

// Byte offset in a subtile's 2 KiB half quad of the 16 B that lane l of a
// 32x32x16 operand reads for (group g, K half t): row l % 16, k-slice 2 t +
// l / 32. A row's eight 16 B pieces are stored XORed with a key of the row, so
// the sixteen lanes of a phase read sixteen different slots of 256 B.
__device__ __forceinline__ int tall_key(int r) { return (r & 7) ^ (r >> 3); }
__device__ __forceinline__ int tall_off(int lane, int g, int t) {
    const int r = lane & 15;
    return ((lane >> 4) & 1) * 2048 + r * 128 + 16 * ((4 * g + 2 * t + (lane >> 5)) ^ tall_key(r));
}

// One tall tile's pass over quads [0, nq): the workgroup's 8 waves are 2 (row
// halves) x 4 (four weight tiles each); a wave computes NB 32-row blocks x two
// 32-column blocks (tiles 2n, 2n + 1) on v_mfma_f32_32x32x16_f16, so every
// activation it reads from LDS feeds four tiles (the short tiles' 1 x 8
// arrangement: two) and an MFMA takes two issue slots for 32 cycles (the
// 16x16x32 form: two for 16; the int4 loop is bound by its VALU and MFMA issue
// slots). wt0, wt1: quad 0 of tiles wave, wave + 8 of the block; sp: this
// lane's 16 B of the wave's scale DMA; xo0, xo1: this lane's 16 B of rows 16
// wave + l / 8 and + 8 (one DMA covers 8 rows x 128 B: whole cache lines; 16
// rows x 64 B ran at half the rate). store(row, tile of the block, gate or
// plain value, value of the tile after it) takes the results.
//
// SEG: segq quads at most go into one running sum (see dense_chain,
// expert.hip). The sums so far are written to this wave's part of a scratch
// buffer, one set after another (nothing waits for the stores), and added at
// the end: a second set of accumulators does not fit the registers (spilled
// inside the loop), and adding to the first set in memory every time waits for
// it behind the ring's DMAs (the 512-row feed-forward of 4096 x 14336 int4: 411
// us as one chain, 480 us with the sums added in memory, 447 us so).
//
// The loop is a sequence of steps, one per (group, row block, column block):
// the step's 2 (4 with lo parts) MFMAs beside the work that needs no result of
// theirs: the LDS reads of the next fragments, the scaling of the previous
// step's products and a quarter of the next group's unpack. Left to itself the
// compiler reads each fragment right before its use and waits for it.
// (sched_barrier: nothing crosses a step; sched_group_barrier: MFMAs and VALU
// work interleave inside it.) The ring is synchronized in the last step of
// each half quad, whose own operands are in registers by then.
// Measured (512 x 14336 x 4096 with lo parts, two MFMAs a product): int4 329 us
// on the GEMV kernel, 155 us with the same tiles scheduled by the compiler,
// 119-139 us here (1.0 PFLOP/s of MFMA work; 1.2 MXFP4; a bf16 library product
// of 8192^3 reaches 1.4 on the card).
template <int KIND, bool LO, bool FOLD, int NB, bool SEG, typename Store>
__device__ __forceinline__ void gemm_tall(uint8_t *lds, const uint8_t *wt0, const uint8_t *wt1, const uint8_t *sp,
                                          const _Float16 *xhi, const _Float16 *xlo, uint32_t xo0, uint32_t xo1, int nq,
                                          int segq, float *sums, int lane, int wave, Store store) {
    using T = GtGeom<KIND>;
    using SG = ScaleGeom<KIND>;
    constexpr int PD = T::pd(LO), NW = T::nw(LO), ACT = T::act(LO), WS = T::kWSlot;
    constexpr int LA = LO ? 4 : 2;   // activation DMAs of a half quad and wave
    uint8_t *const aring = lds, *const wring = lds + PD * ACT;
    const int wm = wave >> 2, wn = wave & 3;
    const int nh = 2 * nq;
    // weights of quad q into weight slot ws, part (half): tile wave + 8 part,
    // and with part 0 the scales
    auto issue_w = [&](int q, uint8_t *ws, int part) {
        q = min(q, nq - 1);
        __builtin_amdgcn_global_load_lds((const void *)((part ? wt1 : wt0) + (size_t)q * COLI_TILE_BYTES + lane * 16),
                                         (lds_void *)(ws + (wave + 8 * part) * COLI_TILE_BYTES), 16, 0, 0);
        if (part == 0)
            __builtin_amdgcn_global_load_lds((const void *)(sp + (size_t)q * SG::kBytes),
                                             (lds_void *)(ws + COLI_GM_BLOCK_TILES * COLI_TILE_BYTES +
                                                          (wave % T::kScInst) * 1024),
                                             16, 0, 0);
    };
    // half quad h (part h & 1) into activation slot xs, and its share of the
    // weights of quad h / 2 + 1 into slot ws. Past the end the last half quad
    // is fetched again and nothing reads it: without a branch the loop's body
    // is one basic block (across a branch the compiler sinks the scaling of
    // the products to the end of the loop and spills them), and the counts of
    // loads in flight stay fixed.
    auto issue = [&](int h, uint8_t *xs, uint8_t *ws, int part) {
        xs += wave * 2048;
        const size_t o = (size_t)min(h, nh - 1) * 64;
        __builtin_amdgcn_global_load_lds((const void *)(xhi + xo0 + o), (lds_void *)xs, 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const void *)(xhi + xo1 + o), (lds_void *)(xs + 1024), 16, 0, 0);
        if constexpr (LO) {
            __builtin_amdgcn_global_load_lds((const void *)(xlo + xo0 + o), (lds_void *)(xs + T::kHalf), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const void *)(xlo + xo1 + o), (lds_void *)(xs + T::kHalf + 1024), 16, 0, 0);
        }
        issue_w((h >> 1) + 1, ws, part);
    };
    // operands, all indices constant: the quad's tiles w[n][t] (the two K
    // halves), reloaded for the next quad once unpacked; bw of this group and
    // the next; fragments of this row block and the next; products of this
    // step and the previous one
    u32x4 w[2][2];
    ScaleRegs<KIND> sc[2];
    half8v bw[2][2][2], xh[2][2], xl[2][2];
    float scl[2][2];
    floatx16 d[2], acc[NB][2];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        d[1][i] = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; b++) acc[b][0][i] = acc[b][1][i] = 0.0f;
    }
    const int l16 = (lane >> 4) & 1, wofs = l16 * COLI_TILE_BYTES + ((lane >> 5) * 16 + (lane & 15)) * 16;
    auto load_w = [&](int n, int t, const uint8_t *ws) {
        w[n][t] = *(const u32x4 *)(ws + (wn * 4 + 2 * n) * COLI_TILE_BYTES + t * 512 + wofs);
    };
    auto load_sc = [&](int n, const uint8_t *ws) {
        sc[n].v = *(const decltype(sc[n].v) *)(ws + COLI_GM_BLOCK_TILES * COLI_TILE_BYTES +
                                               (wn * 4 + 2 * n + l16) * SG::kBytes + (lane & 15) * sizeof(sc[n].v));
    };
    auto unpack = [&](int n, int t, int j) {
        if (t == 0) scl[j & 1][n] = sc[n].get(j);
        if constexpr (FOLD) bw[j & 1][n][t] = unpack_fp4_scaled(w[n][t][j], scl[j & 1][n]);
        else bw[j & 1][n][t] = unpack_b<KIND>(w[n][t][j]);
    };
    const int xofs[2][2] = {{tall_off(lane, 0, 0), tall_off(lane, 0, 1)}, {tall_off(lane, 1, 0), tall_off(lane, 1, 1)}};
    auto load_x = [&](int p, const uint8_t *xs, int g, int b) {   // group g (0, 1) of the half quad, row block b
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint8_t *q = xs + (2 * wm + b) * 4096 + xofs[g][t];
            xh[p][t] = *(const half8v *)q;
            if constexpr (LO) xl[p][t] = *(const half8v *)(q + T::kHalf);
        }
    };
    auto scale = [&](auto pt, auto bt, auto nt, auto jt) {   // products d[p] of blocks (b, n), group parity jp
        constexpr int p = decltype(pt)::value, b = decltype(bt)::value, n = decltype(nt)::value;
        constexpr int jp = decltype(jt)::value;
        if constexpr (!FOLD) {
            floatx16 v = acc[b][n];
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = fmaf(d[p][i], scl[jp][n], v[i]);
            acc[b][n] = v;
        }
    };
    auto wait_lds = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    auto barrier = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto aslot = [&](int k) { return aring + k * ACT; };
    auto wslot = [&](int k) { return wring + k * WS; };
    issue_w(0, wslot(0), 0);
    issue_w(0, wslot(0), 1);
#pragma unroll
    for (int i = 0; i < PD - 1; i++)
        issue(i, aslot(i), wslot(((i >> 1) + 1) % NW), i & 1);
    constexpr int P0 = PD == 3 ? LA + 1 : 3 * LA + 4;   // stages 1 .. PD - 2
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P0) : "memory");
    barrier();
#pragma unroll
    for (int n = 0; n < 2; n++) {
        load_sc(n, wslot(0));
        load_w(n, 0, wslot(0));
        load_w(n, 1, wslot(0));
    }
    wait_lds();
    barrier();   // weight slot 0 is free
    issue(PD - 1, aslot(PD - 1), wslot((((PD - 1) >> 1) + 1) % NW), (PD - 1) & 1);
#pragma unroll
    for (int n = 0; n < 2; n++) {
        unpack(n, 0, 0);
        unpack(n, 1, 0);
        scl[1][n] = 0.0f;
    }
    load_x(0, aslot(0), 0, 0);
    int as = 0, wn1 = 1 % NW;        // activation slot of the half quad; weight slot of the next quad
    int wi = ((PD >> 1) + 1) % NW;   // weight slot of the next issue (half quad PD)
    // step (group j, row block b, column block n) of quad c; the tags keep
    // every index constant
    auto step = [&](int c, auto jt, auto bt, auto nt) {
        constexpr int j = decltype(jt)::value, b = decltype(bt)::value, n = decltype(nt)::value;
        constexpr int s = b * 2 + n, NS = 2 * NB;                    // step of the group
        constexpr int p = (j * NB + b) & 1, dp = n;                  // parity of the fragments, of the products
        constexpr int part = j >> 1;
        constexpr bool lastb = b == NB - 1, half_end = lastb && (j & 1);
        if constexpr (half_end && n == 1) {
            // end of half quad h: its operands are read (their slot is free
            // after the barrier), half quad h + 1 is waited for (stages h + 2
            // .. h + PD - 1 stay in flight)
            const int h = 2 * c + part;
            constexpr int NP = PD == 3 ? (part ? LA + 1 : LA + 2) : 3 * LA + (part ? 4 : 5);
            wait_lds();
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NP) : "memory");
            barrier();
            issue(h + PD, aslot(as), wslot(wi), (part + PD) & 1);
            if ((part + PD) & 1) wi = wi == NW - 1 ? 0 : wi + 1;
            as = as == PD - 1 ? 0 : as + 1;
        }
        // fragments of the next row block: in this block's first step, or
        // after the ring's synchronization
        if constexpr (half_end ? n == 1 : n == 0) load_x(p ^ 1, aslot(as), (lastb ? j + 1 : j) & 1, lastb ? 0 : b + 1);
        floatx16 z = {};
        if constexpr (FOLD) z = acc[b][n];
#pragma unroll
        for (int t = 0; t < 2; t++) z = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh[p][t], bw[j & 1][n][t], z, 0, 0, 0);
        if constexpr (LO) {
#pragma unroll
            for (int t = 0; t < 2; t++)
                z = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl[p][t], bw[j & 1][n][t], z, 0, 0, 0);
        }
        if constexpr (FOLD) acc[b][n] = z;
        else d[dp] = z;
        // scale the previous step's products (n - 1 of this row block, or n =
        // 1 of the one before)
        constexpr int pb = n == 1 ? b : (b == 0 ? NB - 1 : b - 1), pj = n == 1 || b > 0 ? j : j + 3;
        scale(std::integral_constant<int, dp ^ 1>{}, std::integral_constant<int, pb>{},
              std::integral_constant<int, n ^ 1>{}, std::integral_constant<int, pj & 1>{});
        // the next group's operands, 4 / NS of the four (n, t) a step, and of
        // the next quad's tiles once the last group's are unpacked
#pragma unroll
        for (int k = s * (4 / NS); k < (s + 1) * (4 / NS); k++) {
            unpack(k >> 1, k & 1, (j + 1) & 3);
            if constexpr (j == 2) {
                load_w(k >> 1, k & 1, wslot(wn1));
                if (k & 1) load_sc(k >> 1, wslot(wn1));
            }
        }
        // an MFMA first: the wait for this step's operands then comes before
        // the next fragments' reads are queued behind them
        constexpr int NM = LO ? 4 : 2, NV = FOLD ? 6 / NM : (16 + 12 * (4 / NS) + NM - 1) / NM;
#pragma unroll
        for (int k = 0; k < NM; k++) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, NV, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto group = [&](int c, auto jt) {
        using C0 = std::integral_constant<int, 0>;
        using C1 = std::integral_constant<int, 1>;
        step(c, jt, C0{}, C0{});
        step(c, jt, C0{}, C1{});
        if constexpr (NB == 2) {
            step(c, jt, C1{}, C0{});
            step(c, jt, C1{}, C1{});
        }
    };
    auto quad = [&](int c) {
        group(c, std::integral_constant<int, 0>{});
        group(c, std::integral_constant<int, 1>{});
        group(c, std::integral_constant<int, 2>{});
        group(c, std::integral_constant<int, 3>{});
        wn1 = wn1 == NW - 1 ? 0 : wn1 + 1;
    };
    if constexpr (!SEG) {
        for (int c = 0; c < nq; c++) quad(c);
    } else {
        // (the last step's products, not scaled yet, open the next sum)
        for (int c = 0;;) {
            for (const int ce = min(nq, c + segq); c < ce; c++) quad(c);
            if (c >= nq) break;
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int n = 0; n < 2; n++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        floatx4 v;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            v[i] = acc[b][n][4 * k + i];
                            acc[b][n][4 * k + i] = 0.0f;
                        }
                        *(floatx4 *)(sums + (b * 8 + n * 4 + k) * 256 + lane * 4) = v;
                    }
            sums += COLI_GM_SUMS;
        }
    }
    scale(std::integral_constant<int, 1>{}, std::integral_constant<int, NB - 1>{}, std::integral_constant<int, 1>{},
          std::integral_constant<int, 1>{});
    // the last DMAs write this workgroup's LDS: none may outlive it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (SEG) {
        for (int c = segq; c < nq; c += segq) {
            sums -= COLI_GM_SUMS;
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int n = 0; n < 2; n++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const floatx4 v = *(const floatx4 *)(sums + (b * 8 + n * 4 + k) * 256 + lane * 4);
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[b][n][4 * k + i] += v[i];
                    }
        }
    }
    // lane l, register i: row 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            store(wm * 64 + b * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3), 4 * wn + l16, acc[b][0][i], acc[b][1][i]);
}

// SEG: a.segq quads at most in one running sum (plain matrices).
template <int KIND, bool DUAL, bool SEG>
__global__ __launch_bounds__(64 * COLI_GM_W) void coli_gemm_tiles(ColiGemmArgs a) {
    using G = GmGeom<KIND>;
    using SG = ScaleGeom<KIND>;
    constexpr int W = G::kW;
    constexpr int R = G::kR;                  // weight tiles per wave
    constexpr int RT = DUAL ? R / 2 : R;      // distinct output row tiles per wave
    static_assert(W * R == COLI_GM_BLOCK_TILES && R % 2 == 0, "a block covers COLI_GM_BLOCK_TILES weight tiles");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    // readfirstlane: the wave index is wave-uniform, so everything derived from it
    // (tile indices, validity, base pointers) stays in scalar registers.
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const int part = blockIdx.x / a.rb_per_prob, rb = blockIdx.x - part * a.rb_per_prob;
    const int item = part / a.splits, split = part - item * a.splits;
    if (a.n_mt_dev && item >= *a.n_mt_dev) return;
    if (item >= a.n_mt) return;
    int p = 0, mt = item;
    if (a.prob) {
        const int tag = a.mt_list[item];
        p = tag >> 16;
        mt = tag & 0xffff;
        if (p >= a.nprob || (a.nprob_dev && p >= *a.nprob_dev)) return;
    }
    const ColiProb pr = uniform_prob(a.prob ? a.prob[p] : a.prob0);
    const int m0 = mt * a.tile;
    const int nrows = min(a.tile, pr.nrows - m0);
    if (nrows <= 0) return;
    const int Q0 = split * a.qps, nq = min(a.nq, Q0 + a.qps) - Q0;   // this workgroup's quads

    const bool use_lo = *a.haslo >= a.lo_gen;   // >=: stays correct under graph replay
    const int nm = (nrows + 15) >> 4;           // live 16-row subtiles
    // the ring is written behind the compiler's back: let it escape, so the
    // "memory" clobbers of the waits below force fresh reads (plain loads: no
    // read moves across a wait or barrier, and the compiler may batch the
    // reads of one step)
    asm volatile("" ::"v"(lds) : "memory");

    // Value(s) of row bl of the tile, output row 16 k + lane % 16 of the block
    // (DUAL: v, u its gate and up), E the row's exponent: stored scaled back
    // by 2^E, or with a K split as this split's raw partials. The exponents
    // come through LDS with the first DMAs: loaded here they were a chain of
    // one memory round trip a row (16384 rows of K 1024, 2048 outputs: 248 ->
    // 210 us).
    auto store = [&](int bl, int k, int E, float v, float u) {
        if (bl >= nrows) return;
        const int orow = pr.out_row0 + m0 + bl;
        if (a.splits > 1) {
            float *pp = a.partial + ((size_t)split * a.part_rows + orow) * a.rb_per_prob * (COLI_GM_BLOCK_TILES * 16) +
                        (size_t)rb * (COLI_GM_BLOCK_TILES * 16) + (DUAL ? 32 : 16) * k + (lane & 15);
            pp[0] = v;
            if constexpr (DUAL) pp[16] = u;
            return;
        }
        const int o = (rb * (COLI_GM_BLOCK_TILES / (DUAL ? 2 : 1)) + k) * 16 + (lane & 15);
        if (o >= a.O) return;
        float *y = a.out + (size_t)orow * a.ldo + o;
        if constexpr (DUAL) *y = swiglu_out(ldexpf(v, E), ldexpf(u, E), a.swiglu_limit);
        else *y = ldexpf(v, E);
    };

    if (nm > G::kMt) {
        // tall tile: tile k of the block (DUAL: a wave's tiles 4 i .. 4 i + 3 =
        // gate, gate, up, up of the block's row tiles 2 i, 2 i + 1); past the
        // matrix its last row tile is read
        auto tile_of = [&](int k, const uint8_t *&w, const uint8_t *&sc) {
            const int r = min(DUAL ? rb * 8 + 2 * (k >> 2) + (k & 1) : rb * 16 + k, a.nrt - 1);
            const bool second = DUAL && (k & 2);
            const size_t t0 = (size_t)r * a.nq + Q0;
            w = (const uint8_t *)(second ? pr.w1 : pr.w0) + t0 * COLI_TILE_BYTES;
            sc = (const uint8_t *)(second ? pr.s1 : pr.s0) + t0 * SG::kBytes;
        };
        using T = GtGeom<KIND>;
        const uint8_t *wt[2], *sp, *unused;
        tile_of(wave, wt[0], unused);
        tile_of(wave + 8, wt[1], unused);
        // 1 KiB scale DMA wave % kScInst of the quad: lane l fetches 16 B of
        // tile (16 / kScInst) (wave % kScInst) + l / (kBytes / 16)
        constexpr int SL = SG::kBytes / 16;
        tile_of((wave % T::kScInst) * (COLI_GM_BLOCK_TILES / T::kScInst) + lane / SL, unused, sp);
        sp += (lane % SL) * 16;
        // this lane's row and 16 B of the activation DMAs: row 16 wave + 8 k +
        // l / 8, its eight 16 B pieces of a half quad stored XORed
        uint32_t xo[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int r = 8 * k + (lane >> 3), br = pr.xrow_off + m0 + min(16 * wave + r, nrows - 1);
            const int fr = a.xrows ? a.xrows[br] : br;
            xo[k] = (uint32_t)fr * (uint32_t)a.xstride + 128 * Q0 + 8 * ((lane & 7) ^ tall_key(r));
            // the row's exponent, once per lane of the row
            __builtin_amdgcn_global_load_lds((const void *)(a.xexp + fr),
                                             (lds_void *)(lds + GtGeom<KIND>::kExp + (2 * wave + k) * 256), 4, 0, 0);
        }
        const int *const es = (const int *)(lds + GtGeom<KIND>::kExp);
        auto put = [&](int bl, int k, float v, float u) {
            const int E = es[(bl >> 3) * 64 + (bl & 7) * 8];
            if constexpr (DUAL) {
                store(bl, 2 * (k >> 2) + (k & 1), E, v, u);
            } else {
                store(bl, k, E, v, 0.0f);
                store(bl, k + 2, E, u, 0.0f);
            }
        };
        float *sums = nullptr;
        if constexpr (SEG)
            sums = a.sums + (size_t)blockIdx.x * ((a.qps - 1) / a.segq) * COLI_GM_SUMS + wave * (COLI_GM_SUMS / COLI_GM_W);
        // the second row half of a tile of up to 96 rows has one row block
        auto go = [&](auto lo_tag, auto fold_tag) {
            constexpr bool LO = decltype(lo_tag)::value, FOLD = decltype(fold_tag)::value;
            if (nm <= 6 && wave >= 4)
                gemm_tall<KIND, LO, FOLD, 1, SEG>(lds, wt[0], wt[1], sp, a.xhi, a.xlo, xo[0], xo[1], nq, a.segq, sums,
                                                  lane, wave, put);
            else
                gemm_tall<KIND, LO, FOLD, 2, SEG>(lds, wt[0], wt[1], sp, a.xhi, a.xlo, xo[0], xo[1], nq, a.segq, sums,
                                                  lane, wave, put);
        };
        auto by_fold = [&](auto lo_tag) {
            if constexpr (KIND == COLI_KIND_FP4 && !SEG) {
                if (a.fold) go(lo_tag, std::true_type{});
                else go(lo_tag, std::false_type{});
            } else {
                go(lo_tag, std::false_type{});
            }
        };
        if (use_lo) by_fold(std::true_type{});
        else by_fold(std::false_type{});
        return;
    }

    int rt[R];
    bool live[R];
    const uint8_t *wr[R], *sr[R];   // tile (rt, 0) of the wave's weights and scales
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int rr = DUAL ? r >> 1 : r;   // DUAL: tiles 2i, 2i + 1 = gate, up of row tile i
        rt[r] = (rb * W + wave) * RT + rr;
        live[r] = rt[r] < a.nrt;
        const bool second = DUAL && (r & 1);
        const uint8_t *w = (const uint8_t *)(second ? pr.w1 : pr.w0);
        const uint8_t *sc = (const uint8_t *)(second ? pr.s1 : pr.s0);
        // a dead tile re-reads tile (0, q) of the problem: the count of loads
        // stays fixed and no address is hammered by every quad
        const size_t t0 = (live[r] ? (size_t)rt[r] * a.nq : 0) + Q0;
        wr[r] = w + t0 * COLI_TILE_BYTES;
        sr[r] = sc + t0 * SG::kBytes;
    }

    // the rows' exponents: wave w < 4 fetches subtile w's, four copies
    if (wave < G::kMt) {
        const int br = pr.xrow_off + m0 + min(16 * wave + (lane & 15), nrows - 1);
        __builtin_amdgcn_global_load_lds((const void *)(a.xexp + (a.xrows ? a.xrows[br] : br)),
                                         (lds_void *)(lds + G::kLds + wave * 256), 4, 0, 0);
    }

    floatx4 acc[R][G::kMt];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < G::kMt; m++) acc[r][m] = (floatx4){0.f, 0.f, 0.f, 0.f};

    // One pass over K for the wave's tiles RB .. RB + RN - 1.
    auto run = [&](auto lo_tag, auto fold_tag, auto nm_tag, auto rb_tag, auto rn_tag) {
        constexpr bool LO = decltype(lo_tag)::value;
        constexpr bool FOLD = decltype(fold_tag)::value;
        constexpr int NM = decltype(nm_tag)::value;     // live 16-row subtiles
        constexpr int RB = decltype(rb_tag)::value, RN = decltype(rn_tag)::value;
        constexpr int PD = G::pd(NM, LO, RN);
        constexpr int ACT = G::act(NM, LO);             // activation bytes of one stage
        constexpr int LOFF = G::act(NM, false);         // lo half of the stage
        constexpr int SI = G::scale_inst(RN);
        constexpr int WS = G::wslot(RN);
        static_assert(PD >= 3, "the ring needs three stages");
        // Activation chunks of a stage: 4 rows x 256 B (whole cache lines),
        // the NM subtiles' hi chunks, then lo. Wave w fetches chunks w, w + 8,
        // ...: only as many DMAs as the live subtiles need (their count
        // depends on NM alone); a chunk past the end reads row 0 of the tile
        // into the trash slot. The sixteen 16 B pieces of a row are stored
        // XORed with row % 16, so the sixteen lanes of one k-slice read
        // sixteen different slots.
        constexpr int NCH = 4 * NM * (LO ? 2 : 1), CPW = (NCH + W - 1) / W;
        constexpr int L = RN + SI + CPW;   // DMA instructions per wave and stage
        uint32_t xoff[CPW];
#pragma unroll
        for (int k = 0; k < CPW; k++) {
            const int c = (wave + W * k) % (4 * NM), r = 4 * c + (lane >> 4);   // row of the tile
            const int br = pr.xrow_off + m0 + min(wave + W * k < NCH ? r : 0, nrows - 1);
            const int fr = a.xrows ? a.xrows[br] : br;
            xoff[k] = (uint32_t)fr * (uint32_t)a.xstride + 128 * Q0 + 8 * ((lane & 15) ^ (r & 15));
        }
        int xrd[4];   // the lane's 16 B of group j in a subtile
#pragma unroll
        for (int j = 0; j < 4; j++) xrd[j] = (lane & 15) * 256 + 16 * ((4 * j + (lane >> 4)) ^ (lane & 15));
        uint8_t *const ring = lds + G::kRing;
        uint8_t *const wring = ring + PD * ACT + wave * PD * WS;
        auto issue = [&](int q, int slot) {
            uint8_t *ws = wring + slot * WS;
#pragma unroll
            for (int t = 0; t < RN; t++)
                __builtin_amdgcn_global_load_lds((const void *)(wr[RB + t] + (size_t)q * COLI_TILE_BYTES + lane * 16),
                                                 (lds_void *)(ws + t * COLI_TILE_BYTES), 16, 0, 0);
#pragma unroll
            for (int k = 0; k < SI; k++) {
                const int t = min(RN - 1, k * SG::kPerInst + lane / SG::kLanes);
                const uint8_t *base = sr[RB];   // (branch-free: a per-lane select between RN bases)
#pragma unroll
                for (int tt = 1; tt < RN; tt++)
                    if (t == tt) base = sr[RB + tt];
                __builtin_amdgcn_global_load_lds((const void *)(base + (size_t)q * SG::kBytes + (lane % SG::kLanes) * 4),
                                                 (lds_void *)(ws + RN * COLI_TILE_BYTES + k * 256), 4, 0, 0);
            }
            uint8_t *xs = ring + slot * ACT;
#pragma unroll
            for (int k = 0; k < CPW; k++) {
                const int c = wave + W * k;
                const _Float16 *src = LO && c >= 4 * NM ? a.xlo : a.xhi;   // (lo chunks follow the hi ones in the stage)
                __builtin_amdgcn_global_load_lds((const void *)(src + (size_t)xoff[k] + (size_t)q * 128),
                                                 (lds_void *)(c < NCH ? xs + c * 1024 : lds + G::kTrash), 16, 0, 0);
            }
        };
        auto compute = [&](int slot) {
            const uint8_t *ws = wring + slot * WS;
            const uint8_t *xs = ring + slot * ACT;
            u32x4 w[RN];
            ScaleRegs<KIND> sc[RN];
#pragma unroll
            for (int t = 0; t < RN; t++) {
                w[t] = *(const u32x4 *)(ws + t * COLI_TILE_BYTES + lane * 16);
                sc[t].v = *(const decltype(sc[t].v) *)(ws + RN * COLI_TILE_BYTES + t * SG::kBytes +
                                                       (lane & 15) * sizeof(sc[t].v));
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                half8v bw[RN];
                float scl[RN];
#pragma unroll
                for (int t = 0; t < RN; t++) {
                    scl[t] = sc[t].get(j);
                    if constexpr (FOLD) bw[t] = unpack_fp4_scaled(w[t][j], scl[t]);
                    else bw[t] = unpack_b<KIND>(w[t][j]);
                }
                half8v xh[NM], xl[NM];
#pragma unroll
                for (int m = 0; m < NM; m++) {
                    const uint8_t *fo = xs + m * 4096 + xrd[j];
                    xh[m] = *(const half8v *)fo;
                    if constexpr (LO) xl[m] = *(const half8v *)(fo + LOFF);
                }
                if constexpr (FOLD) {
                    // the operand carries the group scale: accumulate in the MFMA
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int t = 0; t < RN; t++)
                            acc[RB + t][m] =
                                __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[m], bw[t], acc[RB + t][m], 0, 0, 0);
                    if constexpr (LO) {
#pragma unroll
                        for (int m = 0; m < NM; m++)
#pragma unroll
                            for (int t = 0; t < RN; t++)
                                acc[RB + t][m] =
                                    __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[m], bw[t], acc[RB + t][m], 0, 0, 0);
                    }
                } else {
                    floatx4 d[RN][NM];
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int t = 0; t < RN; t++)
                            d[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[m], bw[t],
                                                                             (floatx4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    if constexpr (LO) {
#pragma unroll
                        for (int m = 0; m < NM; m++)
#pragma unroll
                            for (int t = 0; t < RN; t++)
                                d[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[m], bw[t], d[t][m], 0, 0, 0);
                    }
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int t = 0; t < RN; t++)
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                acc[RB + t][m][i] = fmaf(d[t][m][i], scl[t], acc[RB + t][m][i]);
                }
            }
        };
        // Step q: wait for this wave's stage q (at most min(PD - 2, nq - 1 - q)
        // younger stages may stay in flight), barrier (every wave's chunks of
        // stage q have landed, and every wave is done with quad q - 1, whose
        // slot the next issue reuses), issue stage q + PD - 1, compute quad q.
#pragma unroll
        for (int i = 0; i < PD - 1; i++)
            if (i < nq) issue(i, i);
        int slot = 0;
        auto pass = [&](int q0, int q1) {
            for (int q = q0; q < q1; q++) {
                dma_wait_tail<L, PD>(min(PD - 2, nq - 1 - q));
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (q + PD - 1 < nq) issue(q + PD - 1, slot == 0 ? PD - 1 : slot - 1);
                compute(slot);
                slot = slot == PD - 1 ? 0 : slot + 1;
            }
        };
        if constexpr (!SEG) {
            pass(0, nq);
        } else {
            // at most segq quads in one running sum (see dense_chain, expert.hip)
            floatx4 tot[RN][NM];
#pragma unroll
            for (int t = 0; t < RN; t++)
#pragma unroll
                for (int m = 0; m < NM; m++) tot[t][m] = (floatx4){0.f, 0.f, 0.f, 0.f};
            for (int q = 0; q < nq; q += a.segq) {
                pass(q, min(nq, q + a.segq));
#pragma unroll
                for (int t = 0; t < RN; t++)
#pragma unroll
                    for (int m = 0; m < NM; m++) {
                        tot[t][m] += acc[RB + t][m];
                        acc[RB + t][m] = (floatx4){0.f, 0.f, 0.f, 0.f};
                    }
            }
#pragma unroll
            for (int t = 0; t < RN; t++)
#pragma unroll
                for (int m = 0; m < NM; m++) acc[RB + t][m] = tot[t][m];
        }
    };
    // one specialization per (lo parts, folded scales, live subtiles); one
    // pass over K when the ring fits three stages of all the wave's tiles,
    // else one pass per half of them (the next pass refills the ring only
    // after every wave is done with the last one)
    auto by_nm = [&](auto lo_tag, auto fold_tag) {
        auto go = [&](auto nm_tag) {
            constexpr bool LO = decltype(lo_tag)::value;
            constexpr int NM = decltype(nm_tag)::value;
            using C0 = std::integral_constant<int, 0>;
            if constexpr (G::passes(NM, LO) == 1) {
                run(lo_tag, fold_tag, nm_tag, C0{}, std::integral_constant<int, R>{});
            } else {
                using H = std::integral_constant<int, R / 2>;
                run(lo_tag, fold_tag, nm_tag, C0{}, H{});
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                run(lo_tag, fold_tag, nm_tag, H{}, H{});
            }
        };
        static_assert(G::kMt == 4, "the subtile dispatch is written for 64-row tiles");
        if (nm == 1) go(std::integral_constant<int, 1>{});
        else if (nm == 2) go(std::integral_constant<int, 2>{});
        else if (nm == 3) go(std::integral_constant<int, 3>{});
        else go(std::integral_constant<int, 4>{});
    };
    auto by_lo = [&](auto fold_tag) {
        if (use_lo) by_nm(std::true_type{}, fold_tag);
        else by_nm(std::false_type{}, fold_tag);
    };
    if constexpr (KIND == COLI_KIND_FP4 && !SEG) {
        if (a.fold) by_lo(std::true_type{});
        else by_lo(std::false_type{});
    } else {
        by_lo(std::false_type{});
    }

    const int *const es = (const int *)(lds + G::kLds);
#pragma unroll
    for (int m = 0; m < G::kMt; m++) {
        if (m >= nm) break;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const int bl = m * 16 + 4 * (lane >> 4) + i;
                const int r = DUAL ? 2 * t : t;   // the gate (DUAL) or the plain tile of row tile t
                store(bl, wave * RT + t, es[m * 64 + (bl & 15)], acc[r][m][i], DUAL ? acc[DUAL ? r + 1 : r][m][i] : 0.0f);
            }
    }
}

// Sum of a K-split GEMM's partials in split order, then the GEMM's epilogue
// (2^E of the row, SwiGLU of the gate / up columns). One thread per output
// value; output row o of the matrix lies in block o / (16 T), column 16 c + o %
// 16 with c its tile in the block (DUAL: tiles 2i, 2i + 1).
template <bool DUAL>
__global__ __launch_bounds__(256) void coli_gemm_reduce(const float *__restrict__ part, int splits, int rows, int rb,
                                                        int O, const int *__restrict__ xexp, float *__restrict__ out,
                                                        int ldo, float swiglu_limit) {
    constexpr int RPB = COLI_GM_BLOCK_TILES * 16 / (DUAL ? 2 : 1);   // output rows of a block
    const int o = blockIdx.x * 256 + threadIdx.x, r = blockIdx.y;
    if (o >= O) return;
    const int ld = rb * COLI_GM_BLOCK_TILES * 16;
    const int c = DUAL ? (o / RPB) * 256 + 32 * ((o % RPB) >> 4) + (o & 15) : o;
    float v = 0.0f, u = 0.0f;
    for (int s = 0; s < splits; s++) {
        const float *p = part + ((size_t)s * rows + r) * ld + c;
        v += p[0];
        if constexpr (DUAL) u += p[16];
    }
    const int E = xexp[r];
    out[(size_t)r * ldo + o] = DUAL ? swiglu_out(ldexpf(v, E), ldexpf(u, E), swiglu_limit) : ldexpf(v, E);
}

template <int KIND>
static hipError_t launch_gemm_kind(const ColiGemmArgs &a, bool dual, hipStream_t st) {
    const dim3 grid((unsigned)a.n_mt * a.splits * a.rb_per_prob), block(64 * COLI_GM_W);
    const size_t shm = GmGeom<KIND>::kLds + 1024;   // the short tiles' exponents after the ring
    if (dual) hipLaunchKernelGGL((coli_gemm_tiles<KIND, true, false>), grid, block, shm, st, a);
    else if (a.segq < a.qps) hipLaunchKernelGGL((coli_gemm_tiles<KIND, false, true>), grid, block, shm, st, a);
    else hipLaunchKernelGGL((coli_gemm_tiles<KIND, false, false>), grid, block, shm, st, a);
    if (a.splits > 1) {
        const dim3 rg((a.O + 255) / 256, a.part_rows);
        if (dual)
            hipLaunchKernelGGL(coli_gemm_reduce<true>, rg, dim3(256), 0, st, a.partial, a.splits, a.part_rows,
                               a.rb_per_prob, a.O, a.xexp, a.out, a.ldo, a.swiglu_limit);
        else
            hipLaunchKernelGGL(coli_gemm_reduce<false>, rg, dim3(256), 0, st, a.partial, a.splits, a.part_rows,
                               a.rb_per_prob, a.O, a.xexp, a.out, a.ldo, 0.0f);
    }
    return hipGetLastError();
}

// rb_per_prob must cover the output rows: 8 (dual) or 16 row tiles per block.
extern "C" hipError_t coli_launch_gemm(int kind, int dual, const ColiGemmArgs *a, hipStream_t st) {
    if (a->n_mt <= 0 || a->rb_per_prob <= 0) return hipSuccess;
    if ((long)a->n_mt * a->splits * a->rb_per_prob > 0x7fffffffL || (a->prob && !a->mt_list)) return hipErrorInvalidValue;
    // a K split: output rows [0, part_rows) in fragment-row order, at most 65535 of them
    if ((a->tile != COLI_GM_ROWS && a->tile != COLI_GM_TILE) || a->splits < 1 || a->qps < 1 || a->segq < 1 || (a->segq < a->qps && (a->prob || (!a->sums && a->prob0.nrows > COLI_GM_ROWS))) || (a->splits > 1 && (!a->partial || a->xrows || a->part_rows < 1 || a->part_rows > 65535)))
        return hipErrorInvalidValue;
    switch (kind) {
    case COLI_KIND_I4_H: return launch_gemm_kind<COLI_KIND_I4_H>(*a, dual != 0, st);
    case COLI_KIND_I4_F: return launch_gemm_kind<COLI_KIND_I4_F>(*a, dual != 0, st);
    case COLI_KIND_FP4: return launch_gemm_kind<COLI_KIND_FP4>(*a, dual != 0, st);
    default: return hipErrorInvalidValue;
    }
}
