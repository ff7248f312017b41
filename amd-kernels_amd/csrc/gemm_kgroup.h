// gemm_kgroup.h -- the K loop of the small-tile GEMMs: workgroups of KG groups
// of waves, each group computing the whole BM x BN tile over its own K-tiles
// (group g takes a contiguous share), the groups' sums added through LDS at
// the end.
//
// What it is for: few rows (or few tiles), where the time is the weights'
// way from memory. A K split across workgroups pays for its partial sums
// (written, counted in and read back through the coherent level: 4 us of a
// 10 us GEMM); a split across the waves of one workgroup costs one LDS
// exchange. The groups also put two or more waves on each SIMD, so one
// wave's LDS reads, promotions and waits run under another's MFMAs without
// fragment double-buffering, and the loop stays small enough for deep rings.
//
// K-tiles are 128 bytes per row (KTile<128>; the last one may hold 64), staged with LDS-direct loads
// into an NS-stage ring per group. Groups of one wave (WM * WN == 1) need no
// barrier: a wave waits for its own loads, reads its fragments and refills
// the stage at once. Groups of several waves share one barrier per K-tile
// round; the ring then holds NS - 1 rounds in flight.
#pragma once
#include "gemm_mainloop.h"

namespace hkq {

// COLS (block-scale): the column scales differ per column (group_n 1) instead
// of per 32-column n-tile.
template <int MODE_, int WM_, int WN_, int KG_, int TM_, int TN_, int NS_, bool COLS_ = false>
struct KgCfg {
    using KT = KTile<128>;
    static constexpr int MODE = MODE_, WM = WM_, WN = WN_, KG = KG_, TM = TM_, TN = TN_, NS = NS_;
    static constexpr bool FP4 = MODE == MODE_MXFP4, BS = MODE == MODE_BLOCKSCALE, COLS = COLS_;
    static constexpr int GW = WM * WN, NW = GW * KG, THREADS = 64 * NW;
    static constexpr int BM = WM * TM * 32, BN = WN * TN * 32, ROWS = BM + BN;
    // operand loads per wave and K-tile: 8 rows of 128 bytes each
    static constexpr int LA = BM / 8 / GW, LB = BN / 8 / GW;
    // loads i and i + SWP of a wave lie a multiple of 16 rows apart: the same
    // chunk swizzle, so one lane offset serves both
    static constexpr int SWP = GW == 1 ? 2 : 1;
    static_assert(BM % (8 * GW) == 0 && BN % (8 * GW) == 0, "whole loads per wave");
    // Scales come in blocks of 4 K-tiles per row: MXFP4 32 bytes (4 x 8 e8m0,
    // rows of A and B), block-scale 16 bytes (4 scale columns of fp32, rows of
    // A). Fetching one K-tile's scale word per row would move a 64-byte sector
    // for every 4 bytes. A load ("piece") carries 32 rows, two lanes per row
    // (MXFP4; the two halves of rows with bit 3 set are swapped, so that 32
    // rows read at one offset hit distinct bank pairs) or 64 rows, one lane per
    // row. Block-scale adds one piece with the column scales: lane 4i + k holds
    // n-tile i (of the workgroup's BN / 32) in scale column k of the block. Two
    // blocks per group, by parity.
    static constexpr int SBK = 4;
    static constexpr int PA = FP4 ? BM / 32 : BS ? (BM + 63) / 64 : 0, PB = FP4 ? BN / 32 : BS && !COLS ? 1 : 0;
    static constexpr int PIECES = PA + PB, PW = (PIECES + GW - 1) / GW;
    static constexpr int SBLK = PA * 1024 + (FP4 ? PB * 1024 : PB * 256);
    static_assert(COLS || !BS || BN <= 512, "the column piece holds 16 n-tiles");
    // COLS: one fp32 per column of every K-tile, after its operand rows
    static constexpr int LC = BS && COLS ? (BN / 64 + GW - 1) / GW : 0, PC = BN / 64;
    static_assert(LC == 0 || BN % 64 == 0, "whole column-scale loads");
    static constexpr int TILE = ROWS * 128 + (LC ? BN * 4 : 0);
    static constexpr int NLD = LA + LB + LC;
    static constexpr int SC_AT = NS * KG * TILE;
    static constexpr int RING = SC_AT + 2 * KG * SBLK;
    static_assert(NS >= 2 && (NS - 1) * NLD <= 63, "vmcnt range");
    static_assert(PIECES == 0 || NS <= SBK + 1, "a block is read out before the ring's look-ahead refills its slot");
    // the sums of groups 1 .. KG-1, added by group 0
    static constexpr int RED = GW * (KG - 1) * TM * TN * 4096;
    // staging of group 0's waves (store_tile_bf16)
    static constexpr int EP = GW * TM * 32 * (TN * 64 + 16);
    static constexpr int LDS = RING > RED ? (RING > EP ? RING : EP) : (RED > EP ? RED : EP);
    static_assert(LDS <= 160 * 1024, "LDS budget of a CDNA4 CU");
};

// Where a workgroup's K-tiles come from: operand buffers of the tile's rows
// (reads at or past their extent give zero) and the lane's row offsets per
// load; the scale buffers likewise. K-tile kt adds 128 * kt to an operand
// offset; its scale column is kt >> sc_shift (MXFP4: kt), scale block B adds
// 32 * B (MXFP4 rows), 16 * B (block-scale rows) or 4 * B * bs_step
// (block-scale columns).
// GATHER: every load of A has its own lane offsets (rows through an index);
// otherwise, as for B, load i's are those of load i % SWP plus a wave-uniform
// step, which rides in the instruction's scalar offset (the range check covers
// it) and costs the loop no vector work.
template <class Cfg, bool GATHER = false>
struct KgSrc {
    static constexpr int NA = GATHER ? Cfg::LA : Cfg::SWP;
    v4i a, b, as, bs;
    uint32_t a_off[NA], b_off[Cfg::SWP];
    uint32_t a_step, b_step;  // bytes between load i and load i + SWP (linear operands)
    uint32_t s_off[Cfg::PW > 0 ? Cfg::PW : 1], c_off[Cfg::LC > 0 ? Cfg::LC : 1];
    uint32_t bs_step;
    int sc_shift;
    int KT;       // K-tiles
    // the last K-tile holds 64 bytes of K per row (linear operands): the lanes
    // that carry its upper four chunks read nothing, so the LDS holds zeros there
    bool half_tail = false;
};

__device__ __forceinline__ uint32_t clamp_bytes(int64_t n) {
    return (uint32_t)(n < 0 ? 0 : n < 0x7FFFFFFF ? n : 0x7FFFFFFF);
}

// tile row of lane `lane` in load i of wave w of a group (rows of one operand)
template <class Cfg>
__device__ __forceinline__ int kg_row(int i, int w, int lane) { return (i * Cfg::GW + w) * 8 + lane / 8; }
template <class Cfg>
__device__ __forceinline__ uint32_t kg_chunk(int r, int lane) { return (uint32_t)(Cfg::KT::load_chunk(lane, r) << 4); }
// scale piece: the lane's row of it and (MXFP4) the byte of the row's 32 that the lane carries
template <class Cfg>
__device__ __forceinline__ int kg_piece_row(int q, int lane) { return Cfg::FP4 ? q * 32 + (lane >> 1) : q * 64 + lane; }
__device__ __forceinline__ uint32_t kg_piece_half(int lane) { return (uint32_t)((lane & 1) ^ ((lane >> 4) & 1)) * 16u; }

// lds_load16 / lds_load4 with a prepared descriptor and a wave-uniform offset
// (measured on MI355X: the buffer's range check is per dword and includes it)
__device__ __forceinline__ void lds_load16_s(const v4i& desc, HKQ_LDS void* dst, uint32_t off, uint32_t soff) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(m0), "v"(off), "s"(desc), "s"(soff)
                 : "memory", "m0");
}
__device__ __forceinline__ void lds_load4_s(const v4i& desc, HKQ_LDS void* dst, uint32_t off, uint32_t soff) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :
                 : "s"(m0), "v"(off), "s"(desc), "s"(soff)
                 : "memory", "m0");
}

// The K loop. On return group 0 of the workgroup holds the sums in
// out[n-tile][m-tile], the LDS is free and every load has landed.
// wg: the wave's index in its group, kg: its group.
template <class Cfg, bool GATHER>
__device__ __forceinline__ void kgroup_kloop(const KgSrc<Cfg, GATHER>& src, HKQ_LDS uint8_t* smem, int lane, int wg, int kg,
                                             v16f (&out)[Cfg::TN][Cfg::TM]) {
    using KT = typename Cfg::KT;
    constexpr int TM = Cfg::TM, TN = Cfg::TN, NS = Cfg::NS, KG = Cfg::KG, GW = Cfg::GW, NLD = Cfg::NLD;
    constexpr int LA = Cfg::LA, LB = Cfg::LB;
    constexpr bool FP4 = Cfg::FP4, BS = Cfg::BS;
    const int wm = wg / Cfg::WN, wn = wg % Cfg::WN;
    const int khalf = lane >> 5, r = lane & 31;
    HKQ_LDS uint8_t* gbase = smem + kg * Cfg::TILE;
    HKQ_LDS uint8_t* sblk = smem + Cfg::SC_AT + kg * 2 * Cfg::SBLK;
    constexpr int STAGE = KG * Cfg::TILE;
    // this group's K-tiles
    const int k0 = kg * src.KT / KG, mine = (kg + 1) * src.KT / KG - k0;

    // OOB in the lanes that carry chunks 4 .. 7 of a row
    uint32_t upper[GATHER ? 1 : Cfg::SWP];
    if constexpr (!GATHER) {
#pragma unroll
        for (int i = 0; i < Cfg::SWP; ++i)
            upper[i] = KT::load_chunk(lane, kg_row<Cfg>(i, wg, lane)) >= 4 ? OOB : 0u;
    }
    // the loads of round t (K-tile k0 + t); past the group's last they read
    // nothing. A scale block goes out before the first K-tile that uses it, so
    // the wait for that K-tile covers it; the waits count operand loads only.
    auto issue_scales = [&](int t) {
        if constexpr (Cfg::PIECES > 0) {
            const int kt = k0 + t, c = kt >> src.sc_shift;
            if (t < mine && (t == 0 || ((c & (Cfg::SBK - 1)) == 0 && (c << src.sc_shift) == kt))) {
                const uint32_t blk = (uint32_t)c / Cfg::SBK;
                HKQ_LDS uint8_t* sl = sblk + (c / Cfg::SBK & 1) * Cfg::SBLK;
#pragma unroll
                for (int i = 0; i < Cfg::PW; ++i) {
                    const int q = i * GW + wg;
                    if (q < Cfg::PA) lds_load16_s(src.as, sl + q * 1024, src.s_off[i], blk * (FP4 ? 32u : 16u));
                    else if (FP4 && q < Cfg::PIECES) lds_load16_s(src.bs, sl + q * 1024, src.s_off[i], blk * 32u);
                    else if (q < Cfg::PIECES) lds_load4_s(src.bs, sl + q * 1024, src.s_off[i], blk * 4u * src.bs_step);
                }
            }
        }
    };
    auto issue_piece = [&](int t, int stage, int idx) {
        const int kt = k0 + t;
        const bool live = t < mine;
        HKQ_LDS uint8_t* st = gbase + stage * STAGE;
        const uint32_t kb = live ? (uint32_t)kt * 128u : OOB;
        constexpr int SWP = Cfg::SWP;
        const uint32_t tail = src.half_tail && kt == src.KT - 1 ? OOB : 0u;
        if (idx < LB) {
            const uint32_t off = GATHER ? src.b_off[idx % SWP] : src.b_off[idx % SWP] | (upper[GATHER ? 0 : idx % SWP] & tail);
            lds_load16_s(src.b, st + Cfg::BM * 128 + (idx * GW + wg) * 1024, off,
                         live ? kb + (uint32_t)(idx / SWP) * src.b_step : OOB);
        } else if (idx < LB + LA) {
            const int i = idx - LB;
            if constexpr (GATHER) lds_load16_s(src.a, st + (i * GW + wg) * 1024, src.a_off[i], kb);
            else
                lds_load16_s(src.a, st + (i * GW + wg) * 1024, src.a_off[i % SWP] | (upper[i % SWP] & tail),
                             live ? kb + (uint32_t)(i / SWP) * src.a_step : OOB);
        } else {
            const int i = idx - LB - LA, q = (i * GW + wg) % Cfg::PC;  // repeated where there are fewer loads than waves
            lds_load4_s(src.bs, st + Cfg::ROWS * 128 + q * 256, src.c_off[i],
                        live ? (uint32_t)(kt >> src.sc_shift) * src.bs_step : OOB);
        }
    };
    auto issue = [&](int t, int stage) {
        issue_scales(t);
#pragma unroll
        for (int i = 0; i < NLD; ++i) issue_piece(t, stage, i);
    };

    // fragment addresses: K-step ks of lane half h reads chunks 4h + 2ks + {0, 1}
    // as in gemm_mainloop, block-scale 4ks + 2h + {0, 1} as in blockscale_core
    // (an MFMA's own sum depends, in the last bit, on which 64 values it holds)
    uint32_t lo[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int q = 0; q < 2; ++q) lo[ks][q] = (uint32_t)KT::swz(r, BS ? 4 * ks + 2 * khalf + q : 4 * khalf + 2 * ks + q);

    v16f acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = v16f{};

    // a K-tile's operands and scales in registers
    struct Frag {
        v4i a[TM][2][2], b[TN][2][2];     // [tile][K-step][half]
        int wa[TM], wb[TN];               // MXFP4: the lane's 4 scale bytes
        float sa[TM], sbt[TN];            // block-scale: row scales, column scale of the n-tile
        v4f sb[Cfg::COLS ? TN : 1][4];    // or (COLS) of each column
    };
    // reads in the order of use: the first sub-tile's operands, then one more
    // tile of A or B at a time (piece p: B 0, A 0, A 1, ..., B 1, ...)
    constexpr int NPIECE = TM + TN;
    auto read_piece = [&](int t, int stage, Frag& f, int p) {
        const HKQ_LDS uint8_t* st = gbase + stage * STAGE;
        const bool isb = p == 0 || p > TM;
        const int i = p == 0 ? 0 : isb ? p - TM : p - 1;
        const HKQ_LDS uint8_t* base = isb ? st + (Cfg::BM + (wn * TN + i) * 32) * 128 : st + (wm * TM + i) * 32 * 128;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int q = 0; q < 2; ++q) (isb ? f.b[isb ? i : 0] : f.a[isb ? 0 : i])[ks][q] = lds_read16(base + lo[ks][q]);
        // the scales of a round past the group's last one are stale, those of a
        // half last K-tile's upper blocks the next row's: zeros
        const bool live = t < mine && !(FP4 && src.half_tail && k0 + t == src.KT - 1 && khalf);
        if constexpr (FP4) {
            const int kt = k0 + t;
            const HKQ_LDS uint8_t* sl = sblk + ((kt / Cfg::SBK) & 1) * Cfg::SBLK + r * 32 +
                                        ((((kt >> 1) & 1) ^ ((r >> 3) & 1)) << 4) + (kt & 1) * 8 + khalf * 4;
            const int w = *reinterpret_cast<const HKQ_LDS int*>(sl + (isb ? Cfg::PA + wn * TN + i : wm * TM + i) * 1024);
            if (isb) f.wb[i] = live ? w : 0;
            else f.wa[i] = live ? w : 0;
        }
        if constexpr (BS) {
            const int c = (k0 + t) >> src.sc_shift;
            const HKQ_LDS uint8_t* blk = sblk + ((c / Cfg::SBK) & 1) * Cfg::SBLK;
            if (!isb) {
                const float v = *reinterpret_cast<const HKQ_LDS float*>(blk + ((wm * TM + i) * 32 + r) * 16 + (c & 3) * 4);
                f.sa[i] = live ? v : 0.0f;
            } else if constexpr (Cfg::COLS) {
                const HKQ_LDS float* cs = reinterpret_cast<const HKQ_LDS float*>(st + Cfg::ROWS * 128);
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    f.sb[i][g] = *reinterpret_cast<const HKQ_LDS v4f*>(cs + (wn * TN + i) * 32 + 8 * g + 4 * khalf);
            } else {
                const float v = *reinterpret_cast<const HKQ_LDS float*>(blk + Cfg::PA * 1024 + ((wn * TN + i) * 4 + (c & 3)) * 4);
                f.sbt[i] = live ? v : 0.0f;
            }
        }
    };
    auto fp8 = [](const v4i (&f)[2]) { return __builtin_shufflevector(f[0], f[1], 0, 1, 2, 3, 4, 5, 6, 7); };
    // the MFMAs of a K-tile; between(s) after those of sub-tile s
    auto mma = [&](const Frag& f, auto between) {
        v16f P, Pq;
#pragma unroll
        for (int s = 0; s < TN * TM; ++s) {
            const int i = s / TM, j = s % TM;
            if constexpr (BS) {
                P = mfma_sel<false, 0, 0>(fp8(f.b[i][0]), fp8(f.a[j][0]), v16f{}, 127, 127);
                P = mfma_sel<false, 0, 0>(fp8(f.b[i][1]), fp8(f.a[j][1]), P, 127, 127);
            } else if constexpr (FP4) {
                const v4i z = v4i{0, 0, 0, 0};
                auto op = [&](const v4i& x) { return __builtin_shufflevector(x, z, 0, 1, 2, 3, 4, 5, 6, 7); };
                acc[i][j] = mfma_sel<true, 0, 0>(op(f.b[i][0][0]), op(f.a[j][0][0]), acc[i][j], f.wb[i], f.wa[j]);
                acc[i][j] = mfma_sel<true, 1, 1>(op(f.b[i][0][1]), op(f.a[j][0][1]), acc[i][j], f.wb[i], f.wa[j]);
                acc[i][j] = mfma_sel<true, 2, 2>(op(f.b[i][1][0]), op(f.a[j][1][0]), acc[i][j], f.wb[i], f.wa[j]);
                acc[i][j] = mfma_sel<true, 3, 3>(op(f.b[i][1][1]), op(f.a[j][1][1]), acc[i][j], f.wb[i], f.wa[j]);
            } else if constexpr (Cfg::MODE == MODE_BF16) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int q = 0; q < 2; ++q) acc[i][j] = mfma_bf16(f.b[i][ks][q], f.a[j][ks][q], acc[i][j]);
            } else {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
                    acc[i][j] = mfma_sel<false, 0, 0>(fp8(f.b[i][ks]), fp8(f.a[j][ks]), acc[i][j], 127, 127);
            }
            // block-scale: promote the previous sub-tile while the matrix pipe
            // works on this one (the last one after the loop)
            auto promote = [&](int q, const v16f& X) {
                const int pi = q / TM, pj = q % TM;
                const float fs = f.sa[pj] * f.sbt[pi];
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    acc[pi][pj][e] =
                        __builtin_fmaf(X[e], Cfg::COLS ? f.sa[pj] * f.sb[Cfg::COLS ? pi : 0][e >> 2][e & 3] : fs, acc[pi][pj][e]);
            };
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (BS) {
                if (s > 0) promote(s - 1, Pq);
                Pq = P;
            }
            between(s);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (BS)
                if (s == TN * TM - 1) promote(s, P);
        }
    };

    if constexpr (GW == 1) {
        // private ring: NS rounds requested ahead; a stage is refilled as soon
        // as its fragments are in registers
#pragma unroll
        for (int s = 0; s < NS; ++s) issue(s, s);
        int stage = 0;
        for (int t = 0; t < mine; ++t) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * NLD) : "memory");
            Frag f;
#pragma unroll
            for (int p = 0; p < NPIECE; ++p) read_piece(t, stage, f, p);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(t + NS, stage);
            mma(f, [](int) {});
            stage = stage + 1 == NS ? 0 : stage + 1;
        }
    } else {
        // one barrier per round: round t + 1 resident, every wave's fragments of
        // round t in registers (read during round t - 1), so its stage takes
        // round t + NS while the MFMAs of round t run between the reads of
        // round t + 1
        const int rounds = (src.KT + KG - 1) / KG;
#pragma unroll
        for (int s = 0; s < NS; ++s) issue(s, s);
        tile_barrier<(NS - 1) * NLD>();
        Frag f[2];
#pragma unroll
        for (int p = 0; p < NPIECE; ++p) read_piece(0, 0, f[0], p);
        int stage = 0;
        auto round = [&](int t, const Frag& cur, Frag& nxt) {
            const int next = stage + 1 == NS ? 0 : stage + 1;
            tile_barrier<(NS - 2) * NLD>();
            issue_scales(t + NS);
            mma(cur, [&](int s) {
#pragma unroll
                for (int i = s * NLD / (TN * TM); i < (s + 1) * NLD / (TN * TM); ++i) issue_piece(t + NS, stage, i);
#pragma unroll
                for (int p = s * NPIECE / (TN * TM); p < (s + 1) * NPIECE / (TN * TM); ++p) read_piece(t + 1, next, nxt, p);
            });
            stage = next;
        };
        int t = 0;
        for (; t + 1 < rounds; t += 2) {
            round(t, f[0], f[1]);
            round(t + 1, f[1], f[0]);
        }
        if (t < rounds) round(t, f[0], f[1]);
    }
    mfma_drain();
    tile_barrier<0>();  // no load in flight, every wave past its reads: the LDS takes the sums

    if constexpr (KG == 1) {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) out[i][j] = acc[i][j];
    } else {
        HKQ_LDS v4f* red = reinterpret_cast<HKQ_LDS v4f*>(smem);
        auto slot = [&](int from) { return red + ((from - 1) * GW + wg) * (TM * TN * 4 * 64) + lane; };
        if (kg != 0) {
            HKQ_LDS v4f* d = slot(kg);
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const v16f& v = acc[i][j];
                        d[((i * TM + j) * 4 + g) * 64] = v4f{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
                    }
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const v16f& o = acc[i][j];
                        v4f v = v4f{o[4 * g], o[4 * g + 1], o[4 * g + 2], o[4 * g + 3]};
#pragma unroll
                        for (int from = 1; from < KG; ++from) v = v + slot(from)[((i * TM + j) * 4 + g) * 64];
#pragma unroll
                        for (int e = 0; e < 4; ++e) out[i][j][4 * g + e] = v[e];
                    }
        }
        __syncthreads();  // the sums are read: the LDS takes the epilogue's staging
    }
}

// Tile of a grouped (MoE) GEMM whose experts hold `routed` rows in all, by the
// mean rows per expert r (the counts themselves are on the GPU). The tiles of
// the MoE kernels have one K group: they add K-tile after K-tile in K order, as
// the block-pair kernels do, so every tile size and both weight layouts give
// the same bits. Bound by the weights' way from HBM: a tile's rows should hold
// an expert's rows, and the rings of the workgroups of a CU 120 to 150 KB of
// K-tiles in flight. Beyond about one routing block per expert (`pairs_short`,
// `pairs_long` rows, for K up to 3072 and above) the block-pair kernels read
// the weights once for 256 rows and win.
// Measured on MI355X (us, gate/up and down together), block-scale, 8 experts of
// 4096 x 14336; 64 x 64 tiles on 4 waves, 64 x 128 on 8, 128 x 128, 128 x 256,
// pairs: r = 0: 85 / 90 / 123 / 149 / 155; 2: 258 / 265 / 288 / 355 / 400; 16: 275
// / 281 / 311 / 367 / 416; 37: 290 / 287 / 324 / 372 / 431; 55: 347 / 340 / 326 /
// 375 / 441; 75: 489 / 462 / 349 / 386 / 459; 125: 593 / 611 / 470 / 425 / 494;
// 225: 853 / 752 / 601 / 521 / 557. With a short K (32 experts of 2048 x 2816) the
// wide tile's fewer, longer rows win: r = 1: 69 / 66 / 96 / 78 / 86; 12: 109 / 105 /
// 140 / 129 / 131; 50: 124 / 123 / 146 / 136 / 140; 112: 219 / 206 / 178 / 160 / 160.
//
// A tile of fewer than 128 rows covers a routing block in row groups, each a
// workgroup of its own: the grid holds the first groups of all blocks, then the
// second ones (most of them empty: they end after two loads). A skewed routing's
// full blocks then run their groups side by side instead of streaming the
// weights once per group in series (64 x 64 tiles; block-scale, 8 experts of 4096
// x 14336, half of the rows on one expert, 90 tokens 315 -> 302 us, 150 tokens 354
// -> 340; MXFP4 down projection, 150 tokens 73 -> 49), and an even one loses less
// than 1 %.
//
// A short K's 64 x 128 tiles that give the CUs no more than one round of two get
// a second one from the experts with more than 64 rows: they end at `rows_short`
// mean rows there (block-scale down projection of 32 experts, K 2816, N 2048,
// 400 tokens: r = 50, 43.0 us on 64 x 128, 36.5 on 128 x 256, pairs 38.1).
enum MoeTile { MOET_64x64, MOET_64x128, MOET_128x128, MOET_128x256, MOET_PAIRS };
// workgroups (at most 512 threads each) of the widest small-tile grid: within
// what one launch can hold
inline bool kg_moe_grid(int64_t grid_m, int64_t N) { return grid_m * ((N + 63) / 64) * 2 < (1ll << 23); }
inline MoeTile moe_tile(int64_t routed, int64_t experts, int64_t N, int64_t K, int64_t ncu, int64_t rows_short,
                        int64_t pairs_short, int64_t pairs_long) {
    const int64_t r = routed / (experts > 0 ? experts : 1);
    if (K <= 3072) {
        const bool one_round = experts * ((N + 127) / 128) <= 2 * ncu;
        return r <= (one_round ? rows_short : 52) ? MOET_64x128 : r <= pairs_short ? MOET_128x256 : MOET_PAIRS;
    }
    if (r <= 48) return MOET_64x64;
    return r > pairs_long ? MOET_PAIRS : r <= 112 ? MOET_128x128 : MOET_128x256;
}

}  // namespace hkq
