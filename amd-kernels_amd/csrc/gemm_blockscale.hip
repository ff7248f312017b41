// gemm_blockscale.hip -- FP8 GEMM with per-K-group fp32 scales (DeepSeek-V3
// style), restating gemm-basic/gemm_a8w8_blockscale/kernel.cpp:129-153 (and
// the formula of gemm_a8w8_blockscale/test_parity.py:57-76):
//
//   C[m, n] = bf16( sum_g (A_g . B_g^T)[m, n] * sa[m, g] * sb[g, n / GN] ),
//   g = 128-wide K group, GN = 128 (128x128 weight blocks) or 1 (per column,
//   the layout of the reference test: b_scale [K/128, N]).
//
// fp32 scales cannot ride in the MFMA's e8m0 scale operands, so every K group
// is "promoted" on the VALU: per 32x32 sub-tile two chained MFMAs (the group's
// two 64-deep K-steps) produce a fresh partial P, then acc += P * sa * sb.
// Large products run the 8-wave K loop of blockscale_core.h over 256 x 256
// tiles, fewer rows smaller tiles with K split over the workgroup's waves
// (gemm_kgroup.h), and a few rows of short K stream the weights through
// registers (blockscale_narrow_kernel).
#include <cstdlib>

#include "blockscale_core.h"
#include "gemm_kgroup.h"
#include "hkq_host.h"

namespace hkq {

struct BlockScaleParams {
    const uint8_t* A;
    const uint8_t* B;
    uint16_t* C;
    const float* sa;  // [M, lsa]: column g = K group
    const float* sb;  // [K/128, lsb]: column n/128 (GN 128) or n (GN 1)
    int M, N, K;
    int64_t lda, ldb, ldc, lsa, lsb;
    int tiles_m, tiles_n, group_m, c16;
    // multiply-add epilogue C = ca * GEMM + cb, ca / cb bf16 [M, ldca] / [M, ldcb]
    // (nullptr: plain GEMM)
    const uint16_t* ca;
    const uint16_t* cb;
    int64_t ldca, ldcb;
};

// Multiply-add epilogue hook: v -> ca[m, n] * v + cb[m, n] on the fp32 sums.
// prefetch(i) loads the lane's 4 x TM groups of 4 bf16 of both operands for
// n-tile i in one batch (rows past M / columns past N: ca = 1, cb = 0).
template <int TM>
struct MulAddElem {
    const uint16_t *ca, *cb;
    int64_t ldca, ldcb;
    int M, N, mw, nw, lane;
    uint2 a[4][TM], b[4][TM];
    __device__ void prefetch(int i) {
        const int m0 = mw + (lane & 31), n0 = nw + i * 32 + 4 * (lane >> 5);
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int m = m0 + j * 32, n = n0 + 8 * g;
                const bool in = m < M && n < N;
                a[g][j] = in ? *reinterpret_cast<const uint2*>(ca + (int64_t)m * ldca + n) : make_uint2(0x3F803F80u, 0x3F803F80u);
                b[g][j] = in ? *reinterpret_cast<const uint2*>(cb + (int64_t)m * ldcb + n) : make_uint2(0u, 0u);
            }
    }
    __device__ float4 operator()(int j, int, int g, float4 v) const {
        const uint2 x = a[g][j], y = b[g][j];
        return make_float4(bf16_to_f32(x.x & 0xFFFF) * v.x + bf16_to_f32(y.x & 0xFFFF),
                           bf16_to_f32(x.x >> 16) * v.y + bf16_to_f32(y.x >> 16),
                           bf16_to_f32(x.y & 0xFFFF) * v.z + bf16_to_f32(y.y & 0xFFFF),
                           bf16_to_f32(x.y >> 16) * v.w + bf16_to_f32(y.y >> 16));
    }
};

// Tiled kernel: the 8-wave K loop of blockscale_core.h over 256 x BN tiles.
// BN 256: waves of 64 x 128 (two per SIMD). BN 224, for grids that the
// 256-wide tiles would leave a CU short (2048 x 7168: 224 tiles of 256 x 256,
// 256 of 256 x 224): waves 0-3 take n-tiles 0-3 and waves 4-7 n-tiles 4-6 of
// their 64 rows, so that each SIMD holds one wave of each kind (the hardware
// places wave w on SIMD w % 4) and does 7/8 of a 256-wide tile's work; the B
// rows past 224 read zero. Scale slot: sa of the tile's 256 rows; sb GN 1 or
// BN 224: one value per tile column (GN 128: its block's), GN 128 with BN
// 256: the tile's two column blocks.
template <bool GN1, int BN>
__global__ __launch_bounds__(64 * BS_NW, 1) void blockscale_gemm_kernel(const BlockScaleParams p) {
    static_assert(BN == BS_BN || BN == BS_BN - 32, "tile widths of 256 or 224 columns");
    constexpr bool W224 = BN != BS_BN;
    constexpr int TM = BS_TM, TN = BS_TN, NW = BS_NW;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem_raw[];
    HKQ_LDS uint8_t* smem = (HKQ_LDS uint8_t*)smem_raw;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = W224 ? wave & 3 : wave / BS_WN, wn = W224 ? wave >> 2 : wave % BS_WN;

    int tm, tn;
    tile_coords(blockIdx.x, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    const int m0 = tm * BS_BM, n0 = tn * BN;
    const int rows_a = min(p.M - m0, BS_BM), rows_b = min(p.N - n0, BN);

    // LDS-direct loads: load i of a wave fills rows (i*NW + wave)*8 .. +7 of
    // its operand tile
    uint32_t a_off[BS_LA], b_off[BS_LB];
#pragma unroll
    for (int i = 0; i < BS_LA; ++i) a_off[i] = dense_row_off<NW, BS_KT>(i, wave, lane, p.lda);
#pragma unroll
    for (int i = 0; i < BS_LB; ++i) b_off[i] = dense_row_off<NW, BS_KT>(i, wave, lane, p.ldb);
    const uint8_t* a_src = p.A + (int64_t)m0 * p.lda;
    const uint8_t* b_src = p.B + (int64_t)n0 * p.ldb;
    // extents end with the last row's bytes: whatever the pitch, an offset past
    // the tile's rows that wraps at 32 bits stays inside the operand
    const int64_t a_bytes = min((int64_t)(rows_a - 1) * p.lda + p.K, (int64_t)0x7FFFFFFF);
    const int64_t b_bytes = min((int64_t)(rows_b - 1) * p.ldb + p.K, (int64_t)0x7FFFFFFF);
    // scales: sa rows (wave & 3) * 64 + lane; sb per column: tile column c =
    // (wave & 3)*64 + lane from sb's row of the K-tile (GN 128: its block's
    // value), per block (GN 128, BN 256): blocks n0/128 + {0, 1}. Waves 4-7
    // repeat the loads of 0-3 so that every wave issues the same loads.
    const float* sa_src = p.sa + (int64_t)m0 * p.lsa;
    const int64_t sa_bytes = min(((int64_t)(rows_a - 1) * p.lsa + p.K / 128) * 4, (int64_t)0x7FFFFFFF);
    const uint32_t sa_off = (uint32_t)(((wave & 3) * 64 + lane) * p.lsa * 4);
    constexpr bool PER_COL = GN1 || W224;
    const int sb_row = GN1 ? p.N : (p.N + 127) / 128;  // values per sb row
    const int sc = (wave & 3) * 64 + lane;
    const uint32_t sb_off = PER_COL ? (sc < rows_b ? (uint32_t)((GN1 ? n0 + sc : (n0 + sc) / 128) * 4) : OOB)
                                    : (lane < 2 ? (uint32_t)((n0 / 128 + lane) * 4) : OOB);
    const uint32_t lds_base = (uint32_t)(uintptr_t)smem;
    const int KTN = p.K / BS_KT;

    // load q (0 .. BS_NLD-1) of K-tile kt: A, B, then the sa and sb scales
    auto issue = [&](int kt, int q) {
        const bool live = kt < KTN;
        const uint32_t kb = (uint32_t)(kt * BS_KT);
        const int st = kt & 1;
        if (q < BS_LA + BS_LB) {
            HKQ_LDS uint8_t* dst = reinterpret_cast<HKQ_LDS uint8_t*>((uintptr_t)(lds_base + bs_load_dst(st, q, wave)));
            if (q < BS_LA)
                lds_load16(a_src + kb, live ? (uint32_t)(a_bytes - kb) : 0u, dst, a_off[q]);
            else
                lds_load16(b_src + kb, live ? (uint32_t)(b_bytes - kb) : 0u, dst, b_off[q - BS_LA]);
        } else {
            HKQ_LDS uint8_t* slot = smem + BS_SC + st * BS_SLOT;
            if (q == BS_LA + BS_LB)
                lds_load4(sa_src + kt, live ? (uint32_t)(sa_bytes - kt * 4) : 0u, slot + (wave & 3) * 256, sa_off);
            else
                lds_load4(p.sb + (int64_t)kt * p.lsb, live ? (uint32_t)(sb_row * 4) : 0u,
                          slot + 1024 + (PER_COL ? (wave & 3) * 256 : 0), sb_off);
        }
    };

    v16f acc[TN][TM];
    constexpr int SBM = GN1 ? BS_SB_COL : W224 ? BS_SB_NTILE : BS_SB_WAVE;
    if (W224 && wn == 1) {
        bs8_kloop<SBM, TN - 1>(smem, lane, wm, TN * 32, KTN, issue, reinterpret_cast<v16f(&)[TN - 1][TM]>(acc));
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[TN - 1][j] = v16f{};
    } else
        bs8_kloop<SBM, TN>(smem, lane, wm, wn * TN * 32, KTN, issue, acc);

    // BN 224: the last n-tile of waves 4-7 lies past the tile (never stored)
    const int mw = m0 + wm * TM * 32, nw = n0 + wn * TN * 32;
    const int n_end = W224 ? min(p.N, n0 + BN) : p.N;
    auto one = [](int) { return 1.0f; };
    auto ones = [](int, int) { return make_float4(1.f, 1.f, 1.f, 1.f); };
    if (p.ca) {
        MulAddElem<TM> e;
        e.ca = p.ca;
        e.cb = p.cb;
        e.ldca = p.ldca;
        e.ldcb = p.ldcb;
        e.M = p.M;
        e.N = n_end;
        e.mw = mw;
        e.nw = nw;
        e.lane = lane;
        store_tile_bf16<TM, TN>(acc, smem, wave, lane, p.C, p.ldc, p.M, n_end, mw, nw, p.c16 != 0, one, ones, NoBias{}, e);
    } else {
        store_tile_bf16<TM, TN>(acc, smem, wave, lane, p.C, p.ldc, p.M, n_end, mw, nw, p.c16 != 0, one, ones, NoBias{});
    }
}

// ---------------------------------------------------------------------------
// Narrow M (M <= 16): the streaming layout of the dense GEMMs' narrow path
// (workgroup = 16*NT columns for all rows, 4 waves splitting K, fragments
// loaded straight into registers for the 16x16x128 MFMA; lane l supplies row
// l % 16, bytes [16q, 16q+16) and [64+16q, 64+16q+16) of the step, q = l/16,
// and holds D[4q + i][l % 16]). A 128-value K-step is exactly one scale
// group, so each step's MFMA starts from zero and is promoted at once:
// acc += P * sa[m, g] * sb[g, n / GN].
constexpr int BSN_WAVES = 4, BSN_MAX_M = 16;

template <bool GN1, int NT>
struct BsNarrowFrag {
    v4i b0[NT], b1[NT], a0, a1;
    float sa;                    // sa[m, g] of the lane's row
    float sb[NT][GN1 ? 4 : 1];   // sb[g, n] of the lane's 4 columns (GN 1) or of the tile's column block
};

template <bool GN1, int NT>
__global__ __launch_bounds__(64 * BSN_WAVES) void blockscale_narrow_kernel(const BlockScaleParams p) {
    constexpr int DEPTH = NT == 1 ? 6 : 4;
    __shared__ v4f red[BSN_WAVES][NT][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16 * NT;
    const int S = p.K / 128;
    const int s0 = wave * S / BSN_WAVES, s1 = (wave + 1) * S / BSN_WAVES;
    const int rows_b = min(16 * NT, p.N - n0);
    const auto rb = make_rsrc(p.B + (int64_t)n0 * p.ldb, (uint32_t)(rows_b * p.ldb));
    const auto ra = make_rsrc(p.A, (uint32_t)(p.M * p.lda));
    // scales: rows of sa past M and groups past S read zero
    const auto rsa = make_rsrc(p.sa, (uint32_t)(((int64_t)(p.M - 1) * p.lsa + S) * 4));
    const auto rsb = make_rsrc(p.sb, (uint32_t)(((int64_t)(S - 1) * p.lsb + (GN1 ? p.N : (p.N + 127) / 128)) * 4));
    const uint32_t a_off = (uint32_t)(r * p.lda + 16 * q);
    const uint32_t sa_row = r < p.M ? (uint32_t)(r * p.lsa) * 4 : OOB;
    uint32_t b_off[NT], sb_col[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        b_off[i] = (uint32_t)((i * 16 + r) * p.ldb + 16 * q);
        sb_col[i] = (uint32_t)(GN1 ? n0 + 16 * i + 4 * q : (n0 + 16 * i) / 128) * 4;
    }

    auto load = [&](int s, BsNarrowFrag<GN1, NT>& f) {
        const uint32_t kill = s < s1 ? 0u : OOB;
        const uint32_t kb = (uint32_t)s * 128 | kill;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            f.b0[i] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_off[i] + kb, 0, 0);
            f.b1[i] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_off[i] + kb + 64, 0, 0);
        }
        f.a0 = __builtin_amdgcn_raw_buffer_load_b128(ra, a_off + kb, 0, 0);
        f.a1 = __builtin_amdgcn_raw_buffer_load_b128(ra, a_off + kb + 64, 0, 0);
        f.sa = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, (sa_row + 4 * (uint32_t)s) | kill, 0, 0));
        const uint32_t srow = ((uint32_t)s * (uint32_t)p.lsb * 4) | kill;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int e = 0; e < (GN1 ? 4 : 1); ++e)
                f.sb[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsb, srow + sb_col[i] + 4 * e, 0, 0));
    };
    v4f acc[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
    auto mma = [&](const BsNarrowFrag<GN1, NT>& f) {
        const v8i b = v8i{f.a0[0], f.a0[1], f.a0[2], f.a0[3], f.a1[0], f.a1[1], f.a1[2], f.a1[3]};
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const v8i a = v8i{f.b0[i][0], f.b0[i][1], f.b0[i][2], f.b0[i][3],
                              f.b1[i][0], f.b1[i][1], f.b1[i][2], f.b1[i][3]};
            const v4f P =
                __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 127, 0, 127);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[i][e] = __builtin_fmaf(P[e], f.sa * f.sb[i][GN1 ? e : 0], acc[i][e]);
        }
    };
    BsNarrowFrag<GN1, NT> f[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(s0 + d, f[d]);
    for (int s = s0; s < s1; s += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            mma(f[d]);
            load(s + d + DEPTH, f[d]);
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) red[wave][i][lane] = acc[i];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int n = n0 + 16 * i + 4 * q, m = r;
        if (n >= p.N || m >= p.M) continue;  // N % 4 == 0: n .. n+3 all in or all out
        v4f v = red[0][i][lane];
#pragma unroll
        for (int w = 1; w < BSN_WAVES; ++w) v += red[w][i][lane];
        if (p.ca) {
            const uint2 x = *reinterpret_cast<const uint2*>(p.ca + (int64_t)m * p.ldca + n);
            const uint2 y = *reinterpret_cast<const uint2*>(p.cb + (int64_t)m * p.ldcb + n);
            v = v4f{bf16_to_f32(x.x & 0xFFFF) * v[0] + bf16_to_f32(y.x & 0xFFFF),
                    bf16_to_f32(x.x >> 16) * v[1] + bf16_to_f32(y.x >> 16),
                    bf16_to_f32(x.y & 0xFFFF) * v[2] + bf16_to_f32(y.y & 0xFFFF),
                    bf16_to_f32(x.y >> 16) * v[3] + bf16_to_f32(y.y >> 16)};
        }
        *reinterpret_cast<v2i*>(p.C + (int64_t)m * p.ldc + n) = v2i{(int)pk_bf16(v[0], v[1]), (int)pk_bf16(v[2], v[3])};
    }
}

// 32-bit offsets of the streaming kernel: 16 activation rows, 32 weight rows and
// the scales
static bool bs_narrow_fits(const BlockScaleParams& p) {
    auto reach = [](int64_t rows, int64_t ld) { return ld <= 0x7FFFFFFF / rows; };
    return reach(32, p.ldb) && reach(BSN_MAX_M, p.lda) && reach(4 * BSN_MAX_M, p.lsa) && reach(8 * (p.K / 128), p.lsb);
}

// 16-column (NT = 1) or 32-column (NT = 2, when N/16 workgroups exceed the
// CUs) slices.
template <bool GN1>
static int launch_blockscale_narrow(const BlockScaleParams& p, hipStream_t stream) {
    const int64_t ncu = cu_count() > 0 ? cu_count() : 256;
    const int64_t wgs16 = (p.N + 15) / 16;
    if (wgs16 > ncu)
        blockscale_narrow_kernel<GN1, 2><<<dim3((unsigned)((p.N + 31) / 32)), 64 * BSN_WAVES, 0, stream>>>(p);
    else
        blockscale_narrow_kernel<GN1, 1><<<dim3((unsigned)wgs16), 64 * BSN_WAVES, 0, stream>>>(p);
    return hkq_launch_status();
}

// ---------------------------------------------------------------------------
// Small tiles (gemm_kgroup.h): 32 x 32 .. 128 x 256, chosen by bs_plan below.
// Bound by the weights' way from memory where the tiles fill the CUs once
// (measured on MI355X: with its MFMAs taken out, 24 x 7168 x 18432 runs as
// long as with them), and from 128 x 64 up by the wave's own chain of LDS
// reads, MFMAs and promotions (0.32, 0.56 and 0.82 us per K-tile of 128 x 64,
// 128 x 128 and 128 x 256 against 0.24, 0.41 and 0.55 for the loads alone).
// Against the 256 x 256 tiles (or, up to 192 rows, the 16-column streaming
// kernel in groups of 64 rows) that served these shapes before: 24x7168x18432
// 46.0 -> 29 us, 64x2112x7168 26.6 -> 8.7, 500x7168x2048 25.3 -> 13.7,
// 256x7168x18432 299 -> 73, 1024x7168x18432 276 -> 152.
template <class Cfg, bool GN1>
__global__ __launch_bounds__(Cfg::THREADS, 1) void blockscale_tile_kernel(const BlockScaleParams p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem_raw[];
    HKQ_LDS uint8_t* smem = (HKQ_LDS uint8_t*)smem_raw;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, TN = Cfg::TN, TM = Cfg::TM;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wg = wave % Cfg::GW, kg = wave / Cfg::GW;
    int tm, tn;
    tile_coords(blockIdx.x, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int rows_a = min(p.M - m0, BM), rows_b = min(p.N - n0, BN);
    const int S = p.K / 128;

    KgSrc<Cfg> src;
    src.a = buffer_desc(p.A + (int64_t)m0 * p.lda, clamp_bytes((int64_t)rows_a * p.lda));
    src.b = buffer_desc(p.B + (int64_t)n0 * p.ldb, clamp_bytes((int64_t)rows_b * p.ldb));
    src.as = buffer_desc(p.sa + (int64_t)m0 * p.lsa, clamp_bytes(((int64_t)(rows_a - 1) * p.lsa + S) * 4));
    src.bs = buffer_desc(p.sb, clamp_bytes(((int64_t)(S - 1) * p.lsb + (GN1 ? p.N : (p.N + 127) / 128)) * 4));
    src.bs_step = (uint32_t)p.lsb * 4u;
    src.sc_shift = 0;
    src.KT = S;
#pragma unroll
    for (int i = 0; i < Cfg::SWP; ++i) {
        const int r = kg_row<Cfg>(i, wg, lane);
        src.a_off[i] = (uint32_t)(r * p.lda) + kg_chunk<Cfg>(r, lane);
        src.b_off[i] = (uint32_t)(r * p.ldb) + kg_chunk<Cfg>(r, lane);
    }
    src.a_step = (uint32_t)(8 * Cfg::GW * Cfg::SWP * p.lda);
    src.b_step = (uint32_t)(8 * Cfg::GW * Cfg::SWP * p.ldb);
    // scale pieces: 64 rows of sa each, then (one scale per 128 columns) the
    // n-tiles' column scales; n-tiles past N repeat the last one
#pragma unroll
    for (int i = 0; i < Cfg::PW; ++i) {
        const int q = i * Cfg::GW + wg;
        const int r = kg_piece_row<Cfg>(q, lane);
        src.s_off[i] = q < Cfg::PA ? (r < rows_a ? (uint32_t)(r * p.lsa) * 4u : OOB)
                                   : (uint32_t)(min(n0 + (lane >> 2) * 32, p.N - 1) / 128) * 4u + (uint32_t)(lane & 3) * src.bs_step;
    }
#pragma unroll
    for (int i = 0; i < Cfg::LC; ++i) {
        const int c = ((i * Cfg::GW + wg) % Cfg::PC) * 64 + lane;
        src.c_off[i] = c < rows_b ? (uint32_t)(n0 + c) * 4u : OOB;
    }

    v16f acc[TN][TM];
    kgroup_kloop<Cfg>(src, smem, lane, wg, kg, acc);
    if (kg != 0) return;

    const int mw = m0 + wg / Cfg::WN * TM * 32, nw = n0 + wg % Cfg::WN * TN * 32;
    auto one = [](int) { return 1.0f; };
    auto ones = [](int, int) { return make_float4(1.f, 1.f, 1.f, 1.f); };
    if (p.ca) {
        MulAddElem<TM> e;
        e.ca = p.ca;
        e.cb = p.cb;
        e.ldca = p.ldca;
        e.ldcb = p.ldcb;
        e.M = p.M;
        e.N = p.N;
        e.mw = mw;
        e.nw = nw;
        e.lane = lane;
        store_tile_bf16<TM, TN>(acc, smem, wg, lane, p.C, p.ldc, p.M, p.N, mw, nw, p.c16 != 0, one, ones, NoBias{}, e);
    } else {
        store_tile_bf16<TM, TN>(acc, smem, wg, lane, p.C, p.ldc, p.M, p.N, mw, nw, p.c16 != 0, one, ones, NoBias{});
    }
}

template <class Cfg, bool GN1>
static int launch_blockscale_tile(BlockScaleParams& p, hipStream_t stream) {
    auto kern = blockscale_tile_kernel<Cfg, GN1>;
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS);
        if (e != hipSuccess) {
            set_error("hipFuncSetAttribute(MaxDynamicSharedMemorySize=%d) failed: %s", Cfg::LDS, hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    p.tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;
    p.tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    if (p.group_m <= 0) p.group_m = 8;
    p.c16 = (p.ldc % 8 == 0) && (reinterpret_cast<uintptr_t>(p.C) % 16 == 0);
    kern<<<dim3((unsigned)(p.tiles_m * p.tiles_n)), Cfg::THREADS, Cfg::LDS, stream>>>(p);
    return hkq_launch_status();
}

template <bool GN1, int BN>
static int launch_blockscale_bn(BlockScaleParams& p, hipStream_t stream) {
    constexpr int BM = BS_BM, LDS = BS_LDS;
    auto kern = blockscale_gemm_kernel<GN1, BN>;
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) {
            set_error("hipFuncSetAttribute(MaxDynamicSharedMemorySize=%d) failed: %s", LDS, hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    if (p.group_m <= 0) p.group_m = 8;
    p.c16 = (p.ldc % 8 == 0) && (reinterpret_cast<uintptr_t>(p.C) % 16 == 0);
    const int64_t nblk = (int64_t)p.tiles_m * p.tiles_n;
    if (nblk == 0) return 0;
    kern<<<dim3((unsigned)nblk), 64 * BS_NW, LDS, stream>>>(p);
    return hkq_launch_status();
}

// Tile size of a block-scale GEMM: the least estimated time,
//   rounds of tiles over the CUs * (K-tiles * us per K-tile + 2.3 us) + 2.3 us,
// with the us per K-tile measured on MI355X as the mean of operands that lie
// in the last-level cache (N, K = 2112, 7168 and 7168, 2048: 0.05, 0.12, 0.17,
// 0.32, 0.56, 0.82, 1.3 in the order below) and in HBM (7168, 18432: 0.15,
// 0.26, 0.33, 0.5, 0.67, 1.03, 1.9). It picks the fastest size at 24 .. 2048
// rows of those shapes and of 24576, 1536 (the runner-up within 6% in all but
// the clear cases). With one scale per column a 128 x 128 K-tile takes 0.66:
// from there the 256-row tiles win where the CUs hold one round of them (1024 x
// 7168 x 18432 204 against 218, 1536 x 4096 x 4096 50.5 against 53.9).
// 224-column tiles of 256 rows do 7/8 of a 256-column tile's work (they fill
// CUs that 256 columns leave idle: 2048 x 7168 is 224 tiles of 256 columns, 256
// of 224). Column scales per column (GN 1) need 64 columns for a whole load and
// leave 128 x 256 no registers.
// HKQ_BLOCKSCALE_W224=0 (read at each call) keeps 256-column tiles.
enum BsTile { BST_32x32, BST_32x64, BST_64x64, BST_128x64, BST_128x128, BST_128x256, BST_256x256, BST_256x224, BST_COUNT,
              BST_NONE  // rows too far apart for every size
};
static int bs_plan(const BlockScaleParams& p, bool gn1) {
    const int64_t M = p.M, N = p.N, K = p.K;
    // Rows `ld` bytes apart that a 32-bit buffer offset reaches: all of a small
    // tile's, the live ones of a 256-row tile (whose extents end with the last)
    auto reach = [](int64_t rows, int64_t ld) { return ld <= 0x7FFFFFFF / rows; };
    auto fits = [&](int t, int64_t bm, int64_t bn) {
        if (t >= BST_256x256) bm = std::min<int64_t>(M, bm), bn = std::min<int64_t>(N, bn);
        return reach(bm, p.lda) && reach(bn, p.ldb) && reach(4 * bm, p.lsa) &&
               (t >= BST_256x256 || reach(8 * (K / 128), p.lsb));
    };
    static const struct { int bm, bn; float us; bool gn1; } T[BST_COUNT] = {
        {32, 32, 0.10f, false},  {32, 64, 0.18f, true},    {64, 64, 0.24f, true},   {128, 64, 0.38f, true},
        {128, 128, 0.60f, true}, {128, 256, 0.97f, false}, {256, 256, 1.5f, true}, {256, 224, 1.3125f, true}};
    const char* w224_env = std::getenv("HKQ_BLOCKSCALE_W224");
    const bool w224_on = !(w224_env && w224_env[0] == '0');
    const int64_t ncu = cu_count() > 0 ? cu_count() : 256;
    int best = BST_NONE;
    float best_us = 0.f;
    for (int t = BST_COUNT - 1; t >= 0; --t) {
        if ((gn1 && !T[t].gn1) || (t == BST_256x224 && !w224_on) || !fits(t, T[t].bm, T[t].bn)) continue;
        const int64_t tiles = ((M + T[t].bm - 1) / T[t].bm) * ((N + T[t].bn - 1) / T[t].bn);
        const float kt_us = gn1 && t == BST_128x128 ? 0.66f : T[t].us;
        const float us = (float)((tiles + ncu - 1) / ncu) * ((float)(K / 128) * kt_us + 2.3f);
        if (best_us == 0.f || us < best_us) {
            best = t;
            best_us = us;
        }
    }
    return best;
}

template <bool GN1>
static int launch_blockscale(BlockScaleParams& p, hipStream_t stream) {
    constexpr int B = MODE_BLOCKSCALE;
    switch (bs_plan(p, GN1)) {
        case BST_32x32:
            if constexpr (!GN1) return launch_blockscale_tile<KgCfg<B, 1, 1, 4, 1, 1, 4>, false>(p, stream);
            break;
        case BST_32x64: return launch_blockscale_tile<KgCfg<B, 1, 1, 4, 1, 2, 3, GN1>, GN1>(p, stream);
        case BST_64x64: return launch_blockscale_tile<KgCfg<B, 1, 1, 4, 2, 2, 2, GN1>, GN1>(p, stream);
        case BST_128x64: return launch_blockscale_tile<KgCfg<B, 4, 1, 2, 1, 2, 3, GN1>, GN1>(p, stream);
        case BST_128x128: return launch_blockscale_tile<KgCfg<B, 4, 2, 1, 1, 2, 4, GN1>, GN1>(p, stream);
        case BST_128x256:
            if constexpr (!GN1) return launch_blockscale_tile<KgCfg<B, 2, 4, 1, 2, 2, 3>, false>(p, stream);
            break;
        case BST_256x224: return launch_blockscale_bn<GN1, BS_BN - 32>(p, stream);
        case BST_NONE: {
            // the streaming kernel over groups of 16 rows
            HKQ_CHECK_ARG(bs_narrow_fits(p), "row pitches too large: 32 rows of each operand (or all of its rows) and of "
                                             "its scales must span less than 2^31 bytes");
            const int M = p.M;
            for (int m0 = 0; m0 < M; m0 += BSN_MAX_M) {
                BlockScaleParams q = p;
                q.A += (int64_t)m0 * p.lda;
                q.sa += (int64_t)m0 * p.lsa;
                q.C += (int64_t)m0 * p.ldc;
                if (p.ca) {
                    q.ca += (int64_t)m0 * p.ldca;
                    q.cb += (int64_t)m0 * p.ldcb;
                }
                q.M = std::min(BSN_MAX_M, M - m0);
                if (int e = launch_blockscale_narrow<GN1>(q, stream)) return e;
            }
            return 0;
        }
    }
    return launch_blockscale_bn<GN1, BS_BN>(p, stream);
}

}  // namespace hkq

using namespace hkq;

static int blockscale_call(const void* A, const void* B, const float* sa, const float* sb, void* C, const void* ca,
                           const void* cb, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t lsa,
                           int64_t lsb, int64_t ldc, int64_t ldca, int64_t ldcb, int64_t group_n, hipStream_t stream);

extern "C" int hkq_gemm_blockscale(const void* A, const void* B, const float* sa, const float* sb, void* C,
                                   int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t lsa,
                                   int64_t lsb, int64_t ldc, int64_t group_n, hipStream_t stream) {
    return blockscale_call(A, B, sa, sb, C, nullptr, nullptr, M, N, K, lda, ldb, lsa, lsb, ldc, 0, 0, group_n,
                           stream);
}

extern "C" int hkq_gemm_blockscale_mul_add(const void* A, const void* B, const float* sa, const float* sb, void* C,
                                           const void* c_a, const void* c_b, int64_t M, int64_t N, int64_t K,
                                           int64_t lda, int64_t ldb, int64_t lsa, int64_t lsb, int64_t ldc,
                                           int64_t ldca, int64_t ldcb, int64_t group_n, hipStream_t stream) {
    HKQ_CHECK_ARG(c_a && c_b, "c_a and c_b are required");
    HKQ_CHECK_ARG(ldca >= N && ldcb >= N && ldca % 4 == 0 && ldcb % 4 == 0,
                  "c_a / c_b row strides must be >= N and multiples of 4");
    HKQ_CHECK_ALIGN(c_a, 8);
    HKQ_CHECK_ALIGN(c_b, 8);
    return blockscale_call(A, B, sa, sb, C, c_a, c_b, M, N, K, lda, ldb, lsa, lsb, ldc, ldca, ldcb, group_n, stream);
}

static int blockscale_call(const void* A, const void* B, const float* sa, const float* sb, void* C, const void* ca,
                           const void* cb, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t lsa,
                           int64_t lsb, int64_t ldc, int64_t ldca, int64_t ldcb, int64_t group_n, hipStream_t stream) {
    HKQ_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "M, N must be >= 0 and K > 0");
    HKQ_CHECK_ARG(M < (1 << 30) && N < (1 << 30) && K < (1 << 30), "dimensions must be < 2^30");
    HKQ_CHECK_ARG(K % 128 == 0, "K must be a multiple of the 128-wide scale group");
    HKQ_CHECK_ARG(N % 4 == 0, "N must be a multiple of 4");
    HKQ_CHECK_ARG(group_n == 1 || group_n == 128, "group_n must be 1 or 128");
    HKQ_CHECK_ARG(lda >= K && ldb >= K && lda % 16 == 0 && ldb % 16 == 0, "lda/ldb must be >= K and multiples of 16");
    HKQ_CHECK_ARG(ldc >= N && ldc % 4 == 0, "ldc must be >= N and a multiple of 4");
    // a stride only matters when there is more than one row to step over
    HKQ_CHECK_ARG(M <= 1 || lsa >= K / 128, "a_scale row stride must be >= K/128");
    HKQ_CHECK_ARG(K / 128 <= 1 || lsb >= (group_n == 1 ? N : (N + 127) / 128),
                  "b_scale row stride must cover N / group_n columns");
    HKQ_CHECK_ALIGN(A, 16);
    HKQ_CHECK_ALIGN(B, 16);
    HKQ_CHECK_ALIGN(C, 8);
    HKQ_CHECK_ALIGN(sa, 4);
    HKQ_CHECK_ALIGN(sb, 4);
    BlockScaleParams p{};
    p.A = static_cast<const uint8_t*>(A);
    p.B = static_cast<const uint8_t*>(B);
    p.C = static_cast<uint16_t*>(C);
    p.sa = sa;
    p.sb = sb;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.lsa = lsa; p.lsb = lsb;
    p.ca = static_cast<const uint16_t*>(ca);
    p.cb = static_cast<const uint16_t*>(cb);
    p.ldca = ldca; p.ldcb = ldcb;
    if (M == 0 || N == 0) return 0;
    // a stride only counts where there is a second row to step to
    if (M == 1) {
        p.lda = K;
        p.lsa = K / 128;
    }
    if (K / 128 == 1) p.lsb = group_n == 1 ? N : (N + 127) / 128;
    // M <= 16 with at most 32 K groups streams the weights through registers
    // (16 x 7168 x 2048: 6.1 us against 5.8 on small tiles, 1 x 24576 x 1536
    // 10.3 against 11). With longer K the tiles' deeper rings win (8 x 7168 x
    // 18432 28.0 against 21.1, 16384 columns of K 5120 17.3 against 15.7 with
    // one scale per column) except where one 16-column slice per CU holds all of
    // N: with one scale per column, whose smallest tile is 64 wide, the stream
    // wins to 12 rows (1 x 2112 x 7168 7.7 against 11.3, 12 x 4096 x 14336 17.6
    // against 19.0) and to 16 rows of up to 56 groups (16 x 2112 x 5632 8.6
    // against 10.1, x 7168 11.3 both); with one per 128, to 2 rows of 48 groups
    // (2 x 2112 x 5632 6.3 against 6.7, 4 x 2112 x 7168 8.0 against 7.4).
    const int64_t groups = K / 128, ncu = cu_count() > 0 ? cu_count() : 256;
    const bool one_slice = (N + 15) / 16 <= ncu;
    const bool stream_long = group_n == 1 ? M <= 12 || groups <= 56 : M <= 2 && groups <= 48;
    if (M <= BSN_MAX_M && (groups <= 32 || (one_slice && stream_long)) && bs_narrow_fits(p))
        return group_n == 1 ? launch_blockscale_narrow<true>(p, stream) : launch_blockscale_narrow<false>(p, stream);
    return group_n == 1 ? launch_blockscale<true>(p, stream) : launch_blockscale<false>(p, stream);
}
