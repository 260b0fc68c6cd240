// The MFMA kernel of the projection + conv + SiLU (proj.hip holds its entry
// points and the rule that picks its tile; proj_packed.hip the launches for
// packed sequences, so that the two sets of instantiations build in parallel).
//
// gdn_proj_conv_mfma_kernel (the fast path) computes the transposed product
// P^T = W x^T in tiles of 32 x 32 up to 256 columns x 256 tokens, chosen from
// the size of the product (choose_tile).  Rows run over a flattened token axis
// where each sequence is 3 cache rows followed by its T tokens; a tile's first
// 3 rows are the causal halo (recomputed), so 253 rows of 256 are written per
// tile, and cache rows take the conv cache (or zero) so no tap reaches into
// another sequence.  Operands reach LDS by DMA (global_load_lds) in a ring of
// 64-wide K stages: every 8 lanes of a copy read one whole 128-byte line (a
// row's K slice), placed with an XOR swizzle that keeps the MFMA fragment
// reads at linear-read speed.  The largest tile's waves form a 4 x 2 grid of
// 64 columns x 128 tokens = 4 x 8 MFMA 16x16x32 tiles.  In the transposed C
// layout a lane holds 4 columns of one token, 16 tokens an MFMA tile; rows
// are staged in an order that makes a lane's tokens consecutive (one per
// MFMA tile) and its columns too, so the conv taps are registers of the lane
// (three a wave edge come from the neighbour lane by DPP) and its results
// leave as 16-byte stores.
//
// What bounds it: with every CU on 256 x 256 tiles of a 2048-wide K a tile
// takes ~57 us, ~43 of them the main loop (1.34 us a 64-wide stage, 1.6
// PFLOP/s over the chip) and ~12 the epilogue, whose VALU work per output (4
// FMA, exp2, reciprocal and 4 more) cannot run under the matrix cores while
// the accumulators fill half the registers.  Smaller tiles are bound by the
// copies' entry into LDS (27-30 B/clk per CU beside fragment reads).  Measured
// at 16384 tokens, 6176 columns, D = 2048: 464 us with all eight waves in step
// and the conv through LDS windows and an LDS output tile; 429 with the waves
// in two alternating groups; 391-399 with the epilogue in registers.
#pragma once

#include <cstddef>
#include <type_traits>

#include "gdn_common.hpp"
#include "proj.hpp"

namespace {

using namespace gdn;

enum { kEqual = 0, kPacked = 1, kPlain = 2 };  // what the rows are (gdn_proj_conv_mfma_kernel)
constexpr int kHalo = 3;  // rows ahead of a tile that its conv taps reach
constexpr int kMK = 64;          // K per stage: one 128-byte line per row
constexpr int kMRowB = kMK * 2;  // 128 bytes per staged row

// A workgroup's tile: CW x TW waves, each WMT 16-column x WNT 16-token MFMA
// tiles, NS K stages in LDS, PER_CU workgroups on a CU.
// PHASED: the two-group main loop (eight waves, one workgroup on a CU).
// KS (kPlain only): KS groups of CW x TW waves, each on its own 64-wide slice
// of a stage of 64 KS, summed at the end.
// KD: 64-wide slices a stage holds (for each group), multiplied in order (the
// sums are those of KD = 1): half the barriers and twice the copies in flight
// for a wave, where a stage's latency binds.
template <int CW_, int TW_, int WMT_, int WNT_, int NS_, int PER_CU_, bool PHASED_ = false, int KS_ = 1, int KD_ = 1>
struct ProjTile {
    static constexpr int KS = KS_, KD = KD_;
    static constexpr bool PHASED = PHASED_;
    static constexpr int CW = CW_, TW = TW_, WMT = WMT_, WNT = WNT_, NS = NS_, PER_CU = PER_CU_;
    static constexpr int cols = 16 * CW * WMT;   // output columns (W rows) per workgroup
    static constexpr int toks = 16 * TW * WNT;   // token rows per workgroup
    static constexpr int outs = toks - kHalo;    // tokens written per workgroup (kPlain: toks)
    static constexpr int gwaves = CW * TW;  // waves of a K group
    static constexpr int waves = gwaves * KS;
    static constexpr int slice_b = (cols + toks) * kMRowB;    // a group's W rows, then x rows
    static constexpr int stage_b = KS * KD * slice_b;
    static constexpr int dma = (cols + toks) / 8 / gwaves;    // 1 KiB copies (8 rows) per wave per slice
    static_assert(PHASED || (cols + toks) % (8 * gwaves) == 0, "copies split evenly");
    static_assert(!PHASED || (KS == 1 && KD == 1), "phased tile");
    static_assert((KS - 1) * gwaves * WMT * WNT * 1024 <= NS * stage_b, "the groups' sums fit the dead stages");
    // PHASED: a stage is staged, and its buffer freed, region by region: the
    // first and second part of every wave's tokens (X0, X1) and columns (W0,
    // W1), in the order X0, W0, W1, X1.  A region of `groups` 8-row copies is
    // split over the waves, each taking groups / 8 whole copies and, where 4
    // are left, one of 4 rows by half its lanes.
    static constexpr int M0n = WMT / 2, M1n = WMT - M0n, X0n = (WNT + 1) / 2, X1n = WNT - X0n;
    static constexpr int groups(int r) { return 2 * (r == 0 ? TW * X0n : r == 1 ? CW * M0n : r == 2 ? CW * M1n : TW * X1n); }
    static constexpr int full(int r) { return groups(r) / 8; }
    static constexpr int half(int r) { return groups(r) % 8 / 4; }
    static constexpr int ncopy(int r) { return full(r) + half(r); }
    static constexpr int first(int r) { return r == 0 ? 0 : first(r - 1) + ncopy(r - 1); }
    static constexpr int ncopies = first(4);
    static_assert(!PHASED || (waves == 8 && PER_CU == 1 && groups(0) % 4 == 0 && groups(1) % 4 == 0 && groups(2) % 4 == 0 &&
                              groups(3) % 4 == 0 && M0n > 0 && X1n > 0),
                  "phased tile");
    // The hand-over area: P of the last 3 tokens of each token wave but the
    // last, fp32 [wave][token][column]; in the dead stages (one more barrier)
    // where the LDS holds no more.
    static constexpr int hand_b = (TW - 1) * kHalo * cols * 4;
    static constexpr bool in_stages = (NS * stage_b + hand_b) * PER_CU > 160 * 1024;
    static constexpr int off_hand = in_stages ? 0 : NS * stage_b;
    static constexpr int lds_b = in_stages ? NS * stage_b : NS * stage_b + hand_b;
    static_assert(lds_b * PER_CU <= 160 * 1024 && hand_b <= NS * stage_b, "LDS");
};

// Staged row r holds its 8 16-byte chunks (k 8c .. 8c+7) at slot c ^ (r & 7):
// a fragment read (16 rows, one chunk each) then spreads every 8 consecutive
// rows over the 8 slots of a 128-byte line, which reads at the rate of a
// linear ds_read_b128 on gfx950 (measured; (r ^ (r >> 3)) & 7 lost a third).
__device__ __forceinline__ int swz(int r) { return r & 7; }

// Packed row table of the launch (ProjParams::row_off), read from the
// kernel's argument block (the ProjParams argument sits at its start):
// indexing the by-value parameter with a runtime index would copy it to
// private memory.
using kconst_i32 = __attribute__((address_space(4))) const int32_t;
__device__ __forceinline__ const kconst_i32* packed_rows() {
    const __attribute__((address_space(4))) char* base =
        (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    return reinterpret_cast<const kconst_i32*>(base + offsetof(gdn_proj::ProjParams, row_off));
}

// Groups whose output goes out in 16-byte stores (8 columns): 8-column
// aligned, 8-column head_dim (or token-major), 16-byte aligned destination.
__device__ __forceinline__ bool wide_group(const gdn_proj::ProjGroup& g) {
    return ((g.col0 | g.width | g.head_dim) & 7) == 0 && (reinterpret_cast<uintptr_t>(g.dst) & 15) == 0;
}

// Workgroup barrier alone (no LDS access of this wave is outstanding); no
// memory access moves across it.
__device__ __forceinline__ void wave_barrier() { asm volatile("s_barrier" ::: "memory"); }

// The group holding column c, by compare-and-select over constant indices
// (indexing the parameter block with a runtime index would copy it to
// private memory).
__device__ __forceinline__ gdn_proj::ProjGroup select_group(const gdn_proj::ProjParams& p, int c) {
    gdn_proj::ProjGroup g = p.groups[0];
#pragma unroll
    for (int q = 1; q < gdn_proj::kMaxGroups; ++q)
        if (q < p.ngroups && c >= p.groups[q].col0) g = p.groups[q];
    return g;
}

// kEqual: p.B sequences of p.T tokens.  kPacked: sequences of unequal lengths
// (ProjParams::packed > 0), rows mapped through the row table.  kPlain: the
// product alone, [p.T, D_out], no conv (and no halo, so a tile writes all of
// its rows).  Instantiations of their own, so that none carries the others'
// code.
template <class TL, int MODE>
__global__ __launch_bounds__(TL::waves * 64)
    __attribute__((amdgpu_waves_per_eu(TL::PER_CU * TL::waves / 4, TL::PER_CU * TL::waves / 4))) void gdn_proj_conv_mfma_kernel(
        gdn_proj::ProjParams p, int n_tok, int n_col) {
    constexpr int kMCols = TL::cols, kMToks = TL::toks, kMWaves = TL::waves, kMStages = TL::NS;
    constexpr int kWMT = TL::WMT, kWNT = TL::WNT, kMStageB = TL::stage_b, kMDma = TL::dma;
    __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[TL::lds_b];
    lds_u8* const smem = (lds_u8*)&smem_raw[0];

    // Workgroup -> tile.  Dispatch deals workgroups to the 8 XCDs round-robin;
    // give each XCD a contiguous range of tiles, ordered in bands of 4 column
    // tiles with the token tile slowest, so the workgroups resident on one
    // XCD share W and x tiles in its L2.
    const int ntiles = n_tok * n_col;
    int lin;
    {
        const int id = blockIdx.x, xcd = id & 7, j = id >> 3, q = ntiles >> 3, r = ntiles & 7;
        lin = xcd < r ? xcd * (q + 1) + j : r * (q + 1) + (xcd - r) * q + j;
        const int band = lin / (4 * n_tok), base = 4 * band, gs = min(n_col - base, 4);
        const int within = lin - band * 4 * n_tok;
        lin = (within / gs) * n_col + base + within % gs;
    }
    const int tile_t = lin / n_col, tile_c = lin % n_col;
    // Row space: each sequence is kHalo cache rows (t = -3 .. -1) followed by
    // its tokens, so row r is (b, t) = (r / T3, r % T3 - 3) for equal lengths
    // T, or, for packed sequences, b the last with row_off[b] <= r and
    // t = r - row_off[b] - 3.  Cache rows take the cached projections (or
    // zero) after the product, so conv taps never reach into another
    // sequence.
    constexpr bool packed = MODE == kPacked, plain = MODE == kPlain;
    constexpr int kMOut = plain ? kMToks : TL::outs;
    const int T3 = p.T + kHalo;
    const kconst_i32* prow = packed_rows();
    const int nseq = packed ? p.packed : p.B;
    const int F3 = packed ? prow[p.packed] : plain ? p.T : p.B * T3;
    const int f0 = tile_t * kMOut - (plain ? 0 : kHalo);  // row of tile row 0 (>= -3; rows < 0 are never used)
    // Packed: the sequence of the tile's first row (uniform), the start of
    // every per-row search below.
    int pb0 = 0;
    if (packed) {
        int lo = 0, hi = p.packed;  // prow[lo] <= max(f0, 0) < prow[hi]
        const int r = max(f0, 0);
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (prow[mid] <= r) lo = mid; else hi = mid;
        }
        pb0 = lo;
    }
    auto len3 = [&](int b) { return packed ? prow[b + 1] - prow[b] : T3; };     // rows of sequence b
    auto tok0 = [&](int b) { return packed ? prow[b] - kHalo * b : b * p.T; };  // x row of its first token
    // (b, t3 = t + 3) of row r >= 0 (packed rows past the last sequence stay in it).
    auto locate = [&](int r, int& b, int& t3) {
        if (packed) {
            int bb = pb0;
            while (bb + 1 < p.packed && prow[bb + 1] <= r) ++bb;
            b = bb;
            t3 = r - prow[bb];
        } else {
            b = r / T3;
            t3 = r - b * T3;
        }
    };
    const int c0 = tile_c * kMCols;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: DMA bases stay scalar
    static_assert(TL::KS == 1 || MODE == kPlain, "K groups are for the plain product");
    const int ks = TL::KS > 1 ? wave / TL::gwaves : 0, gw = TL::KS > 1 ? wave % TL::gwaves : wave;  // K group, wave in it
    const int wm = gw / TL::TW, wn = gw % TL::TW;                 // column slice, token slice
    const int r16 = lane & 15, g4 = lane >> 4;

    // x row feeding row r: the token itself, the sequence's first token for
    // cache rows, clamped at both ends (those products are never used).
    auto xrow_of = [&](int r) {
        if constexpr (plain) {
            return min(r, F3 - 1);
        } else if constexpr (packed) {
            const int ntok = F3 - kHalo * p.packed;  // x rows
            if (r < 0) return 0;
            if (r >= F3) return ntok - 1;
            int b, t3;
            locate(r, b, t3);
            return min(tok0(b) + max(t3 - kHalo, 0), ntok - 1);  // an empty last sequence has no token of its own
        } else {
            if (r < 0) return 0;
            if (r >= F3) return p.B * p.T - 1;
            const int b = r / T3, t = r - b * T3 - kHalo;
            return b * p.T + max(t, 0);
        }
    };

    // DMA sources.  Staged rows 0 .. cols - 1 are W rows, the others x rows.  Copy
    // j of a wave moves 8 of them, from 8 (gw + gwaves j) on, or, in the phased
    // tiles, a region's (copy_row); lane l takes row l / 8 of those and fills
    // slot l % 8 with chunk (l % 8) ^ swz(row): every 8 lanes read one whole
    // 128-byte line.  Columns >= D_out are clamped to a valid row; their
    // products are never stored.
    const int xrow0 = xrow_of(f0);
    const unsigned char* wsrc = reinterpret_cast<const unsigned char*>(p.W + static_cast<size_t>(c0) * p.D);
    const unsigned char* xsrc = reinterpret_cast<const unsigned char*>(p.x + static_cast<size_t>(xrow0) * p.D);
    // Which row a staged row holds is free, as every fragment is read whole:
    // the order below gives a lane of the product WNT consecutive tokens and
    // 4 WMT consecutive columns (its accumulator (mt, nt) is token WNT n + nt
    // of the wave's, columns 4 WMT g + 4 mt .. + 3), so the conv taps are its
    // own registers and its outputs leave in 16-byte stores.
    auto src_off = [&](int srow) {
        int row;
        if (srow < kMCols) {
            const int w = srow / (16 * kWMT), s = srow % (16 * kWMT);
            const int col = 16 * kWMT * w + 4 * kWMT * ((s & 15) >> 2) + 4 * (s >> 4) + (s & 3);
            row = min(c0 + col, p.D_out - 1) - c0;
        } else {
            const int w = (srow - kMCols) / (16 * kWNT), s = (srow - kMCols) % (16 * kWNT);
            row = xrow_of(f0 + 16 * kWNT * w + kWNT * (s & 15) + (s >> 4)) - xrow0;
        }
        const int chunk = (lane & 7) ^ swz(srow);
        return static_cast<uint32_t>(row) * static_cast<uint32_t>(p.D) * 2u + 16u * chunk;
    };
    // Copy j of region r in the phased loop: the first staged row, the same
    // for the wave.
    auto copy_row = [&](int r, int j) {
        const int g2 = j < TL::full(r) ? 2 * (wave + kMWaves * j) : 2 * kMWaves * TL::full(r) + wave;  // in 4-row units
        const int per = 4 * (r == 0 ? TL::X0n : r == 1 ? TL::M0n : r == 2 ? TL::M1n : TL::X1n);       // units of one wave's part
        const int w = g2 / per, within = 4 * (g2 % per);
        return r == 0 || r == 3 ? kMCols + 16 * kWNT * w + (r == 3 ? 16 * TL::X0n : 0) + within
                                : 16 * kWMT * w + (r == 2 ? 16 * TL::M0n : 0) + within;
    };
    constexpr int kCopies = TL::PHASED ? TL::ncopies : kMDma;
    uint32_t voff[kCopies];
    int crow[kCopies];  // staged row of the copy's first lane (wave-uniform)
    if constexpr (TL::PHASED) {
        static_for<0, 4>([&](auto R) {
            constexpr int r = decltype(R)::value;
            static_for<0, TL::ncopy(r)>([&](auto J) {
                constexpr int j = decltype(J)::value, c = TL::first(r) + j;
                crow[c] = __builtin_amdgcn_readfirstlane(copy_row(r, j));
                voff[c] = src_off(crow[c] + (j < TL::full(r) ? lane >> 3 : (lane >> 3) & 3));
            });
        });
    } else {
#pragma unroll
        for (int j = 0; j < kMDma; ++j) {
            crow[j] = 8 * (gw + TL::gwaves * j);
            voff[j] = src_off(crow[j] + (lane >> 3));
        }
    }
    auto issue_copy = [&](int stage, int kk, int d, int j) {
        int slice = (kk * TL::KD + d) * TL::KS + ks;
        if (TL::KD > 1) slice = min(slice, p.D / kMK - 1);  // an odd count's last stage repeats its slice (not multiplied)
        const unsigned char* src = (crow[j] < kMCols ? wsrc : xsrc) + slice * kMRowB;
        dma16(src, voff[j], smem + stage * kMStageB + (d * TL::KS + ks) * TL::slice_b + crow[j] * kMRowB);
    };
    auto issue = [&](int stage, int kk) {
#pragma unroll
        for (int d = 0; d < TL::KD; ++d)
#pragma unroll
            for (int j = 0; j < kCopies; ++j) issue_copy(stage, kk, d, j);
    };
    // Half `half` of the copies of a stage's slice d.
    auto issue_part = [&](int stage, int kk, int d, int half) {
#pragma unroll
        for (int j = 0; j < kCopies; ++j)
            if ((j >= (kCopies + 1) / 2) == (half == 1)) issue_copy(stage, kk, d, j);
    };
    // Region r of stage kk (phased loop).
    auto issue_region = [&](auto R, int stage, int kk) {
        constexpr int r = decltype(R)::value;
        const unsigned char* src = (r == 0 || r == 3 ? xsrc : wsrc) + kk * kMRowB;
        static_for<0, TL::ncopy(r)>([&](auto J) {
            constexpr int j = decltype(J)::value, c = TL::first(r) + j;
            lds_u8* dst = smem + stage * kMStageB + crow[c] * kMRowB;
            if (j < TL::full(r) || lane < 32) dma16(src, voff[c], dst);
        });
    };

    // Fragment reads: lane l takes row 16 f + l % 16, chunk 4 h + l / 16 of
    // the staged rows (h: which 32-wide half of the stage's K); rd[h] is the
    // lane's byte offset within the fragment.
    uint32_t rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd[h] = r16 * kMRowB + 16u * ((4 * h + g4) ^ swz(r16));

    // Conv weights of this lane's columns, fetched now so their latency hides
    // under the main loop: for conv_k == 4 the 4 columns' taps are 16
    // adjacent bf16 (32-byte aligned: groups start on 4 columns).
    u32x4 wraw[kWMT][2];
#pragma unroll
    for (int mt = 0; mt < kWMT; ++mt) {
        wraw[mt][0] = wraw[mt][1] = u32x4{0u, 0u, 0u, 0u};
        const int cb = c0 + 16 * kWMT * wm + 4 * kWMT * g4 + 4 * mt;
        if (!plain && cb < p.D_out && p.conv_k == 4) {
            const gdn_proj::ProjGroup gq = select_group(p, cb);
            if (gq.conv) {
                const u32x4* src = reinterpret_cast<const u32x4*>(p.conv_w + static_cast<size_t>(gq.cw_row0 + cb - gq.col0) * 4);
                wraw[mt][0] = src[0];
                wraw[mt][1] = src[1];
            }
        }
    }

    f32x4 acc[kWMT][kWNT];
#pragma unroll
    for (int mt = 0; mt < kWMT; ++mt)
#pragma unroll
        for (int nt = 0; nt < kWNT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    static_assert(TL::KS == 1 || TL::KD == 1, "whole stages with K groups");
    constexpr int kStageK = kMK * TL::KS * TL::KD;
    const int nk = (p.D + (TL::KD > 1 ? kStageK - 1 : 0)) / kStageK;
    if constexpr (TL::PHASED) {
        // Two groups of four waves, one wave of each on every SIMD, take
        // turns: while one multiplies, the other reads its next fragments and
        // issues its copies.  A stage is four phases, each a part of the
        // wave's tile (first or second half of its columns x of its tokens)
        // over the stage's whole K: (W0, X0), (W1, X0), (W1, X1), (W0, X1).
        // Phase 0 reads W0 and X0, phase 1 W1, phase 2 X1, phase 3 nothing.
        // A region's buffer is free once both groups have read it, so stage
        // kt + NS's X0, W0 and W1 go out in phases 1, 2 and 3 of stage kt and
        // its X1 in phase 0 of the next: about five phases a region has to
        // land.  The waits count the copies issued after the region that the
        // next phase reads; T >= 0: T stages are left after this one and no
        // new ones are issued.
        bf16x8 w0[TL::M0n][2], w1[TL::M1n][2], xf[TL::X0n][2];
        constexpr int cX0 = TL::ncopy(0), cW1 = TL::ncopy(2), cX1 = TL::ncopy(3), cAll = TL::ncopies;
        auto read = [&](const lds_u8* st, int row, int h) {
            return *reinterpret_cast<const lds_bf16x8*>(st + row * kMRowB + rd[h]);
        };
        auto next_buf = [](int b, int n) {
            b += n;
            return b >= kMStages ? b - kMStages : b;
        };
        auto stage = [&](int kt, int rs, auto Tc) {
            constexpr int T = decltype(Tc)::value;
            constexpr bool steady = T < 0;
            const lds_u8* st = smem + rs * kMStageB;
            const lds_u8* stx = st + (kMCols + 16 * kWNT * wn) * kMRowB;
            const lds_u8* stw = st + 16 * kWMT * wm * kMRowB;
            static_for<0, 4>([&](auto Pc) {
                constexpr int ph = decltype(Pc)::value;
                static_for<0, 2>([&](auto H) {
                    constexpr int h = decltype(H)::value;
                    if constexpr (ph == 0) {
                        static_for<0, TL::M0n>([&](auto I) { w0[decltype(I)::value][h] = read(stw, 16 * decltype(I)::value, h); });
                        static_for<0, TL::X0n>([&](auto I) { xf[decltype(I)::value][h] = read(stx, 16 * decltype(I)::value, h); });
                    } else if constexpr (ph == 1) {
                        static_for<0, TL::M1n>([&](auto I) {
                            w1[decltype(I)::value][h] = read(stw, 16 * (TL::M0n + decltype(I)::value), h);
                        });
                    } else if constexpr (ph == 2) {
                        static_for<0, TL::X1n>([&](auto I) {
                            xf[decltype(I)::value][h] = read(stx, 16 * (TL::X0n + decltype(I)::value), h);
                        });
                    }
                });
                if constexpr (ph == 0 && (steady || T == kMStages - 1))
                    issue_region(std::integral_constant<int, 3>{}, next_buf(rs, kMStages - 1), kt + kMStages - 1);
                else if constexpr (ph > 0 && steady)
                    issue_region(std::integral_constant<int, ph - 1>{}, rs, kt + kMStages);
                if constexpr (ph == 0)
                    wait_vm<cX1 + (steady ? kMStages - 1 : T) * cAll>();
                else if constexpr (ph == 1)
                    wait_vm<steady ? cX0 + (kMStages - 1) * cAll : T * cAll>();
                else if constexpr (ph == 3 && T != 0)
                    wait_vm<cW1 + (steady ? (kMStages - 1) * cAll : cX1 + (T - 1) * cAll)>();
                lds_barrier();  // this group's fragments are here, the other's multiplications issued
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(1);
                static_for<0, 2>([&](auto H) {
                    constexpr int h = decltype(H)::value;
                    constexpr int m0 = ph == 0 || ph == 3 ? 0 : TL::M0n, mn = ph == 0 || ph == 3 ? TL::M0n : TL::M1n;
                    constexpr int n0 = ph < 2 ? 0 : TL::X0n, nn = ph < 2 ? TL::X0n : TL::X1n;
#pragma unroll
                    for (int nt = 0; nt < nn; ++nt)
#pragma unroll
                        for (int mt = 0; mt < mn; ++mt)
                            acc[m0 + mt][n0 + nt] =
                                mfma16x16x32(m0 == 0 ? w0[mt][h] : w1[mt][h], xf[nt][h], acc[m0 + mt][n0 + nt]);
                });
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_sched_barrier(0);
                wave_barrier();
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        // Fill the ring as the phases would have.
        static_for<0, kMStages>([&](auto S) {
            constexpr int s = decltype(S)::value;
            if (s < nk) {
                static_for<0, s + 1 < kMStages ? 4 : 3>([&](auto R) { issue_region(R, s, s); });
            }
        });
        if (nk >= kMStages)
            wait_vm<cW1 + (kMStages - 1) * cAll>();  // X0 and W0 of stage 0
        else
            wait_vm<0>();
        wave_barrier();
        const bool second = wave >= kMWaves / 2;
        if (second) wave_barrier();
        int kt = 0, rs = 0;
        for (; kt + kMStages < nk; ++kt) {
            stage(kt, rs, std::integral_constant<int, -1>{});
            rs = next_buf(rs, 1);
        }
        static_for<0, kMStages>([&](auto I) {
            constexpr int T = kMStages - 1 - decltype(I)::value;
            if (T < nk) {
                stage(kt, rs, std::integral_constant<int, T>{});
                ++kt;
                rs = next_buf(rs, 1);
            }
        });
        if (!second) wave_barrier();
    } else {
        // Ring of NS stages: stage kt + NS - 1 is issued while stage kt is
        // multiplied, into the buffer that stage kt - 1 was read from.
#pragma unroll
        for (int st = 0; st < kMStages - 1; ++st)
            if (st < nk) issue(st, st);
        int rs = 0, ws = kMStages - 1;  // buffers of stage kt and of stage kt + NS - 1
        for (int kt = 0; kt < nk; ++kt) {
            const bool next = kt + kMStages - 1 < nk;
            // Stage kt has landed (later ones may be in flight; the last NS - 1
            // stages wait for every copy).
            if (kMStages > 2 && next)
                wait_vm<(kMStages - 2) * TL::KD * kMDma>();
            else
                wait_vm<0>();
            lds_barrier();  // for every wave; the buffer of stage kt - 1 is fully read
            // The new stage's copies go out in two halves, one before each K
            // half's MFMAs: a wave that issues all of them at once stalls on
            // the copy queue before its first MFMA.
            const lds_u8* st0 = smem + rs * kMStageB + ks * TL::slice_b;
            static_for<0, 2 * TL::KD>([&](auto H) {
                constexpr int d = decltype(H)::value / 2, h = decltype(H)::value % 2;
                const lds_u8* st = st0 + d * TL::KS * TL::slice_b;
                if (next) issue_part(ws, kt + kMStages - 1, d, h);
                bf16x8 a[kWMT], bx[kWNT];
                static_for<0, kWMT>([&](auto MT) {
                    constexpr int mt = decltype(MT)::value;
                    a[mt] = *reinterpret_cast<const lds_bf16x8*>(st + (16 * kWMT * wm + 16 * mt) * kMRowB + rd[h]);
                });
                static_for<0, kWNT>([&](auto NT) {
                    constexpr int nt = decltype(NT)::value;
                    bx[nt] = *reinterpret_cast<const lds_bf16x8*>(st + (kMCols + 16 * kWNT * wn + 16 * nt) * kMRowB + rd[h]);
                });
                if (TL::KD > 1 && (kt * TL::KD + d) * kMK >= p.D) return;
#pragma unroll
                for (int nt = 0; nt < kWNT; ++nt)
#pragma unroll
                    for (int mt = 0; mt < kWMT; ++mt) acc[mt][nt] = mfma16x16x32(a[mt], bx[nt], acc[mt][nt]);
            });
            rs = rs + 1 == kMStages ? 0 : rs + 1;
            ws = ws + 1 == kMStages ? 0 : ws + 1;
        }
    }

    if constexpr (TL::KS > 1) {
        lds_barrier();  // every wave is past its last stage read
        const auto part = [&](int k, int i) {
            return reinterpret_cast<lds_f32x4*>(smem + (((k - 1) * TL::gwaves + gw) * kWMT * kWNT + i) * 1024 + 16 * lane);
        };
        if (ks > 0) {
#pragma unroll
            for (int i = 0; i < kWMT * kWNT; ++i) *part(ks, i) = acc[i / kWNT][i % kWNT];
        }
        lds_barrier();
        if (ks > 0) return;
#pragma unroll
        for (int k = 1; k < TL::KS; ++k)
#pragma unroll
            for (int i = 0; i < kWMT * kWNT; ++i) acc[i / kWNT][i % kWNT] += *part(k, i);
    }

    // Epilogue, in registers: this lane holds rows R0 + nt (tile row nloc0 +
    // nt) of columns cl0 + 4 mt .. + 3 of the tile.
    const int nloc0 = 16 * kWNT * wn + kWNT * r16;
    const int R0 = f0 + nloc0;
    const int cl0 = 16 * kWMT * wm + 4 * kWMT * g4;
    if constexpr (plain) {
        uint16_t* const dst = p.groups[0].dst;
        static_for<0, kWNT>([&](auto NT) {
            constexpr int nt = decltype(NT)::value;
            if (R0 + nt >= F3) return;
            uint16_t* const row = dst + static_cast<size_t>(R0 + nt) * p.D_out + c0 + cl0;
            static_for<0, kWMT>([&](auto MT) {
                constexpr int mt = decltype(MT)::value;
                if constexpr (kWMT == 1) {
                    if (c0 + cl0 < p.D_out) *reinterpret_cast<u32x2*>(row) = pack4_bf16(acc[0][nt]);
                } else if constexpr (mt % 2 == 0) {
                    const u32x2 lo = pack4_bf16(acc[mt][nt]), hi = pack4_bf16(acc[mt + 1][nt]);
                    if (c0 + cl0 + 4 * mt < p.D_out)
                        *reinterpret_cast<u32x4*>(row + 4 * mt) = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
            });
        });
        return;
    }
    auto split = [&](int r, int& b, int& t3) {
        if (r < 0) {
            b = 0;
            t3 = r;
        } else {
            locate(r, b, t3);
        }
    };
    int b0, t30;  // sequence and t + 3 of row R0
    split(R0, b0, t30);
    // (b, t3) of the next row (packed rows past the last sequence stay in it).
    auto step = [&](int& b, int& t3) {
        ++t3;
        while ((!packed || b + 1 < nseq) && t3 >= len3(b)) {
            t3 -= len3(b);
            ++b;
        }
    };
    const int ncache = p.conv_k - 1;
    // Lean epilogue when the wave's 16 kWNT rows are all tokens of one
    // sequence (no cache rows, no sequence start) and none of them is in the
    // conv cache refresh window (the last ncache tokens).
    bool lean;
    {
        const int RW = f0 + 16 * kWNT * wn;
        int bR, t3R;
        split(RW, bR, t3R);
        lean = RW >= 0 && RW + 16 * kWNT <= F3 && t3R >= kHalo && t3R + 16 * kWNT <= len3(bR) - ncache;
    }
    // Where the lane's rows meet the conv caches, two bits a row: cache_row its
    // place t + 3 among its sequence's cache rows, last_row its place among the
    // last ncache tokens, 3 for neither; from last_row's bit 16 on the rows that
    // begin another sequence than the row before.  (Walked once: in packed rows a
    // step reads the row table, and walking again for each column quad cost 8 us
    // of 99 over ten prompts.)
    uint32_t last_row = 0xffffu;
    static_assert(kWNT <= 8, "two bits a row");
    // Cache rows (t < 0) of conv groups take the cached projection of token t
    // (cache index t + ncache, oldest first), zero before the cache or
    // without one.  With 3 cached tokens a sequence's 12 values of a column
    // quad are 24 adjacent bytes, fetched once for the lane's rows of it (and
    // stored so below): 1000 sequences of 2 tokens, D = 2048, 6176 columns,
    // 162 us a call, a value at a time 240; of 1 token 150 against 232.
    const auto by_quad = [&](const uint16_t* cache) { return ncache == 3 && (reinterpret_cast<uintptr_t>(cache) & 7) == 0; };
    const auto any_lane = [](bool x) { return __builtin_amdgcn_ballot_w64(x) != 0; };
    const auto begins = [&](int nt) { return static_cast<int>(last_row >> (16 + nt)) & 1; };
    if (!lean) {
        uint32_t cache_row = 0xffffu;
        int b = b0, t3 = t30;
        static_for<0, kWNT>([&](auto NT) {
            constexpr int nt = decltype(NT)::value;
            if (nt > 0) {
                const int before = b;
                step(b, t3);
                last_row |= (b != before ? 0x10000u : 0u) << nt;
            }
            if (R0 + nt < 0 || R0 + nt >= F3) return;
            if (t3 < kHalo) cache_row ^= (3u ^ static_cast<uint32_t>(t3)) << (2 * nt);
            const int j = t3 - (len3(b) - ncache);  // token t = T - ncache + j
            if (nloc0 + nt >= kHalo && j >= 0) last_row ^= (3u ^ static_cast<uint32_t>(j)) << (2 * nt);
        });
        if (any_lane(cache_row != 0xffffu)) {
            static_for<0, kWMT>([&](auto MT) {
                constexpr int mt = decltype(MT)::value;
                const int cb = c0 + cl0 + 4 * mt;
                if (cb >= p.D_out) return;
                const gdn_proj::ProjGroup gq = select_group(p, cb);
                if (!gq.conv) return;
                const bool quads = gq.cache_in != nullptr && by_quad(gq.cache_in);
                u32x2 held[3] = {};
                int b = b0;
                static_for<0, kWNT>([&](auto NT) {
                    constexpr int nt = decltype(NT)::value;
                    b += begins(nt);
                    const int t3 = (cache_row >> (2 * nt)) & 3;
                    if (t3 == 3) return;
                    const int q = t3 - kHalo + ncache;
                    const size_t at = (static_cast<size_t>(b) * gq.width + cb - gq.col0) * ncache;
                    f32x4 v = {0.f, 0.f, 0.f, 0.f};
                    if (quads) {
                        if (nt == 0 || t3 == 0) {
                            const u32x2* src = reinterpret_cast<const u32x2*>(gq.cache_in + at);
#pragma unroll
                            for (int u = 0; u < 3; ++u) held[u] = src[u];
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {  // value 3 i + q, q = 0..2: a half of one of two words
                            const int w0 = 3 * i / 2, w1 = w0 + 1, e = 3 * i % 2 + q;  // e: half, from w0's first
                            const uint32_t w = e < 2 ? held[w0 / 2][w0 % 2] : held[w1 / 2][w1 % 2];
                            v[i] = __uint_as_float((e & 1) ? w & 0xffff0000u : w << 16);
                        }
                    } else if (gq.cache_in != nullptr && q >= 0) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = bf2f(gq.cache_in[at + i * ncache + q]);
                    }
                    acc[mt][nt] = v;
                });
            });
        }
    }

    // Token waves meet inside the tile: a wave's first tokens take their conv
    // taps from the previous token wave's last three, handed over through LDS.
    if constexpr (TL::TW > 1) {
        if constexpr (TL::in_stages) lds_barrier();  // every wave is past its last stage read
        if (wn + 1 < TL::TW) {
            static_for<0, kWNT>([&](auto NT) {
                constexpr int nt = decltype(NT)::value;
                const int j = nloc0 + nt - (16 * kWNT * (wn + 1) - kHalo);  // 0..2 for the wave's last three tokens
                if (nt + kHalo >= kWNT || kWNT < kHalo) {
                    if (j >= 0) {
#pragma unroll
                        for (int mt = 0; mt < kWMT; ++mt)
                            *reinterpret_cast<lds_f32x4*>(smem + TL::off_hand +
                                                          ((wn * kHalo + j) * kMCols + cl0 + 4 * mt) * 4) = acc[mt][nt];
                    }
                }
            });
        }
        lds_barrier();
    }

    // Conv + SiLU per column quad, the results as packed bf16.
    u32x2 y[kWMT][kWNT];
    static_for<0, kWMT>([&](auto MT) {
        constexpr int mt = decltype(MT)::value;
        const int cb = c0 + cl0 + 4 * mt;
        const bool in = cb < p.D_out;
        const gdn_proj::ProjGroup gq = select_group(p, in ? cb : 0);
        if (!in || !gq.conv) {
#pragma unroll
            for (int nt = 0; nt < kWNT; ++nt) y[mt][nt] = pack4_bf16(acc[mt][nt]);
            return;
        }
        float w[4][4];  // [column][tap], taps right-aligned: tap 3 multiplies the current token
        if (p.conv_k == 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u32x4 q = wraw[mt][i >> 1];
                const uint32_t lo = q[2 * (i & 1)], hi = q[2 * (i & 1) + 1];
                w[i][0] = __uint_as_float(lo << 16);
                w[i][1] = __uint_as_float(lo & 0xffff0000u);
                w[i][2] = __uint_as_float(hi << 16);
                w[i][3] = __uint_as_float(hi & 0xffff0000u);
            }
        } else {
            const int cc = cb - gq.col0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int jw = j - (4 - p.conv_k);  // weight index of tap j
                    w[i][j] = jw >= 0 ? bf2f(p.conv_w[static_cast<size_t>(gq.cw_row0 + cc + i) * p.conv_k + jw]) : 0.f;
                }
        }
        // P of token nt - j of the lane's tokens: its own register, or, d
        // lanes down, that lane's; before the wave's first token the handed
        // over one (the tile's first tokens are halo: any value does).
        auto hand = [&](int j) {  // the j-th of the three tokens before the wave's, per lane
            if constexpr (TL::TW > 1)
                return wn > 0 ? *reinterpret_cast<const lds_f32x4*>(
                                    smem + TL::off_hand + (((wn - 1) * kHalo + j) * kMCols + cl0 + 4 * mt) * 4)
                              : f32x4{0.f, 0.f, 0.f, 0.f};
            else
                return f32x4{0.f, 0.f, 0.f, 0.f};
        };
        f32x4 before[kHalo];  // [j]: token j - 3 relative to the lane's first
        static_for<0, kHalo>([&](auto J) {
            constexpr int j = decltype(J)::value;
            constexpr int d = (kHalo - j + kWNT - 1) / kWNT;  // lanes down
            constexpr int nt = j - kHalo + d * kWNT;          // that lane's accumulator
            // lanes 0 .. d - 1 take token WNT n + j - 3 < 0 of the wave
            const f32x4 old = hand(kWNT >= kHalo ? j : min(kWNT * r16 + j, kHalo - 1));
#pragma unroll
            for (int i = 0; i < 4; ++i)
                before[j][i] = __int_as_float(__builtin_amdgcn_update_dpp(
                    __float_as_int(old[i]), __float_as_int(acc[mt][nt][i]), 0x110 + d, 0xf, 0xf, false));
        });
        static_for<0, kWNT>([&](auto NT) {
            constexpr int nt = decltype(NT)::value;
            auto tap = [&](auto Jc) {
                constexpr int t = nt - decltype(Jc)::value;
                if constexpr (t >= 0)
                    return acc[mt][t];
                else
                    return before[kHalo + t];
            };
            const f32x4 t0 = acc[mt][nt], t1 = tap(std::integral_constant<int, 1>{}),
                        t2 = tap(std::integral_constant<int, 2>{}), t3 = tap(std::integral_constant<int, 3>{});
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i)  // one order of sums in every tile
                v[i] = silu_f(fmaf(w[i][0], t3[i], fmaf(w[i][1], t2[i], fmaf(w[i][3], t0[i], w[i][2] * t1[i]))));
            y[mt][nt] = pack4_bf16(v);
        });
    });

    // New cache: P of rows t = T - ncache .. T - 1 of the extended sequence
    // (cache rows included when T < ncache).  A lane that holds all 3 of them
    // stores a quad's 24 bytes at once.
    if (!lean && any_lane((last_row & 0xffffu) != 0xffffu)) {
        static_for<0, kWMT>([&](auto MT) {
            constexpr int mt = decltype(MT)::value;
            const int cb = c0 + cl0 + 4 * mt;
            if (cb >= p.D_out) return;
            const gdn_proj::ProjGroup gq = select_group(p, cb);
            if (!gq.conv || !gq.cache_out) return;
            const bool quads = by_quad(gq.cache_out);
            int b = b0;
            static_for<0, kWNT>([&](auto NT) {
                constexpr int nt = decltype(NT)::value;
                b += begins(nt);
                const int j = (last_row >> (2 * nt)) & 3;
                if (j == 3) return;
                uint16_t* const dst = gq.cache_out + (static_cast<size_t>(b) * gq.width + cb - gq.col0) * ncache;
                const int first = nt - j;  // accumulator of the oldest of the three
                if (quads && first >= 0 && first + 2 < kWNT && nloc0 + first >= kHalo) {
                    if constexpr (nt >= 2) {
                        if (j == 2) {
                            const f32x4 o = acc[mt][nt - 2], m = acc[mt][nt - 1], n = acc[mt][nt];
                            u32x2* const d = reinterpret_cast<u32x2*>(dst);
                            d[0] = u32x2{pack2_bf16(o[0], m[0]), pack2_bf16(n[0], o[1])};
                            d[1] = u32x2{pack2_bf16(m[1], n[1]), pack2_bf16(o[2], m[2])};
                            d[2] = u32x2{pack2_bf16(n[2], o[3]), pack2_bf16(m[3], n[3])};
                        }
                    }
                    return;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) dst[i * ncache + j] = f2bf_bits(acc[mt][nt][i]);
            });
        });
    }

    // Stores.  Element index of (b, t, column cc) of a group: b width T_out +
    // t tstride + coff (token-major: tstride = width, coff = cc; head-major
    // [B, width/hd, T, hd]: tstride = hd, coff = (cc / hd) T hd + cc % hd);
    // packed, the token's offset in the packed outputs times tstride + coff.
    constexpr int kPair = kWMT > 1 ? 2 : 1;
    static_for<0, kWMT / kPair>([&](auto PR) {
        constexpr int m0 = decltype(PR)::value * kPair;
        const int cb = c0 + cl0 + 4 * m0;
        if (cb >= p.D_out) return;
        const gdn_proj::ProjGroup gq = select_group(p, cb);
        const bool wide = kPair == 2 && wide_group(gq);
        // rows in order, each told its address offset
        auto rows = [&](const gdn_proj::ProjGroup& g, auto&& put) {
            const int tstride = g.head_dim ? g.head_dim : g.width;
            const size_t seq = static_cast<size_t>(g.width) * p.T_out;
            auto orow = [&](int b, int t) {
                return packed ? static_cast<size_t>(tok0(b) + t) * tstride
                              : static_cast<size_t>(b) * seq + static_cast<size_t>(t) * tstride;
            };
            if (lean) {
                const size_t o = orow(b0, t30 - kHalo);
                static_for<0, kWNT>([&](auto NT) {
                    constexpr int nt = decltype(NT)::value;
                    if (nloc0 + nt >= kHalo) put(NT, o + static_cast<size_t>(nt) * tstride);
                });
            } else {
                int b = b0, t3 = t30;
                static_for<0, kWNT>([&](auto NT) {
                    constexpr int nt = decltype(NT)::value;
                    if (nt > 0) step(b, t3);
                    if (nloc0 + nt >= kHalo && R0 + nt < F3 && t3 >= kHalo) put(NT, orow(b, t3 - kHalo));
                });
            }
        };
        if (wide) {
            const int cc = cb - gq.col0, hd = gq.head_dim;
            uint16_t* const base = gq.dst + (hd ? static_cast<size_t>(cc / hd) * p.T_out * hd + cc % hd : static_cast<size_t>(cc));
            rows(gq, [&](auto NT, size_t o) {
                constexpr int nt = decltype(NT)::value;
                *reinterpret_cast<u32x4*>(base + o) =
                    u32x4{y[m0][nt][0], y[m0][nt][1], y[m0 + kPair - 1][nt][0], y[m0 + kPair - 1][nt][1]};
            });
        } else {
            // 4 columns at a time (a lane's 4 columns share a group): adjacent
            // in memory, or (head_dim 1..3) one by one.
            static_for<m0, m0 + kPair>([&](auto MT) {
                constexpr int mt = decltype(MT)::value;
                const int cm = c0 + cl0 + 4 * mt;
                if (cm >= p.D_out) return;
                const gdn_proj::ProjGroup gm = select_group(p, cm);
                const int cc = cm - gm.col0, hd = gm.head_dim;
                size_t coff[4];
                int h = hd ? cc / hd : 0, d = hd ? cc - h * hd : cc;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    coff[i] = hd ? static_cast<size_t>(h) * p.T_out * hd + d : static_cast<size_t>(cc + i);
                    if (hd && ++d == hd) {
                        d = 0;
                        ++h;
                    }
                }
                const bool vec = hd == 0 || (hd & 3) == 0;
                rows(gm, [&](auto NT, size_t o) {
                    constexpr int nt = decltype(NT)::value;
                    uint16_t* const row = gm.dst + o;
                    if (vec) {
                        *reinterpret_cast<u32x2*>(row + coff[0]) = y[mt][nt];
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) row[coff[i]] = static_cast<uint16_t>(y[mt][nt][i >> 1] >> (16 * (i & 1)));
                    }
                });
            });
        }
    });
}

}  // namespace

namespace gdn_proj {

// The tiles, largest first.
using Tile256x256 = ProjTile<4, 2, 4, 8, 2, 1, true>;
using Tile256x224 = ProjTile<4, 2, 4, 7, 2, 1, true>;
using Tile256x192 = ProjTile<4, 2, 4, 6, 2, 1, true>;
using Tile256x160 = ProjTile<4, 2, 4, 5, 3, 1, true>;
using Tile128x160 = ProjTile<4, 2, 2, 5, 4, 1, true>;
using Tile128x128Deep = ProjTile<4, 2, 2, 4, 4, 1>;
using Tile128x128 = ProjTile<4, 2, 2, 4, 2, 2>;
using Tile64x128Deep = ProjTile<2, 4, 2, 2, 4, 1>;
using Tile64x64Wide = ProjTile<4, 2, 1, 2, 4, 2>;
using Tile64x64 = ProjTile<2, 2, 2, 2, 4, 2>;
using Tile64x32 = ProjTile<2, 2, 2, 1, 3, 2, false, 1, 2>;
using Tile32x32 = ProjTile<2, 2, 1, 1, 3, 3, false, 1, 2>;
// Of the plain product, which sums K in KS groups of waves (the order of a sum
// follows KS alone).
using Plain32x32K4 = ProjTile<2, 2, 1, 1, 3, 1, false, 4>;
using Plain32x32K2 = ProjTile<2, 2, 1, 1, 3, 2, false, 2>;
using Plain64x32K4 = ProjTile<2, 2, 2, 1, 3, 1, false, 4>;
using Plain64x32K2 = ProjTile<2, 2, 2, 1, 3, 2, false, 2>;
using Plain64x64K4 = ProjTile<2, 2, 2, 2, 2, 1, false, 4>;
using Plain64x64K2 = ProjTile<2, 2, 2, 2, 3, 1, false, 2>;
using Plain64x128K2 = ProjTile<2, 2, 2, 4, 3, 1, false, 2>;

template <class TL, int MODE>
int launch_tile(const ProjParams& p, int F3, hipStream_t stream) {
    constexpr int outs = MODE == kPlain ? TL::toks : TL::outs;
    const int n_tok = (F3 + outs - 1) / outs, n_col = (p.D_out + TL::cols - 1) / TL::cols;
    const dim3 grid(static_cast<unsigned>(n_tok) * n_col), block(TL::waves * 64);
    hipLaunchKernelGGL((gdn_proj_conv_mfma_kernel<TL, MODE>), grid, block, 0, stream, p, n_tok, n_col);
    return gdn_host::check_launch("gdn_proj_conv_mfma_kernel");
}

// Launch tile number `tile` over F3 rows.
template <int MODE>
int launch_mfma_tile(int tile, const ProjParams& p, int F3, hipStream_t stream) {
    switch (tile) {
        case 1: return launch_tile<Tile256x224, MODE>(p, F3, stream);
        case 2: return launch_tile<Tile256x192, MODE>(p, F3, stream);
        case 3: return launch_tile<Tile256x160, MODE>(p, F3, stream);
        case 4: return launch_tile<Tile128x160, MODE>(p, F3, stream);
        case 5: return launch_tile<Tile128x128Deep, MODE>(p, F3, stream);
        case 6: return launch_tile<Tile128x128, MODE>(p, F3, stream);
        case 7: return launch_tile<Tile64x128Deep, MODE>(p, F3, stream);
        case 8: return launch_tile<Tile64x64Wide, MODE>(p, F3, stream);
        case 9: return launch_tile<Tile64x64, MODE>(p, F3, stream);
        case 10: return launch_tile<Tile64x32, MODE>(p, F3, stream);
        case 11: return launch_tile<Tile32x32, MODE>(p, F3, stream);
        default: return launch_tile<Tile256x256, MODE>(p, F3, stream);
    }
}
int launch_mfma_packed(int tile, const ProjParams& p, int F3, hipStream_t stream);  // proj_packed.hip

}  // namespace gdn_proj
