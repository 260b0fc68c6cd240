// Projection GEMM + causal depthwise conv (<= 4 taps) + SiLU, bf16 MFMA.
//
// Reference: kernels/fused_proj_conv_silu.cu:105-295 (WMMA, 125-token tile +
// 3-token halo, cp.async pipeline) and reference/fused_proj_conv_silu_ref.py
// for the math.  P = x W^T is accumulated in fp32 and never rounded before the
// conv (as the reference kernel does; the PyTorch reference rounds P to bf16).
//
// Two kernels:
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
// layout a lane holds 4 adjacent columns of one token, 16 tokens a tile: the
// conv taps are reads of a per-wave LDS window shifted by whole tokens.  The
// bf16 results go into an output tile in LDS (the stages) and leave as whole
// rows, 16 bytes per lane.
//
// gdn_proj_conv_kernel (general shapes: group boundaries not on 4 columns,
// unaligned outputs, K not a multiple of 64) computes 128 x 128 tiles of P whose rows are
// tokens t0-3 .. t0+124 of one sequence and parks P in LDS for the conv.
//
// Output routing: up to 5 column groups, each written either token-major
// [B, T, width] or head-major [B, width/hd, T, hd], with or without the
// conv + SiLU (a plain projection takes the current token's row of P).
#include <cstddef>
#include <type_traits>

#include "gdn_common.hpp"
#include "proj.hpp"

namespace {

using namespace gdn;

constexpr int kBM = 128, kBN = 128, kBK = 64;
constexpr int kHalo = 3;
constexpr int kOutT = kBM - kHalo;  // 125 outputs per tile
constexpr int kLD = kBK + 8;        // padded LDS row, bf16
constexpr int kPLD = kBN + 4;       // padded LDS row, fp32 epilogue

__device__ __forceinline__ int group_of(const gdn_proj::ProjParams& p, int c) {
    int gi = 0;
#pragma unroll
    for (int q = 1; q < gdn_proj::kMaxGroups; ++q)
        if (q < p.ngroups && c >= p.groups[q].col0) gi = q;
    return gi;
}

__global__ __launch_bounds__(256, 2) void gdn_proj_conv_kernel(gdn_proj::ProjParams p) {
    const int tile_t = blockIdx.x, tile_c = blockIdx.y, b = blockIdx.z;
    const int t0 = tile_t * kOutT;
    const int c0 = tile_c * kBN;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = wave >> 1, wn = wave & 1;
    const int m16 = lane & 15, g4 = lane >> 4;

    // Union: two K stages of A/B tiles, or the fp32 P tile in the epilogue.
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * 2 * kBM * kLD * 2 > kBM * kPLD * 4
                                                                 ? 2 * 2 * kBM * kLD * 2
                                                                 : kBM * kPLD * 4];
    bf16(*As)[kBM][kLD] = reinterpret_cast<bf16(*)[kBM][kLD]>(smem);
    bf16(*Bs)[kBM][kLD] = reinterpret_cast<bf16(*)[kBM][kLD]>(smem + 2 * kBM * kLD * 2);
    float(*Pt)[kPLD] = reinterpret_cast<float(*)[kPLD]>(smem);

    // Each thread moves 4 A chunks and 4 B chunks (16 B) per K step.
    u32x4 ra[4], rb[4];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int idx = tid + 256 * u;
            const int row = idx >> 3, c8 = (idx & 7) * 8;
            const int tok = t0 - kHalo + row;
            ra[u] = (tok >= 0 && tok < p.T)
                        ? *reinterpret_cast<const u32x4*>(p.x + (static_cast<size_t>(b) * p.T + tok) * p.D + k0 + c8)
                        : u32x4{0u, 0u, 0u, 0u};
            const int col = c0 + row;
            rb[u] = col < p.D_out ? *reinterpret_cast<const u32x4*>(p.W + static_cast<size_t>(col) * p.D + k0 + c8)
                                  : u32x4{0u, 0u, 0u, 0u};
        }
    };
    auto lstore = [&](int st) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int idx = tid + 256 * u;
            const int row = idx >> 3, c8 = (idx & 7) * 8;
            *reinterpret_cast<u32x4*>(&As[st][row][c8]) = ra[u];
            *reinterpret_cast<u32x4*>(&Bs[st][row][c8]) = rb[u];
        }
    };

    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nk = p.D / kBK;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int st = kt & 1;
        if (kt + 1 < nk) gload((kt + 1) * kBK);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            bf16x8 af[4], bfr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                af[i] = *reinterpret_cast<const bf16x8*>(&As[st][64 * wm + 16 * i + m16][32 * s + 8 * g4]);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bfr[j] = *reinterpret_cast<const bf16x8*>(&Bs[st][64 * wn + 16 * j + m16][32 * s + 8 * g4]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mfma16x16x32(af[i], bfr[j], acc[i][j]);
        }
        if (kt + 1 < nk) lstore(st ^ 1);
        __syncthreads();
    }

    // Epilogue: P tile to LDS (the staging buffers are dead after the last barrier).
    // In the first tile, halo rows of tokens < 0 take the group's cached
    // projections when it has a cache (x rows there are zero, so P is 0).
    const int ncache = p.conv_k - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 64 * wm + 16 * i + 4 * g4 + e, col = 64 * wn + 16 * j + m16;
                float val = acc[i][j][e];
                if (t0 == 0 && row < kHalo && row >= kHalo - ncache && c0 + col < p.D_out) {
                    const gdn_proj::ProjGroup& gq = p.groups[group_of(p, c0 + col)];
                    if (gq.conv && gq.cache_in)
                        val = bf2f(gq.cache_in[(static_cast<size_t>(b) * gq.width + (c0 + col - gq.col0)) * ncache +
                                               (row - (kHalo - ncache))]);
                }
                Pt[row][col] = val;
            }
    __syncthreads();

    const int cl = tid & (kBN - 1);
    const int c = c0 + cl;
    if (c >= p.D_out) return;
    const gdn_proj::ProjGroup grp = p.groups[group_of(p, c)];
    const int cc = c - grp.col0;
    // The workgroup holding the last token refreshes the cache: bf16(P) of
    // tokens T-ncache .. T-1 (rows of negative tokens hold the old cache).
    if (grp.conv && grp.cache_out && tid < kBN && t0 + kOutT >= p.T) {
        for (int j = 0; j < ncache; ++j) {
            const int tok = p.T - ncache + j;
            grp.cache_out[(static_cast<size_t>(b) * grp.width + cc) * ncache + j] = f2bf_bits(Pt[tok - t0 + kHalo][cl]);
        }
    }
    float w[4] = {0.f, 0.f, 0.f, 0.f};
    if (grp.conv) {
        // Taps aligned to the right: tap conv_k-1 multiplies the current token.
        for (int j = 0; j < p.conv_k; ++j) w[4 - p.conv_k + j] = bf2f(p.conv_w[static_cast<size_t>(grp.cw_row0 + cc) * p.conv_k + j]);
    }
    for (int tl = tid >> 7; tl < kOutT; tl += 2) {
        const int t = t0 + tl;
        if (t >= p.T) break;
        float y;
        if (grp.conv) {
            const float s = w[0] * Pt[tl][cl] + w[1] * Pt[tl + 1][cl] + w[2] * Pt[tl + 2][cl] + w[3] * Pt[tl + 3][cl];
            y = s / (1.f + expf(-s));
        } else {
            y = Pt[tl + kHalo][cl];
        }
        size_t idx;
        if (grp.head_dim > 0) {
            const int hh = cc / grp.head_dim, dd = cc % grp.head_dim;
            idx = ((static_cast<size_t>(b) * (grp.width / grp.head_dim) + hh) * p.T_out + t) * grp.head_dim + dd;
        } else {
            idx = (static_cast<size_t>(b) * p.T_out + t) * grp.width + cc;
        }
        grp.dst[idx] = f2bf_bits(y);
    }
}


// ---------------------------------------------------------------------------
// Fast path: transposed MFMA tiles, DMA staging, register epilogue.
// ---------------------------------------------------------------------------
constexpr int kMK = 64;          // K per stage: one 128-byte line per row
constexpr int kMRowB = kMK * 2;  // 128 bytes per staged row

// A workgroup's tile: CW x TW waves, each WMT 16-column x WNT 16-token MFMA
// tiles, NS K stages in LDS, PER_CU workgroups on a CU.
// PHASED: the two-group main loop (eight waves, one workgroup on a CU).
template <int CW_, int TW_, int WMT_, int WNT_, int NS_, int PER_CU_, bool PHASED_ = false>
struct ProjTile {
    static constexpr bool PHASED = PHASED_;
    static constexpr int CW = CW_, TW = TW_, WMT = WMT_, WNT = WNT_, NS = NS_, PER_CU = PER_CU_;
    static constexpr int cols = 16 * CW * WMT;   // output columns (W rows) per workgroup
    static constexpr int toks = 16 * TW * WNT;   // token rows per workgroup
    static constexpr int outs = toks - kHalo;    // tokens written per workgroup
    static constexpr int waves = CW * TW;
    static constexpr int stage_b = (cols + toks) * kMRowB;    // W rows, then x rows
    static constexpr int dma = (cols + toks) / 8 / waves;     // 1 KiB copies (8 rows) per wave per stage
    static_assert(PHASED || (cols + toks) % (8 * waves) == 0, "copies split evenly");
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
    // Epilogue LDS: the bf16 output tile; the hand-over area (the last
    // 16-token fp32 tile of each token wave but the last); the conv windows,
    // for each wave and column quad a strip of 32 16-byte slots (slots 0..2:
    // the previous 16-token tile's last 3 tokens, 3..18: the current tile's
    // tokens, fp32 x 4 columns), so a tap is a plain b128 read shifted by
    // whole slots, conflict free like a linear read.
    static constexpr int out_b = toks * cols * 2;
    static constexpr int hand_b = CW * (TW - 1) * WMT * 1024;
    static constexpr int conv_b = waves * 4 * 32 * 16;
    // All three lie in the dead stages where they fit (one more barrier),
    // else the hand-over and windows get an area of their own.
    static constexpr bool in_stages = out_b + hand_b + conv_b <= NS * stage_b;
    static_assert(out_b <= NS * stage_b, "the stages hold the bf16 output tile");
    static constexpr int off_hand = in_stages ? out_b : NS * stage_b;
    static constexpr int off_conv = off_hand + hand_b;
    static constexpr int lds_b = in_stages ? NS * stage_b : NS * stage_b + hand_b + conv_b;
    static_assert(lds_b * PER_CU <= 160 * 1024, "LDS");
    static constexpr int units = cols / 16;  // 32-byte units of an output row
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

// Groups whose output goes out through the LDS output tile in 16-byte
// chunks: 8-column aligned, 8-column head_dim (or token-major), 16-byte
// aligned destination.
__device__ __forceinline__ bool staged_group(const gdn_proj::ProjGroup& g) {
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

// PACKED: sequences of unequal lengths (ProjParams::packed > 0), rows mapped
// through the row table; a separate instantiation, so the equal-length kernel
// carries none of that code.
template <class TL, bool PACKED>
__global__ __launch_bounds__(TL::waves * 64)
    __attribute__((amdgpu_waves_per_eu(TL::PER_CU * TL::waves / 4, TL::PER_CU * TL::waves / 4))) void gdn_proj_conv_mfma_kernel(
        gdn_proj::ProjParams p, int n_tok, int n_col) {
    constexpr int kMCols = TL::cols, kMToks = TL::toks, kMOut = TL::outs, kMWaves = TL::waves, kMStages = TL::NS;
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
    const int T3 = p.T + kHalo;
    constexpr bool packed = PACKED;
    const kconst_i32* prow = packed_rows();
    const int nseq = packed ? p.packed : p.B;
    const int F3 = packed ? prow[p.packed] : p.B * T3;
    const int f0 = tile_t * kMOut - kHalo;  // row of tile row 0 (>= -3; rows < 0 are never used)
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
    const int wm = wave / TL::TW, wn = wave % TL::TW;             // column slice, token slice
    const int r16 = lane & 15, g4 = lane >> 4;

    // x row feeding row r: the token itself, the sequence's first token for
    // cache rows, clamped at both ends (those products are never used).
    auto xrow_of = [&](int r) {
        if constexpr (PACKED) {
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

    // DMA sources.  Copy j of a wave moves staged rows 8 q .. 8 q + 7 with
    // q = wave + 8 j (q < 32: W rows, else x rows); lane l takes row 8 q + l / 8
    // and fills slot l % 8 with chunk (l % 8) ^ swz(row): every 8 lanes read
    // one whole 128-byte line.  Columns >= D_out are clamped to a valid row;
    // their products are never stored.
    const int xrow0 = xrow_of(f0);
    const unsigned char* wsrc = reinterpret_cast<const unsigned char*>(p.W + static_cast<size_t>(c0) * p.D);
    const unsigned char* xsrc = reinterpret_cast<const unsigned char*>(p.x + static_cast<size_t>(xrow0) * p.D);
    auto src_off = [&](int srow) {
        const int row = srow < kMCols ? min(c0 + srow, p.D_out - 1) - c0 : xrow_of(f0 + srow - kMCols) - xrow0;
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
            crow[j] = 8 * (wave + kMWaves * j);
            voff[j] = src_off(crow[j] + (lane >> 3));
        }
    }
    auto issue_copy = [&](int stage, int kk, int j) {
        const unsigned char* src = (crow[j] < kMCols ? wsrc : xsrc) + kk * kMRowB;
        dma16(src, voff[j], smem + stage * kMStageB + crow[j] * kMRowB);
    };
    auto issue = [&](int stage, int kk) {
#pragma unroll
        for (int j = 0; j < kCopies; ++j) issue_copy(stage, kk, j);
    };
    // Half `half` of a stage's copies.
    auto issue_part = [&](int stage, int kk, int half) {
#pragma unroll
        for (int j = 0; j < kCopies; ++j)
            if ((j >= (kCopies + 1) / 2) == (half == 1)) issue_copy(stage, kk, j);
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
        const int cb = c0 + 16 * kWMT * wm + 16 * mt + 4 * g4;
        if (cb < p.D_out && p.conv_k == 4) {
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

    const int nk = p.D / kMK;
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
            // Stage kt has landed (later ones may be in flight; the last NS - 2
            // stages wait for every copy).
            if (kMStages > 2 && next)
                wait_vm<(kMStages - 2) * kMDma>();
            else
                wait_vm<0>();
            lds_barrier();  // for every wave; the buffer of stage kt - 1 is fully read
            // The new stage's copies go out in two halves, one before each K
            // half's MFMAs: a wave that issues all of them at once stalls on
            // the copy queue before its first MFMA.
            const lds_u8* st = smem + rs * kMStageB;
            static_for<0, 2>([&](auto H) {
                constexpr int h = decltype(H)::value;
                if (next) issue_part(ws, kt + kMStages - 1, h);
                bf16x8 a[kWMT], bx[kWNT];
                static_for<0, kWMT>([&](auto MT) {
                    constexpr int mt = decltype(MT)::value;
                    a[mt] = *reinterpret_cast<const lds_bf16x8*>(st + (16 * kWMT * wm + 16 * mt) * kMRowB + rd[h]);
                });
                static_for<0, kWNT>([&](auto NT) {
                    constexpr int nt = decltype(NT)::value;
                    bx[nt] = *reinterpret_cast<const lds_bf16x8*>(st + (kMCols + 16 * kWNT * wn + 16 * nt) * kMRowB + rd[h]);
                });
#pragma unroll
                for (int nt = 0; nt < kWNT; ++nt)
#pragma unroll
                    for (int mt = 0; mt < kWMT; ++mt) acc[mt][nt] = mfma16x16x32(a[mt], bx[nt], acc[mt][nt]);
            });
            rs = rs + 1 == kMStages ? 0 : rs + 1;
            ws = ws + 1 == kMStages ? 0 : ws + 1;
        }
    }

    // Token waves meet inside the tile: a wave's first 16-token tile takes
    // its conv taps from the previous token wave's last one, handed over
    // through LDS (the stages become the output tile below).
    if constexpr (TL::in_stages) lds_barrier();  // every wave is past its last stage read
    auto hand = [&](int w, int mt) { return smem + TL::off_hand + ((w * TL::CW + wm) * kWMT + mt) * 1024 + lane * 16; };
    if (wn + 1 < TL::TW) {
#pragma unroll
        for (int mt = 0; mt < kWMT; ++mt) *reinterpret_cast<lds_f32x4*>(hand(wn, mt)) = acc[mt][kWNT - 1];
    }
    lds_barrier();  // hand-over written; every wave is past its last stage read

    // This lane's row in token tile 0 of the wave, as (b, t3 = t + 3); tile
    // nt adds 16 rows.  Rows before local row kHalo are the tile's halo.
    const int nloc0 = 16 * kWNT * wn + r16;
    auto split = [&](int r, int& b, int& t3) {
        if (r < 0) {
            b = 0;
            t3 = r;
        } else {
            locate(r, b, t3);
        }
    };
    int b0, t30;
    split(f0 + nloc0, b0, t30);
    int bx, t3x;  // row of the handed-over tile (16 rows before tile 0)
    split(f0 + nloc0 - 16, bx, t3x);
    const int ncache = p.conv_k - 1;
    // Lean epilogue when the wave's 16 kWNT rows are all tokens of one
    // sequence (no cache rows, no sequence start) and none of them is in the
    // conv cache refresh window (the last ncache tokens).
    bool lean;
    {
        const int R0 = f0 + 16 * kWNT * wn;
        int bR, t3R;
        split(R0, bR, t3R);
        lean = R0 >= 0 && R0 + 16 * kWNT <= F3 && t3R >= kHalo && t3R + 16 * kWNT <= len3(bR) - ncache;
    }

    // Output tile in LDS (the stages): row = token of the tile (its columns
    // as bf16), 32-byte unit u of a row stored at unit u ^ (row % units), so
    // the 16 tokens of a fragment write spread over the banks and a row reads
    // back whole.
    lds_u8* const otile = smem;
    auto ounit = [](int row, int u) { return row * kMCols * 2 + ((u ^ (row & (TL::units - 1))) << 5); };

    static_for<0, kWMT>([&](auto MT) {
        constexpr int mt = decltype(MT)::value;
        const int cb = c0 + 16 * kWMT * wm + 16 * mt + 4 * g4;  // this lane's 4 columns (same for the tile's 16 tokens)
        if (cb >= p.D_out) return;
        const gdn_proj::ProjGroup gq = select_group(p, cb);
        const int cc = cb - gq.col0, width = gq.width, hd = gq.head_dim;
        const bool conv = gq.conv != 0;
        const bool staged = staged_group(gq);
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
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int jw = j - (4 - p.conv_k);  // weight index of tap j
                    w[i][j] = conv && jw >= 0
                                  ? bf2f(p.conv_w[static_cast<size_t>(gq.cw_row0 + cc + i) * p.conv_k + jw])
                                  : 0.f;
                }
        }
        // Cache row (t < 0) of a conv group: the cached projection of token t
        // (cache index t + ncache, oldest first), zero before the cache or
        // without one.
        auto cache_row = [&](f32x4 v, int b, int t3) {
            const int q = t3 - kHalo + ncache;
            if (conv && t3 < kHalo) {
                const uint16_t* cin = gq.cache_in;
                const bool has = cin != nullptr && q >= 0;
                // rows past the last sequence (in the last tile; never stored)
                // read the last sequence's entries, not past the buffer
                const uint16_t* src =
                    has ? cin + (static_cast<size_t>(min(b, nseq - 1)) * width + cc) * ncache + q : nullptr;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = has ? bf2f(src[i * ncache]) : 0.f;
            }
            return v;
        };
        f32x4 pv = f32x4{0.f, 0.f, 0.f, 0.f};
        if (wn > 0) pv = cache_row(*reinterpret_cast<const lds_f32x4*>(hand(wn - 1, mt)), bx, t3x);
        // This lane's conv window strip; the previous tile's last 3 tokens
        // (lanes 13..15) go to slots 0..2.
        lds_u8* const cw = smem + TL::off_conv + (wave * 4 + g4) * 512;
        if (conv && r16 >= 13) *reinterpret_cast<lds_f32x4*>(cw + (r16 - 13) * 16) = pv;
        // The window is shared by the wave's lanes, which the compiler's
        // per-lane view does not see: these fences keep its accesses in
        // program order (the hardware then runs them in order).
        asm volatile("" ::: "memory");
        // Unstaged groups (head_dim 1..3 or 4-column aligned only) store from
        // registers.  Element index of (b, t, column cc + i): b width T + t
        // tstride + coff[i] (token-major: tstride = width, coff = cc + i;
        // head-major [B, width/hd, T, hd]: tstride = hd, coff = ((cc + i) /
        // hd) T hd + (cc + i) % hd).
        const size_t seq = static_cast<size_t>(width) * p.T_out;
        const int tstride = hd ? hd : width;
        // token t of sequence b: b width T_out + t tstride, or, packed, its
        // token offset in the packed outputs times tstride
        auto orow = [&](int b, int t) {
            return packed ? static_cast<size_t>(tok0(b) + t) * tstride
                          : static_cast<size_t>(b) * seq + static_cast<size_t>(t) * tstride;
        };
        const bool vec = hd == 0 || (hd & 3) == 0;  // the 4 columns are adjacent in memory
        size_t coff[4] = {0, 0, 0, 0};
        if (!staged) {
            int h = hd ? cc / hd : 0, d = hd ? cc - h * hd : cc;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                coff[i] = hd ? static_cast<size_t>(h) * p.T_out * hd + d : static_cast<size_t>(cc + i);
                if (hd && ++d == hd) {
                    d = 0;
                    ++h;
                }
            }
        }
        auto store = [&](uint16_t* row, const float (&y)[4]) {
            if (vec) {
                *reinterpret_cast<u32x2*>(row + coff[0]) = u32x2{pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3])};
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) row[coff[i]] = f2bf_bits(y[i]);
            }
        };
        const int unit = kWMT * wm + mt;  // 32-byte unit of the output row holding this fragment's columns
        int b = b0, t3 = t30;
        static_for<0, kWNT>([&](auto NT) {
            constexpr int nt = decltype(NT)::value;
            if (nt > 0 && !lean) {
                t3 += 16;
                if (packed) {
                    while (b + 1 < p.packed && t3 >= len3(b)) {
                        t3 -= len3(b);
                        ++b;
                    }
                } else if (t3 >= T3) {
                    b += t3 / T3;
                    t3 %= T3;
                }
            }
            const int nloc = nloc0 + 16 * nt;
            f32x4 cur = acc[mt][nt];
            if (!lean) cur = cache_row(cur, b, t3);
            // conv + SiLU (plain groups: the current row)
            float y[4];
            if (conv) {
                // Taps through the window: tokens n - 1, n - 2, n - 3 are
                // slots n + 2, n + 1, n (one wave: its LDS accesses run in
                // order, so the reads see this tile's writes and the slide of
                // the last 3 tokens to slots 0..2 comes after every read).
                *reinterpret_cast<lds_f32x4*>(cw + (3 + r16) * 16) = cur;
                asm volatile("" ::: "memory");
                const f32x4 t1 = *reinterpret_cast<const lds_f32x4*>(cw + (2 + r16) * 16);
                const f32x4 t2 = *reinterpret_cast<const lds_f32x4*>(cw + (1 + r16) * 16);
                const f32x4 t3v = *reinterpret_cast<const lds_f32x4*>(cw + r16 * 16);
                asm volatile("" ::: "memory");
                if (r16 >= 13) *reinterpret_cast<lds_f32x4*>(cw + (r16 - 13) * 16) = cur;
                asm volatile("" ::: "memory");
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float s = w[i][3] * cur[i] + w[i][2] * t1[i] + w[i][1] * t2[i] + w[i][0] * t3v[i];
                    y[i] = silu_f(s);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = cur[i];
            }
            if (staged) {
                *reinterpret_cast<lds_u32x2*>(otile + ounit(nloc, unit) + 8 * g4) =
                    u32x2{pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3])};
            } else if (lean) {
                if (!(nt == 0 && nloc0 < kHalo))  // the tile's halo rows
                    store(gq.dst + orow(b0, t30 - kHalo + 16 * nt), y);
            } else if (nloc >= kHalo && f0 + nloc < F3 && t3 >= kHalo) {
                store(gq.dst + orow(b, t3 - kHalo), y);
            }
            // New cache: rows t = T - ncache .. T - 1 of the extended sequence
            // (cache rows included when T < ncache).
            const int Tb = len3(b) - kHalo;
            if (!lean && conv && gq.cache_out && nloc >= kHalo && f0 + nloc < F3 && t3 - kHalo >= Tb - ncache) {
                const int t = t3 - kHalo;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    gq.cache_out[(static_cast<size_t>(b) * width + cc + i) * ncache + (t - (Tb - ncache))] =
                        f2bf_bits(cur[i]);
            }
        });
    });
    lds_barrier();  // output tile complete

    // Store the tile's staged columns row by row: thread tid takes one
    // 16-byte chunk (8 columns) of every kRows-th tile row, so a wave writes
    // whole rows per instruction (256 columns: two 512-byte rows, or, for
    // head-major groups, two 256-byte token rows of each head).
    {
        constexpr int kChunks = kMCols / 8, kRows = kMWaves * 64 / kChunks;
        const int j = tid % kChunks;
        const int c = c0 + 8 * j;
        if (c >= p.D_out) return;
        const gdn_proj::ProjGroup gq = select_group(p, c);
        if (!staged_group(gq)) return;
        const int cc = c - gq.col0, hd = gq.head_dim;
        const size_t seq = static_cast<size_t>(gq.width) * p.T_out;
        const size_t tstride = hd ? hd : gq.width;
        uint16_t* const colp = gq.dst + (hd ? static_cast<size_t>(cc / hd) * p.T_out * hd + cc % hd : static_cast<size_t>(cc));
        const int row0 = tid / kChunks;
        int b, t3;
        split(f0 + row0, b, t3);
#pragma unroll 4
        for (int i = 0; i < (kMToks + kRows - 1) / kRows; ++i) {
            const int row = row0 + kRows * i;
            if (i > 0) {
                t3 += kRows;
                while ((!packed || b + 1 < p.packed) && t3 >= len3(b)) {
                    t3 -= len3(b);
                    ++b;
                }
            }
            if (row >= kHalo && row < kMToks && f0 + row < F3 && t3 >= kHalo) {
                const u32x4 v = *reinterpret_cast<const lds_u32x4*>(otile + ounit(row, j >> 1) + 16 * (j & 1));
                const size_t o = packed ? static_cast<size_t>(tok0(b) + t3 - kHalo) * tstride
                                        : static_cast<size_t>(b) * seq + static_cast<size_t>(t3 - kHalo) * tstride;
                *reinterpret_cast<u32x4*>(colp + o) = v;
            }
        }
    }
}

}  // namespace

namespace gdn_proj {

// The fast kernel needs every group to start on a 4-column boundary (a lane's
// 4 columns share a group), 8-byte aligned outputs for its vector stores,
// 16-byte aligned conv weights (read 4 columns x 4 taps at a time) and 32-bit
// DMA offsets.
static_assert(kCacheRows == kHalo, "row space");
constexpr int kMaxToks = 256;  // token rows of the largest tile

bool mfma_path_ok(const ProjParams& p) {
    if (p.D % kMK != 0 || p.D_out % 4 != 0) return false;
    if (!gdn_host::aligned(p.conv_w, 16)) return false;
    if (static_cast<long long>(p.D_out) * p.D * 2 >= (1ll << 31)) return false;
    if (static_cast<long long>(kMaxToks) * p.D * 2 >= (1ll << 31)) return false;
    if (static_cast<long long>(p.B) * (p.T + kHalo) >= (1ll << 30)) return false;
    if (p.packed < 0 || p.packed > kPackMax) return false;
    for (int g = 0; g < p.ngroups; ++g) {
        const ProjGroup& q = p.groups[g];
        if (q.col0 % 4 != 0 || q.width % 4 != 0 || q.cw_row0 % 4 != 0) return false;
        // 8-byte stores where a lane's 4 columns are adjacent in memory;
        // head_dim 1..3 (the layer's a/b) stores element by element.
        const bool vec = q.head_dim == 0 || q.head_dim % 4 == 0;
        if (!gdn_host::aligned(q.dst, vec ? 8 : 2)) return false;
    }
    return true;
}

// The tiles of the MFMA kernel and what a CU takes for them, in us: one
// workgroup alone (a1 + b1 per 64-wide K stage) and PER_CU = 2 of them side by
// side (a2 + b2 per stage; for PER_CU = 1 twice one).  Least squares over
// 256 CUs x 1..4 tiles each at D = 1024, 2048 and 4096 (T with whole tiles,
// D_out = 1024 or 2048).  What bounds a stage is the copies' entry into LDS
// (~27-30 B/clk per CU while fragments are read) and, with few stages in
// flight, their latency, so a small tile streams its operands in a third of
// the time of a large one and a large tile does more per byte.
using Tile256x256 = ProjTile<4, 2, 4, 8, 2, 1, true>;
using Tile256x128 = ProjTile<4, 2, 4, 4, 3, 1, true>;
using Tile128x128 = ProjTile<2, 2, 4, 4, 2, 2>;
using Tile64x128 = ProjTile<2, 2, 2, 4, 3, 2>;
using Tile64x64 = ProjTile<2, 2, 2, 2, 4, 2>;
using Tile32x128 = ProjTile<2, 2, 1, 4, 4, 2>;
using Tile32x64 = ProjTile<2, 2, 1, 2, 6, 2>;
using Tile32x32 = ProjTile<2, 2, 1, 1, 8, 2>;

struct TileCost {
    int cols, outs;
    float a1, b1, a2, b2;
};
template <class TL>
constexpr TileCost cost_of(float a1, float b1, float a2, float b2) {
    return TileCost{TL::cols, TL::outs, a1, b1, a2, b2};
}
constexpr TileCost kTileCost[] = {
    cost_of<Tile256x256>(20.f, 1.45f, 40.f, 2.9f),     cost_of<Tile256x128>(12.f, 0.91f, 24.f, 1.82f),
    cost_of<Tile128x128>(10.5f, 0.75f, 13.8f, 0.87f),  cost_of<Tile64x128>(7.8f, 0.44f, 8.7f, 0.555f),
    cost_of<Tile64x64>(6.f, 0.27f, 6.f, 0.355f),       cost_of<Tile32x128>(6.2f, 0.335f, 5.8f, 0.425f),
    cost_of<Tile32x64>(4.2f, 0.235f, 4.7f, 0.277f),    cost_of<Tile32x32>(3.8f, 0.197f, 3.7f, 0.235f),
};

// The tile whose busiest CU finishes first: its tiles run in pairs, the odd
// one alone.  Every tile sums K in the same order, so the choice does not
// change a bit of the result.  At D = 2048 and 6176 columns, against
// 256 x 256 tiles for everything: 1 token 66 -> 10.3 us, 77 tokens 61.9 ->
// 14.3, 253 tokens 61.4 -> 18.5, 509 tokens 61.9 -> 26.9, 1000 tokens 63.8 ->
// 41.5, 3000 tokens 125 -> 110; the choice was within 7% of the best of the
// eight on each of 60 sizes (1 to 16384 tokens, 2048 to 8224 columns).
int choose_tile(int F3, int D, int D_out) {
    constexpr long long kCUs = 256;
    const float nk = static_cast<float>(D / kMK);
    int best = 0;
    float best_us = 0.f;
    for (int i = 0; i < static_cast<int>(sizeof(kTileCost) / sizeof(kTileCost[0])); ++i) {
        const TileCost& t = kTileCost[i];
        const long long tiles = static_cast<long long>((F3 + t.outs - 1) / t.outs) * ((D_out + t.cols - 1) / t.cols);
        const long long n = (tiles + kCUs - 1) / kCUs;
        const float us = static_cast<float>(n / 2) * (t.a2 + t.b2 * nk) + static_cast<float>(n % 2) * (t.a1 + t.b1 * nk);
        if (i == 0 || us < best_us) {
            best = i;
            best_us = us;
        }
    }
    return best;
}

template <class TL>
int launch_tile(const ProjParams& p, int F3, hipStream_t stream) {
    const int n_tok = (F3 + TL::outs - 1) / TL::outs, n_col = (p.D_out + TL::cols - 1) / TL::cols;
    const dim3 grid(static_cast<unsigned>(n_tok) * n_col), block(TL::waves * 64);
    if (p.packed > 0)
        hipLaunchKernelGGL((gdn_proj_conv_mfma_kernel<TL, true>), grid, block, 0, stream, p, n_tok, n_col);
    else
        hipLaunchKernelGGL((gdn_proj_conv_mfma_kernel<TL, false>), grid, block, 0, stream, p, n_tok, n_col);
    return gdn_host::check_launch("gdn_proj_conv_mfma_kernel");
}

int launch_mfma(const ProjParams& p, int F3, hipStream_t stream) {
    const int tile = choose_tile(F3, p.D, p.D_out);
    switch (tile) {
        case 1: return launch_tile<Tile256x128>(p, F3, stream);
        case 2: return launch_tile<Tile128x128>(p, F3, stream);
        case 3: return launch_tile<Tile64x128>(p, F3, stream);
        case 4: return launch_tile<Tile64x64>(p, F3, stream);
        case 5: return launch_tile<Tile32x128>(p, F3, stream);
        case 6: return launch_tile<Tile32x64>(p, F3, stream);
        case 7: return launch_tile<Tile32x32>(p, F3, stream);
        default: return launch_tile<Tile256x256>(p, F3, stream);
    }
}

int launch_proj(const ProjParams& pin, hipStream_t stream) {
    ProjParams p = pin;
    if (p.T_out < p.T) p.T_out = p.T;
    if (p.packed > 0) {
        // Packed sequences: the MFMA kernel only (callers check mfma_path_ok
        // first); rows: kHalo cache rows + the tokens of every sequence.
        if (!mfma_path_ok(p)) return gdn_host::fail(GDN_ERR_UNSUPPORTED, "proj: packed launch off the MFMA path");
        return launch_mfma(p, p.row_off[p.packed], stream);
    }
    if (p.B == 0 || p.T == 0 || p.D_out == 0) return GDN_OK;
    // rows: kHalo cache rows + T tokens per sequence
    if (mfma_path_ok(p)) return launch_mfma(p, p.B * (p.T + kHalo), stream);
    const dim3 grid((p.T + kOutT - 1) / kOutT, (p.D_out + kBN - 1) / kBN, p.B);
    hipLaunchKernelGGL(gdn_proj_conv_kernel, grid, dim3(256), 0, stream, p);
    return gdn_host::check_launch("gdn_proj_conv_kernel");
}

}  // namespace gdn_proj

extern "C" int gdn_proj_conv_silu_hip(const gdn_bf16_t* x, const gdn_bf16_t* W, const gdn_bf16_t* conv_w,
                                      gdn_bf16_t* out, int B, int T, int D, int D_out, int conv_k, void* stream) {
    using gdn_host::aligned;
    using gdn_host::fail;
    if (B < 0 || T < 0 || D <= 0 || D_out <= 0)
        return fail(GDN_ERR_INVALID_ARGUMENT, "proj: B=%d T=%d D=%d D_out=%d", B, T, D, D_out);
    if (D % 64 != 0) return fail(GDN_ERR_UNSUPPORTED, "proj: D=%d must be a multiple of 64", D);
    if (D_out % 16 != 0) return fail(GDN_ERR_UNSUPPORTED, "proj: D_out=%d must be a multiple of 16", D_out);
    if (conv_k < 1 || conv_k > 4) return fail(GDN_ERR_UNSUPPORTED, "proj: conv_k=%d must be in 1..4", conv_k);
    if (B == 0 || T == 0) return GDN_OK;
    if (!x || !W || !conv_w || !out) return fail(GDN_ERR_INVALID_ARGUMENT, "proj: null pointer argument");
    if (!aligned(x, 16) || !aligned(W, 16)) return fail(GDN_ERR_INVALID_ARGUMENT, "proj: x/W need 16-byte alignment");
    gdn_proj::ProjParams p = {};
    p.x = x;
    p.W = W;
    p.conv_w = conv_w;
    p.B = B;
    p.T = T;
    p.D = D;
    p.D_out = D_out;
    p.conv_k = conv_k;
    p.ngroups = 1;
    p.groups[0] = gdn_proj::ProjGroup{0, D_out, 0, 1, 0, out, nullptr, nullptr};
    return gdn_proj::launch_proj(p, static_cast<hipStream_t>(stream));
}
