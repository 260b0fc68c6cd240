// Projection GEMM + causal depthwise conv (<= 4 taps) + SiLU, bf16 MFMA.
//
// Reference: kernels/fused_proj_conv_silu.cu:105-295 (WMMA, 125-token tile +
// 3-token halo, cp.async pipeline) and reference/fused_proj_conv_silu_ref.py
// for the math.  P = x W^T is accumulated in fp32 and never rounded before the
// conv (as the reference kernel does; the PyTorch reference rounds P to bf16).
//
// Two kernels:
//
// gdn_proj_conv_mfma_kernel (the fast path, proj_mfma.hpp) computes the
// transposed product in MFMA tiles chosen from its size.
//
// gdn_proj_conv_kernel (general shapes: group boundaries not on 4 columns,
// unaligned outputs, K not a multiple of 64) computes 128 x 128 tiles of P whose rows are
// tokens t0-3 .. t0+124 of one sequence and parks P in LDS for the conv.
//
// Output routing: up to 5 column groups, each written either token-major
// [B, T, width] or head-major [B, width/hd, T, hd], with or without the
// conv + SiLU (a plain projection takes the current token's row of P).
#include "gdn_common.hpp"
#include "proj.hpp"
#include "proj_mfma.hpp"

namespace {

using namespace gdn;

constexpr int kBM = 128, kBN = 128, kBK = 64;
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

// What a CU takes for each tile, in us: one workgroup (a1 + b1 per 64-wide K
// stage) and two of them (a2 + b2 per stage), side by side where two fit a CU
// and in turn where one does.  Least squares over 256 CUs x 1..4 tiles each at
// D = 1024, 2048 and 4096 (whole token tiles, D_out = 1024 or 2048), within 13%
// of each of the 12 times.
struct TileCost {
    int cols, outs;
    float a1, b1, a2, b2;
};
template <class TL>
constexpr TileCost cost_of(float a1, float b1, float a2, float b2) {
    return TileCost{TL::cols, TL::outs, a1, b1, a2, b2};
}
constexpr TileCost kTileCost[] = {  // in the order of launch_mfma_tile
    cost_of<Tile256x256>(23.3f, 1.22f, 37.0f, 2.5f),
    cost_of<Tile256x224>(21.3f, 1.13f, 31.2f, 2.38f),
    cost_of<Tile256x192>(18.0f, 1.02f, 29.7f, 2.05f),
    cost_of<Tile256x160>(16.8f, 0.898f, 26.6f, 1.81f),
    cost_of<Tile128x160>(10.9f, 0.6f, 17.5f, 1.18f),
    cost_of<Tile128x128Deep>(9.05f, 0.488f, 13.5f, 0.979f),
    cost_of<Tile128x128>(5.26f, 0.693f, 9.63f, 0.872f),
    cost_of<Tile64x128Deep>(7.26f, 0.294f, 12.3f, 0.578f),
    cost_of<Tile64x64Wide>(5.14f, 0.239f, 6.38f, 0.355f),
    cost_of<Tile64x64>(6.29f, 0.267f, 5.64f, 0.358f),
    cost_of<Tile64x32>(4.3f, 0.276f, 5.3f, 0.306f),
    cost_of<Tile32x32>(3.58f, 0.209f, 4.27f, 0.242f),
};

// The tile whose busiest CU finishes first: its tiles run in pairs, the odd
// one alone.  Every tile sums K and the taps in the same order, so the choice
// does not change a bit of the result.  At D = 2048 and 6176 columns, against
// 256 x 256 tiles with the waves in step for everything: 1 token 66 -> 10.3
// us, 77 tokens 61.9 -> 13.5, 253 tokens 61.4 -> 17.6, 509 tokens 61.9 ->
// 24.1, 1000 tokens 63.8 -> 35.4, 1500 tokens 64.2 -> 44.9, 3000 tokens 125 ->
// 84, 16384 tokens 464 -> 399.  The choice was the best of fourteen tiles on
// 60 of 61 sizes timed (1 to 16384 tokens, 2048 to 8224 columns, D = 1024 to
// 4096), and within 1% on the other.  The two smallest tiles came to hold two
// slices a stage later: 1 token 10.4 -> 8.6, 77 tokens 13.4 -> 12.9, 120 tokens
// 16.4 -> 13.5, and 77 tokens at 8224 columns 16.8 -> 13.4.  (32 x 32 tiles run
// up to three on a CU at less than the cost of a pair and one, which the
// estimate leaves out: 12% at the one size where it misses the best tile by most.)
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

int launch_mfma(const ProjParams& p, int F3, hipStream_t stream) {
    const int tile = choose_tile(F3, p.D, p.D_out);
    return p.packed > 0 ? launch_mfma_packed(tile, p, F3, stream) : launch_mfma_tile<kEqual>(tile, p, F3, stream);
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
