// The layer's output projection y = o W^T, up to one round of tiles and in the
// decode step above 16 sequences, on the MFMA projection kernel without the
// conv (proj_mfma.hpp).
//
// Reference: gdn_layer.py:263, 309 (o @ W_o.T, a library GEMM there).
//
// What bounds it: at these sizes every CU has one tile or none, so the time is
// a tile's chain of K stages, and that is the latency of a stage's copies and
// fragment reads over the waves that share it.  The tiles therefore sum K in
// two or four groups of waves, each on its own slice of a stage, which halves
// or quarters the chain and doubles the waves that hide it; the groups' fp32
// sums meet in LDS.  N = 2048, K = 2048 / 4096, us, one group -> these tiles
// (library call): 77 rows 9.0 / 15.6 -> 5.9 / 8.6 (7.6 / 10.4); 256 rows 10.5 /
// 18.4 -> 7.2 / 11.8 (10.5 / 14.4); 512 rows 11.9 / 20.8 -> 8.4 / 14.1 (12.2 /
// 19.4); 1024 rows 14.7 / 25.2 -> 12.7 / 22.3 (16.6 / 26.4).
#include "proj_mfma.hpp"

namespace gdn_proj {

namespace {

constexpr long long kCUs = 256;
long long tiles(const ProjParams& p, int cols, int toks) {
    return static_cast<long long>((p.T + toks - 1) / toks) * ((p.D_out + cols - 1) / cols);
}

ProjParams plain_params(const uint16_t* o, const uint16_t* W, uint16_t* y, int M, int K, int N) {
    ProjParams p = {};
    p.x = o;
    p.W = W;
    p.B = 1;
    p.T = p.T_out = M;
    p.D = K;
    p.D_out = N;
    p.ngroups = 1;
    p.groups[0] = ProjGroup{0, N, 0, 0, 0, y, nullptr, nullptr};
    return p;
}

}  // namespace

// The smallest tile whose grid is one round on 256 CUs (the next larger one
// was the slower at every size timed, 1 to 1024 rows), 64 x 128 from there on.
int launch_plain(const ProjParams& p, hipStream_t stream) {
    if (tiles(p, 32, 32) <= kCUs && p.D % (4 * kMK) == 0) return launch_tile<Plain32x32K4, kPlain>(p, p.T, stream);
    if (tiles(p, 64, 32) <= kCUs) return launch_tile<Plain64x32K2, kPlain>(p, p.T, stream);
    if (tiles(p, 64, 64) <= kCUs) return launch_tile<Plain64x64K2, kPlain>(p, p.T, stream);
    return launch_tile<Plain64x128K2, kPlain>(p, p.T, stream);
}

// The decode step's: a sequence's y must not depend on the batch it steps in,
// so the number of K groups follows K and N alone and the batch only picks
// among tiles of that number.  Four groups where tiles of four fit one round up
// to 256 sequences (N <= 2048), else two: K = 2048 / 4096, N = 2048, us, four
// against two groups: B = 48 6.0 / 8.5 against 6.3 / 9.8, B = 256 6.9 / 10.3
// against 7.1 / 11.2; N = 4096: B = 64 6.3 / 9.5 against 6.4 / 10.7, but B = 256
// 9.2 / 17.8 against 8.3 / 14.1, where tiles of four no longer fit.  (At N = 2048
// above 256 sequences two groups would be 1 to 3% of a step faster: 300 sequences
// 141.4 us a step against 143.8, 1024 418 against 425; the former 64 x 32 tiles
// 146.3 and 428.)
int launch_step_out_proj(const uint16_t* o, const uint16_t* W, uint16_t* y, int B, int K, int N, hipStream_t stream) {
    const ProjParams p = plain_params(o, W, y, B, K, N);
    if (K % (4 * kMK) == 0 && N <= 2048) {
        if (tiles(p, 32, 32) <= kCUs) return launch_tile<Plain32x32K4, kPlain>(p, B, stream);
        if (tiles(p, 64, 32) <= kCUs) return launch_tile<Plain64x32K4, kPlain>(p, B, stream);
        return launch_tile<Plain64x64K4, kPlain>(p, B, stream);
    }
    if (tiles(p, 32, 32) <= kCUs) return launch_tile<Plain32x32K2, kPlain>(p, B, stream);
    if (tiles(p, 64, 32) <= kCUs) return launch_tile<Plain64x32K2, kPlain>(p, B, stream);
    if (tiles(p, 64, 64) <= kCUs) return launch_tile<Plain64x64K2, kPlain>(p, B, stream);
    return launch_tile<Plain64x128K2, kPlain>(p, B, stream);
}

}  // namespace gdn_proj

// One round of the largest tile (64 x 128).  Beyond it the best of eleven tiles up
// to 256 x 256, found size by size, takes against a library call, N = 2048, us: K =
// 2048, 1100 rows 17.3 (20.2), 1500 18.6 (19.6), 2048 20.5 (21.3), 2683 27.3
// (29.8), 3000 28.0 (27.2), 4096 32.7 (33.5); K = 4096, 1300 rows 31.1 (27.8),
// 2683 48.1 (48.2), 3500 52.2 (57.0).  The tiles and a rule that finds the best are
// not built.
extern "C" int gdn_out_proj_fits(int64_t M, int64_t K, int64_t N) {
    constexpr int64_t kMost = 1 << 20;
    if (M <= 0 || M > kMost || K <= 0 || K > kMost || K % 128 != 0 || N <= 0 || N > kMost || N % 8 != 0) return 0;
    return (M + 127) / 128 * ((N + 63) / 64) <= 256 ? 1 : 0;
}

extern "C" int gdn_out_proj_hip(const gdn_bf16_t* o, const gdn_bf16_t* W, gdn_bf16_t* y, int M, int K, int N,
                                void* stream) {
    using gdn_host::aligned;
    using gdn_host::fail;
    if (M < 0 || K <= 0 || N <= 0) return fail(GDN_ERR_INVALID_ARGUMENT, "out_proj: M=%d K=%d N=%d", M, K, N);
    if (K % 128 != 0) return fail(GDN_ERR_UNSUPPORTED, "out_proj: K=%d must be a multiple of 128", K);
    if (N % 8 != 0) return fail(GDN_ERR_UNSUPPORTED, "out_proj: N=%d must be a multiple of 8", N);
    // 32-bit copy offsets within a tile
    if (K > (1 << 20)) return fail(GDN_ERR_UNSUPPORTED, "out_proj: K=%d too large", K);
    if (static_cast<long long>(M) * N >= (1ll << 40) || (static_cast<long long>(M) + 127) / 128 * ((N + 63) / 64) > 0x7fffffffLL)
        return fail(GDN_ERR_UNSUPPORTED, "out_proj: problem too large");
    if (M == 0) return GDN_OK;
    if (!o || !W || !y) return fail(GDN_ERR_INVALID_ARGUMENT, "out_proj: null pointer argument");
    if (!aligned(o, 16) || !aligned(W, 16) || !aligned(y, 16))
        return fail(GDN_ERR_INVALID_ARGUMENT, "out_proj: buffers need 16-byte alignment");
    const gdn_proj::ProjParams p = gdn_proj::plain_params(o, W, y, M, K, N);
    return gdn_proj::launch_plain(p, static_cast<hipStream_t>(stream));
}
