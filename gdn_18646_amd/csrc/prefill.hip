// GDN chunked prefill (chunk C = 64, dk = 128).
//
// Reference: kernels/prefill_chunked.cu:41-417 (one fused block per (b,h),
// WMMA for two products, the rest scalar) with the semantics of
// reference/prefill_ref.py:11-132.  Per chunk (Appendix-A notation):
//   gamma_t = exp(sum_{s<=t} log g_s)            Gamma_ts = gamma_t / gamma_s
//   A_ts    = beta_t m_t (k_t.k_s) Gamma_ts, t>s T = (I + A)^-1
//   dV      = T diag(beta m) (V - diag(gamma) K S)
//   O       = m (scale gamma (Q S) + scale (Q K^T o Gamma)_causal dV)
//   S      <- gamma_C S + (K o gamma_C/gamma)^T dV
//
// Kernel 1, gdn_prefill_intra_kernel — one wave per (chunk, head, sequence);
// every chunk in parallel.  Builds K K^T (and Q K^T) on bf16 MFMA, the decay
// matrix, the fp32 forward substitution for T, and writes per chunk (bf16
// unless noted), already in the register order the state kernels' MFMA
// operands need (one 16-byte load per lane per fragment):
//   Tp  = T diag(beta m)                       the 6 nonzero fragments (6 KiB)
//   Aq  = m scale (Q K^T o Gamma), t >= s      the 6 nonzero fragments (6 KiB)
//   G   = [gamma_t, m_t scale gamma_t, gamma_C / gamma_t, -]   256 fp32
// The state update's K^T operand is not stored: the state kernels build it
// from the K tile they stage anyway, with transposing LDS reads, and apply
// gamma_C / gamma_t to the rows of dV instead.
// Kernel 2, gdn_prefill_state_kernel — each wave owns 16*NT state columns of
// one (sequence, head) and walks chunks in order.  The fp32 state tile lives
// in MFMA accumulator registers the whole time; its bf16 copy feeds the next
// chunk's products directly (no LDS), because the k order inside an MFMA
// operand is free: the state rows are assigned to accumulator slots so that
// the accumulator of the state update IS the B operand of K S and Q S.
// When (sequence, head) pairs alone cannot fill the chip, each sequence is cut
// into G chunk groups (S maps affinely across a group: S_out = phi S_in + psi):
//   map pass   (kernel 2, map mode)  psi and phi of every group but the last,
//   scan       (gdn_prefill_scan_kernel)  S_in of every group, in order,
//   output pass (kernel 2, output mode) every group from its S_in, in parallel.
//
// Fragment k-order conventions (lane l: m = l%16 row/column, g = l/16 group):
//   pi(g, j)   = j < 4 ? 4g + j : 16 + 4g + (j-4)   chunk position inside a
//                32-wide k-step, the order produced by two stacked accumulators
//   rho(r,g,i) = 32(r/2) + 8g + 4(r%2) + i          state row held in
//                accumulator tile r, slot i, of lane group g
#include <algorithm>
#include <cmath>
#include <mutex>

#include "gdn_common.hpp"

namespace {

using namespace gdn;

constexpr int kC = 64;    // chunk length
constexpr int kDK = 128;  // key / query dim

// Workspace record of one (chunk, head), written by the intra kernel and read
// by the state kernels, in 1 KiB MFMA fragments (lane l's 16 bytes at 16 l).
// For the 16-column state kernel: the six nonzero fragments of Tp, the six of
// Aq, the gate block.  The 32-column state kernel forms Aq itself and reads
// the six of Tp, the gate block and the token block (log2 of the in-chunk
// decay, m scale).  Gate block: gamma, m scale gamma, gamma_C / gamma.
constexpr int kRecTp = 0;
constexpr int kRecAq = 6;
constexpr int kRecFull = 13;   // Tp, Aq, gates
constexpr int kRecShort = 8;   // Tp, gates, tokens
constexpr int kRecGShort = 6;  // gate block of the short record
constexpr int kRecH = 7;       // token block of the short record

struct PrefillParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    const uint16_t* a;
    const uint16_t* b;
    const float* A_log;
    const float* mask;      // nullable: all ones
    const float* state_in;  // nullable: zero state
    uint16_t* out;
    float* state_out;
    const int32_t* cu;  // varlen offsets (nullable: batch mode)
    u32x4* wsR;          // per (chunk, head) workspace records (rec_frags 1 KiB fragments each)
    float dt_bias;
    float scale;
    int H;
    int dv;
    int T_stride;        // tokens per (b, h) row block of q/k/v/a/b/out
    int T_len;           // batch mode: sequence length
    int chunks_per_seq;  // batch mode: ceil(T_len / 64)
    int xcd_heads;       // (sequence, head) pairs are a multiple of 8: head-aligned XCD mapping
    int out_tm;          // out is token-major ([B, T, H, dv] / [T_total, H, dv]) instead of head-major
    int nseq;
    int intra_items;     // intra kernel: chunks per (sequence, head); packed sequences: chunks or chunk slots per head
    int intra_chunks;    // packed sequences: chunks per sequence of the intra kernel's grid, 0 = chunk slots
};

struct SeqInfo {
    int b, tok0, len, slot0;
};

__device__ __forceinline__ SeqInfo seq_info(const PrefillParams& p, int sidx) {
    SeqInfo s;
    if (p.cu) {
        s.b = 0;
        s.tok0 = p.cu[sidx];
        s.len = p.cu[sidx + 1] - s.tok0;
        // Chunk slots floor(tok0/64) + sidx never overlap between sequences
        // and total at most T_total/64 + num_seqs.
        s.slot0 = s.tok0 / kC + sidx;
    } else {
        s.b = sidx;
        s.tok0 = 0;
        s.len = p.T_len;
        s.slot0 = sidx * p.chunks_per_seq;
    }
    return s;
}

__device__ __forceinline__ int pi_pos(int g, int j) { return j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4); }
__device__ __forceinline__ int rho_row(int r, int g, int i) { return 32 * (r >> 1) + 8 * g + 4 * (r & 1) + i; }

// Workgroups are dealt to the 8 XCDs round robin by linear id, and each XCD
// has its own L2.  With a multiple of 8 (sequence, head) pairs every prefill
// kernel puts head `hd` on XCD hd % 8, so what one kernel writes for a head
// is read from the same L2 by the next: linear id L -> head (L % 8) + 8 q,
// item r of that head, where L / 8 = q * per_head + r.
struct HeadItem {
    int head, item;
};
__device__ __forceinline__ HeadItem head_major_xcd(int L, int per_head) {
    const int q = (L >> 3) / per_head;
    return {(L & 7) + 8 * q, (L >> 3) - q * per_head};
}

// Slot of the nonzero fragment (mt, s) of the causal Aq (and of Tp), whose order
// is (0,0), (1,0), (2,0), (2,1), (3,0), (3,1) (s = 1 needs mt >= 2).
__device__ __forceinline__ constexpr int aq_index(int mt, int s) { return mt < 2 ? mt : 2 * mt - 2 + s; }

// ---------------------------------------------------------------------------
// Kernel 1
// ---------------------------------------------------------------------------
// Inclusive prefix sum over the 64 lanes with DPP: shifts by 1, 2, 4, 8 within
// each 16-lane row, then lane 15 broadcast into rows 1 and 3 and lane 31 into
// rows 2 and 3.  Lanes without a source add 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add_src(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, true));
}
__device__ __forceinline__ float wave_inclusive_sum(float v) {
    v += dpp_add_src<0x111, 0xf>(v);  // row_shr:1
    v += dpp_add_src<0x112, 0xf>(v);  // row_shr:2
    v += dpp_add_src<0x114, 0xf>(v);  // row_shr:4
    v += dpp_add_src<0x118, 0xf>(v);  // row_shr:8
    v += dpp_add_src<0x142, 0xa>(v);  // row_bcast:15 into rows 1, 3
    v += dpp_add_src<0x143, 0xc>(v);  // row_bcast:31 into rows 2, 3
    return v;
}

// One (chunk, sequence-head) unit of kernel 1.  Batches: unit u maps to head,
// chunk through head_major_xcd when the head count allows.  Packed sequences:
// to head, sequence and chunk, or to head, chunk slot (every slot belongs to at
// most one sequence), whichever makes the smaller grid.
struct IntraUnit {
    SeqInfo sq;
    size_t row_base, wc;
    int h, t0, nvalid;
};
__device__ __forceinline__ bool intra_unit(const PrefillParams& p, int u, int lane, IntraUnit& U) {
    int head, item;
    if (p.xcd_heads) {
        const HeadItem hi = head_major_xcd(u, p.intra_items);
        head = hi.head;
        item = hi.item;
    } else {
        head = u / p.intra_items;
        item = u - head * p.intra_items;
    }
    if (p.intra_chunks) {
        const int seq = item / p.intra_chunks;
        U.h = head;
        U.sq = seq_info(p, seq);
        U.t0 = (item - seq * p.intra_chunks) * kC;
    } else if (p.cu) {
        // The slot's sequence: the last one whose first slot is not past it
        // (first slots grow with the sequence).  How many those are lies in
        // [before, hi]; a step probes 64 of them, 64 sequences take one, 4096
        // two.  (64 at a time in turn, 128 loads one after the other for 8192
        // sequences of 1 or 2 tokens: H = 4, dv = 128 944 us a call, 835 now; 1024
        // of them at H = 1 37.0, now 34.8.)
        int before = 0, hi = p.nseq;
        while (before < hi) {
            const int step = (hi - before + kWave - 1) / kWave;
            const int i = before + step * (lane + 1) - 1;
            const bool le = i < hi && p.cu[i] / kC + i <= item;
            before += step * __builtin_popcountll(__builtin_amdgcn_ballot_w64(le));
            hi = min(hi, before + step - 1);
        }
        if (before == 0) return false;
        U.h = head;
        U.sq = seq_info(p, __builtin_amdgcn_readfirstlane(before - 1));
        U.t0 = (item - U.sq.slot0) * kC;
    } else {
        U.h = head % p.H;
        U.sq = seq_info(p, head / p.H);
        U.t0 = item * kC;
    }
    if (U.t0 >= U.sq.len) return false;  // packed: past its sequence's end
    U.nvalid = min(kC, U.sq.len - U.t0);
    U.row_base = static_cast<size_t>(U.sq.b * p.H + U.h) * p.T_stride + U.sq.tok0 + U.t0;
    U.wc = static_cast<size_t>(U.sq.slot0 + U.t0 / kC) * p.H + U.h;
    return true;
}

// A unit's gates, one token per lane: log2 of the in-chunk decay cumsum,
// beta m, m scale, and the gate block gamma, m scale gamma, gamma_C / gamma.
// Tokens past the sequence end: no decay, beta m = m = 0.
struct GateVals {
    float lg2, bm, ms, g0, g1, g2;
};
__device__ __forceinline__ GateVals gate_vals(const PrefillParams& p, float alog, float mask, uint32_t a, uint32_t b,
                                              bool valid) {
    float lg = 0.f, bm = 0.f, m = 0.f;
    if (valid) {
        m = mask;
        lg = -expf(alog) * softplus_f(__uint_as_float(a << 16) + p.dt_bias);
        bm = sigmoid_f(__uint_as_float(b << 16)) * m;
    }
    const float s = wave_inclusive_sum(lg);
    const float last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), kWave - 1));
    const float gam = expf(s);
    return {s * 1.4426950408889634f, bm, m * p.scale, gam, m * p.scale * gam, expf(last - s)};
}

// t[i] += a[i] of lane J of each 16-lane row, times tj, for N <= 4 registers.
// One v_fmac_f32 each with its DPP operand (the compiler emits a DPP move, a
// wait and an FMA instead: 0.1 to 0.8 us more a call); the s_nop covers the two wait states between a
// VALU write of a[i] and its DPP read, which the compiler cannot see in here.
#define GDN_FMAC_BCAST(I) "v_fmac_f32_dpp %" #I ", %[a" #I "], %[x] row_newbcast:%[j] row_mask:0xf bank_mask:0xf\n\t"
template <int J, int N>
__device__ __forceinline__ void fmac_row_bcast(float* t, const float* a, float tj) {
    if constexpr (N == 4)
        asm("s_nop 1\n\t" GDN_FMAC_BCAST(0) GDN_FMAC_BCAST(1) GDN_FMAC_BCAST(2) GDN_FMAC_BCAST(3)
            : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3])
            : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [x] "v"(tj), [j] "n"(J));
    else if constexpr (N == 3)
        asm("s_nop 1\n\t" GDN_FMAC_BCAST(0) GDN_FMAC_BCAST(1) GDN_FMAC_BCAST(2)
            : "+v"(t[0]), "+v"(t[1]), "+v"(t[2])
            : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [x] "v"(tj), [j] "n"(J));
    else if constexpr (N == 2)
        asm("s_nop 1\n\t" GDN_FMAC_BCAST(0) GDN_FMAC_BCAST(1)
            : "+v"(t[0]), "+v"(t[1])
            : [a0] "v"(a[0]), [a1] "v"(a[1]), [x] "v"(tj), [j] "n"(J));
    else
        asm("s_nop 1\n\t" GDN_FMAC_BCAST(0)
            : "+v"(t[0])
            : [a0] "v"(a[0]), [x] "v"(tj), [j] "n"(J));
}
#undef GDN_FMAC_BCAST

// acc + A B on 16 x 16 fp32 blocks.  A's lane l holds A[l % 16][4 (l / 16) + i],
// i.e. the accumulator layout of its transpose; B is in accumulator layout.
// MFMA i carries k = 4 (l / 16) + i in both.
__device__ __forceinline__ f32x4 mul16(const f32x4 a, const f32x4 b, f32x4 acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc, 0, 0, 0);
    return acc;
}

// One wave per (chunk, head), no barrier between waves.  The chunk's K is held
// as MFMA fragments (64 VGPRs, the A and the B operand of K K^T alike); A's
// ten lower 16 x 16 blocks, negated, stay in registers, and T = (I + A)^-1 is
// formed as U = T^T, whose accumulators are the record's Tp fragments as they
// stand:
//   diagonal blocks: forward substitution in fp32, the four blocks at once,
//     block g in lanes 16 g .. 16 g + 15, a column a lane and A's entries
//     broadcast along the row by DPP: 120 FMAs, no LDS read between them;
//   the others: U_JI = U_JJ sum_{J < K <= I} (-A_KJ)^T U_KI on fp32 MFMA
//     16x16x4.  An A operand is the accumulator of its transpose, so -A_KJ
//     (computed with rows in K) and T_JJ go in unchanged, and a product's
//     accumulator is the next one's B operand.
// LDS holds only this wave's gates and the two re-layouts of the diagonal
// blocks (5.5 KiB).
//
// Large calls are bound by HBM (16 KiB read and 8 KiB written a unit, 4.5-5
// TB/s), small ones by the one chain of loads, gates, products and
// substitution.  With 256-thread workgroups, five barriers a unit and four
// units in flight a CU (16 here) the same work took: B=8, T=2000 (H = 16)
// 33.9 us, 21.7 now; 24,674 packed tokens 50.9, now 29.1; B=1, T=8192 18.4, now
// 12.9; T=333 7.6, now 5.2.
// AQ: also form the causal Aq (for the 16-column state kernel; the 32-column
// one forms it itself).
template <bool AQ>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 4))) void gdn_prefill_intra_kernel(
    PrefillParams p) {
    constexpr int RF = AQ ? kRecFull : kRecShort;       // record length (fragments)
    constexpr int RG = AQ ? kRecFull - 1 : kRecGShort;  // gate block
    // Diagonal block g, element (row r, column c) at dg[g][c][r]: rows of 20
    // floats put 16 lanes' 16-byte accesses in 16 bank groups.
    constexpr int kDS = 20;
    __shared__ __attribute__((aligned(16))) float dg[4][16][kDS];
    __shared__ __attribute__((aligned(16))) float s_lg2[kC], s_bm[kC], s_ms[AQ ? kC : 4];
    const int lane = threadIdx.x;
    const int m16 = lane & 15;
    const int g4 = lane >> 4;

    IntraUnit U;
    if (!intra_unit(p, blockIdx.x, lane, U)) return;
    u32x4* const rec = p.wsR + U.wc * RF * 64;

    // 1) The gate inputs, then K (rows past the sequence end read as zeros).
    const bool valid = lane < U.nvalid;
    const float alog = p.A_log[U.h];
    float gm = 0.f;
    uint32_t ga = 0u, gb = 0u;
    if (valid) {
        gm = p.mask ? p.mask[static_cast<size_t>(U.sq.b) * p.T_stride + U.sq.tok0 + U.t0 + lane] : 1.f;
        ga = p.a[U.row_base + lane];
        gb = p.b[U.row_base + lane];
    }
    const __amdgpu_buffer_rsrc_t kr = buffer_rsrc(p.k + U.row_base * kDK, U.nvalid * kDK * 2);
    // The whole offset goes in the lane's: the resource's range check, which
    // zeroes those rows, leaves the scalar offset out.
    auto row_off = [&](int t) { return static_cast<uint32_t>((16 * t + m16) * kDK * 2 + 16 * g4); };
    bf16x8 kf[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s) kf[t][s] = as_bf16x8(buffer_load16(kr, row_off(t) + 64 * s, 0));

    // 2) Gates and the in-chunk log-cumsum, one token per lane.
    {
        const GateVals gv = gate_vals(p, alog, gm, ga, gb, valid);
        s_lg2[lane] = gv.lg2;
        s_bm[lane] = gv.bm;
        if constexpr (AQ) s_ms[lane] = gv.ms;
        float* G = reinterpret_cast<float*>(rec + RG * 64);
        G[lane] = gv.g0;
        G[64 + lane] = gv.g1;
        G[128 + lane] = gv.g2;
        if constexpr (!AQ) {
            float* Hb = reinterpret_cast<float*>(rec + kRecH * 64);
            Hb[lane] = gv.lg2;
            Hb[64 + lane] = gv.ms;
        }
    }
    __syncthreads();
    auto quad = [&](const float* x, int t) { return *reinterpret_cast<const f32x4*>(x + 16 * t + 4 * g4); };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

    // 3) Aq fragments (mt, s): lane holds Aq[16 mt + m][32 s + pi(g, j)], i.e.
    //    the accumulators of the transposed tiles K_J Q_mt^T, J = 2 s, 2 s + 1.
    if constexpr (AQ) {
        const __amdgpu_buffer_rsrc_t qr = buffer_rsrc(p.q + U.row_base * kDK, U.nvalid * kDK * 2);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            bf16x8 qf[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) qf[s] = as_bf16x8(buffer_load16(qr, row_off(t) + 64 * s, 0));
            const float lc = s_lg2[16 * t + m16], mc = s_ms[16 * t + m16];
            f32x4 x[4];
#pragma unroll
            for (int J = 0; J < 4; ++J) {
                x[J] = zero;
                if (J > t) continue;
#pragma unroll
                for (int s = 0; s < 4; ++s) x[J] = mfma16x16x32(kf[J][s], qf[s], x[J]);
                const f32x4 lr = quad(s_lg2, J);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float y = mc * x[J][i] * __builtin_amdgcn_exp2f(lc - lr[i]);
                    x[J][i] = J < t || m16 >= 4 * g4 + i ? y : 0.f;
                }
            }
#pragma unroll
            for (int s = 0; s <= t / 2; ++s)
                rec[(kRecAq + aq_index(t, s)) * 64 + lane] = as_u32x4(pack8(x[2 * s], x[2 * s + 1]));
        }
    }

    // 4) -A: block (K, J) has rows t = 16 K + 4 g4 + i and column s = 16 J + m16.
    auto neg_a = [&](int K, int J) {
        f32x4 x = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) x = mfma16x16x32(kf[K][s], kf[J][s], x);
        const f32x4 lr = quad(s_lg2, K), br = quad(s_bm, K);
        const float lc = s_lg2[16 * J + m16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float y = -br[i] * x[i] * __builtin_amdgcn_exp2f(lr[i] - lc);
            x[i] = K > J || 4 * g4 + i > m16 ? y : 0.f;
        }
        return x;
    };
#pragma unroll
    for (int t = 0; t < 4; ++t) *reinterpret_cast<f32x4*>(&dg[t][m16][4 * g4]) = neg_a(t, t);
    const f32x4 a10 = neg_a(1, 0), a20 = neg_a(2, 0), a30 = neg_a(3, 0), a21 = neg_a(2, 1), a31 = neg_a(3, 1),
                a32 = neg_a(3, 2);
    __syncthreads();

    // 5) Diagonal blocks: lane (c, g) solves column c of block g.
    float a[16], T[16];
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(&dg[g4][m16][r]);
#pragma unroll
        for (int i = 0; i < 4; ++i) a[r + i] = x[i];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) T[r] = r == m16 ? 1.f : 0.f;
    static_for<0, 15>([&](auto j) {
        static_for<(j + 1) / 4, 4>([&](auto q) {  // rows j + 1 .. 15, in quads from the first row's
            constexpr int r0 = 4 * q > j ? 4 * q : j + 1;
            fmac_row_bcast<j, 4 * q + 4 - r0>(&T[r0], &a[r0], T[j]);
        });
    });
#pragma unroll
    for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<f32x4*>(&dg[g4][m16][r]) = f32x4{T[r], T[r + 1], T[r + 2], T[r + 3]};
    __syncthreads();
    f32x4 td[4], ud[4];  // T_JJ (the A operand of U_JJ) and U_JJ, in accumulator layout
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        td[t] = *reinterpret_cast<const f32x4*>(&dg[t][m16][4 * g4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) ud[t][i] = dg[t][4 * g4 + i][m16];
    }

    // 6) The other blocks of U, and the Tp fragments (mt, s) = U's blocks
    //    (2 s, mt) and (2 s + 1, mt), their rows times beta m.
    const f32x4 u01 = mul16(td[0], mul16(a10, ud[1], zero), zero);
    const f32x4 u12 = mul16(td[1], mul16(a21, ud[2], zero), zero);
    const f32x4 u23 = mul16(td[2], mul16(a32, ud[3], zero), zero);
    const f32x4 u02 = mul16(td[0], mul16(a10, u12, mul16(a20, ud[2], zero)), zero);
    const f32x4 u13 = mul16(td[1], mul16(a21, u23, mul16(a31, ud[3], zero)), zero);
    const f32x4 u03 = mul16(td[0], mul16(a10, u13, mul16(a20, u23, mul16(a30, ud[3], zero))), zero);
    auto put_tp = [&](int mt, int s, const f32x4 lo, const f32x4 hi) {
        rec[(kRecTp + aq_index(mt, s)) * 64 + lane] =
            as_u32x4(pack8(lo * quad(s_bm, 2 * s), hi * quad(s_bm, 2 * s + 1)));
    };
    put_tp(0, 0, ud[0], zero);
    put_tp(1, 0, u01, ud[1]);
    put_tp(2, 1, ud[2], zero);
    put_tp(3, 1, u23, ud[3]);
    put_tp(2, 0, u02, u12);
    put_tp(3, 0, u03, u13);
}

// ---------------------------------------------------------------------------
// Kernel 2
// ---------------------------------------------------------------------------
// Per-chunk operands staged in LDS (one buffer; the kernels double-buffer).
// Every block is a run of 1 KiB "fragments": 64 lanes x 16 bytes, lane l's
// 16 bytes at offset 16 l, i.e. exactly one MFMA operand register quad.
constexpr int kFragB = 1024;
enum { kModeOut = 0, kModeMap = 1 };

// Staging layout of one buffer.  The map pass (no outputs) stages neither Q
// nor Aq.  V is per wave: [64 rows][16 NT columns] bf16.
template <int MODE, int NW, int NT>
struct Stage {
    static constexpr bool out = MODE == kModeOut;
    static constexpr int offK = 0;                                  // 16: (mt, s), lane slots swizzled (kslot)
    static constexpr int offQ = offK + 16 * kFragB;                 // 16 (out only)
    static constexpr int offT = offQ + (out ? 16 : 0) * kFragB;     // 6: nonzero Tp fragments
    static constexpr int offA = offT + 6 * kFragB;                  // 6 (out only): Aq slots used
    static constexpr int offG = offA + (out ? 6 : 0) * kFragB;      // gamma, m scale gamma, gamma_C/gamma
    static constexpr int offV = offG + kFragB;
    static constexpr int vWave = 2 * NT * kFragB;
    static constexpr int bytes = offV + NW * vWave;
    static constexpr int stores = out ? 4 * NT : 0;                 // output stores per chunk per wave
};



// Per-lane byte offsets of the staging copies, fixed for the whole kernel.
struct StageLane {
    uint32_t k;   // K fragment slot `lane`: row kslot_row(lane), k offset 8 (lane >> 4)
    uint32_t q;   // Q fragment: row (lane & 15), k offset 8 (lane >> 4)
    uint32_t fr;  // workspace fragment or gate block: 16 lane
    uint32_t v;   // V tile: row lane / (2 NT), 8 columns (lane % (2 NT))
};

// K fragments are staged with their 16-byte lane slots swizzled: the data of
// fragment lane (m, g) (row m, k group g) sits in slot 16 g + (m ^ 4 g).
// Plain fragment reads stay conflict free, and the transposing reads that
// build K^T (16 lanes reading rows T0..T0+3 of four k groups) hit 16
// different slots modulo 16 instead of 4.
__device__ __forceinline__ int kslot(int m, int g) { return 16 * g + (m ^ (4 * g)); }
__device__ __forceinline__ int kslot_row(int slot) { return (slot & 15) ^ (4 * (slot >> 4)); }

// Copies of one chunk's operands into `buf`, all issued together at the start
// of the previous chunk's work (spreading them between its MFMA phases was
// measured slower: a copy that meets a full memory pipeline stalls the MFMA
// work queued behind it).  Shared jobs (K, Q, Tp, Aq and Kt fragments, the
// gate block) are dealt round robin to the NW waves; each wave copies its own
// V tile when `v_on`.  Full chunks use uniform bases plus the lane offsets;
// the last, partial chunk clamps rows to the sequence (so no load leaves the
// tensors) and its padded rows are zeroed after arrival.

template <int MODE, int NW, int NT>
struct Stager {
    using St = Stage<MODE, NW, NT>;
    static constexpr int nK = 16, nQ = St::out ? 16 : 0, nT = 6, nA = St::out ? 6 : 0;
    static constexpr int NJ = nK + nQ + nT + nA + 1;  // + the gate block
    const PrefillParams* p;
    lds_u8* buf;
    size_t row_base, wc;
    int nvalid, wave, lane, col0_wave;
    bool on, v_on;
    const StageLane* L;

    __device__ __forceinline__ void issue() const {
        if (!on) return;
        const bool full = nvalid == kC;
        const int m = lane & 15, g = lane >> 4;
        const unsigned char* kb = reinterpret_cast<const unsigned char*>(p->k + row_base * kDK);
        const unsigned char* qb = reinterpret_cast<const unsigned char*>(p->q + row_base * kDK);
        // The shared jobs are staged contiguously in job order (K, Q, Tp, Aq,
        // gate block), so job f lands at f KiB.  Each wave walks only its own
        // jobs f = wave, wave + NW, ... (a uniform loop).
        static_assert(St::offK == 0 && St::offQ == nK * kFragB && St::offT == (nK + nQ) * kFragB &&
                          St::offG == (nK + nQ + nT + nA) * kFragB && (!St::out || St::offA == St::offT + nT * kFragB),
                      "staging layout must follow job order");
        for (int f = wave; f < NJ; f += NW) {
            lds_u8* const dst = buf + f * kFragB;
            if (f < nK + nQ) {
                const bool isq = f >= nK;
                const int ff = isq ? f - nK : f;
                const unsigned char* base = isq ? qb : kb;
                if (full) {
                    dma16(base + (ff >> 2) * 16 * kDK * 2 + (ff & 3) * 64, isq ? L->q : L->k, dst);
                } else {
                    const int row = min(16 * (ff >> 2) + (isq ? m : kslot_row(lane)), nvalid - 1);
                    dma16(base, static_cast<uint32_t>((row * kDK + 32 * (ff & 3) + 8 * g) * 2), dst);
                }
            } else {
                // record fragments: Tp, then Aq (output only), then the gate block
                const unsigned char* rec = reinterpret_cast<const unsigned char*>(p->wsR + wc * kRecFull * 64);
                const int j = f - nK - nQ;
                dma16(rec + (j < nT + nA ? j : kRecFull - 1) * kFragB, L->fr, dst);
            }
        }
        if (v_on) {
            constexpr int kRowsPerV = 32 / NT;  // V rows per 1 KiB copy
#pragma unroll
            for (int it = 0; it < 2 * NT; ++it) {
                if (full) {
                    dma16(p->v + (row_base + kRowsPerV * it) * p->dv, L->v,
                          buf + St::offV + wave * St::vWave + it * kFragB);
                } else {
                    const int row = min(kRowsPerV * it + lane / (2 * NT), nvalid - 1);
                    dma16(p->v + row_base * p->dv,
                          static_cast<uint32_t>((row * p->dv + col0_wave + 8 * (lane % (2 * NT))) * 2),
                          buf + St::offV + wave * St::vWave + it * kFragB);
                }
            }
        }
    }
};

// Zero the rows >= nvalid of the staged K, Q and V (partial chunk only).
template <int MODE, int NW, int NT>
__device__ __forceinline__ void zero_pad_rows(lds_u8* buf, int nvalid, int wave, int lane) {
    using St = Stage<MODE, NW, NT>;
    const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int f = 0; f < (St::out ? 32 : 16); ++f)  // K then Q (contiguous); K slots are swizzled
        if (f % NW == wave && 16 * ((f & 15) >> 2) + (f < 16 ? kslot_row(lane) : (lane & 15)) >= nvalid)
            *reinterpret_cast<lds_u32x4*>(buf + St::offK + f * kFragB + 16 * lane) = z;
#pragma unroll
    for (int it = 0; it < 2 * NT; ++it)
        if ((32 / NT) * it + lane / (2 * NT) >= nvalid)
            *reinterpret_cast<lds_u32x4*>(buf + St::offV + wave * St::vWave + it * kFragB + 16 * lane) = z;
}

__device__ __forceinline__ bf16x8 frag(const lds_u8* buf, int off, int lane) {
    return *reinterpret_cast<const lds_bf16x8*>(buf + off + 16 * lane);
}

// K fragment f = 4 mt + s (rows 16 mt + m, k 32 s + 8 g) from the swizzled slots.
__device__ __forceinline__ bf16x8 kfrag(const lds_u8* kbuf, int f, int lane) {
    return *reinterpret_cast<const lds_bf16x8*>(kbuf + f * kFragB + 16 * kslot(lane & 15, lane >> 4));
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// K^T fragment (r, s), the A operand of the state update: lane (m, g) gets
// K[32 s + pi(g, j)][rho(r, m / 4, m % 4)] for j = 0..7, from the staged K.
// ds_read_b64_tr_b16 hands output lane i of each 16-lane group element i % 4
// of the 8 bytes read by lanes 4 j + i / 4 (j = 0..3); so source lane 4 j + a
// reads row T0 + j at columns base(a) .. base(a) + 3, base(a) = rho(r, a, 0),
// and output lane m = 4 a + p receives column rho(r, a, p) of rows T0 .. T0 + 3.
// Two such reads (T0 = 32 s + 4 g and 32 s + 16 + 4 g) give the pi order.
// Only the K slot depends on the lane (row 4 g + j of the 16-row block,
// k group a): `kt_lane` = 16 kslot(4 g + j, a), computed once; the rest of
// the address is a compile-time offset.
__device__ __forceinline__ uint32_t kt_lane_offset(int lane) {
    return 16u * static_cast<uint32_t>(kslot(4 * (lane >> 4) + ((lane >> 2) & 3), lane & 3));
}
__device__ __forceinline__ bf16x8 ktfrag(const lds_u8* kbuf, uint32_t kt_lane, int r, int s) {
    const lds_u8* base = kbuf + kt_lane + (r >> 1) * kFragB + 8 * (r & 1);
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(base + (2 * s) * 4 * kFragB));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(base + (2 * s + 1) * 4 * kFragB));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return as_bf16x8(u32x4{l2[0], l2[1], h2[0], h2[1]});
}

// bf16 of (x - bf16(x)) for a pair of accumulator quads: the low half of a
// two-term bf16 split.
__device__ __forceinline__ bf16x8 pack8_lo(const f32x4 lo, const f32x4 hi, const bf16x8 h) {
    f32x4 dl, dh;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        dl[i] = lo[i] - bf2f(h[i]);
        dh[i] = hi[i] - bf2f(h[4 + i]);
    }
    return pack8(dl, dh);
}


// One chunk of the state recurrence for a 128 x (16 NT) column tile, operands
// in LDS.  `ob` points at out[row_base][0] (uniform).  Operand fragments are
// read from LDS one phase ahead of their use (none depends on the state), so
// the MFMA chain that does depend on it rarely waits on LDS, without holding
// every fragment in registers at once.  `v_zero`: the tile has no V (identity
// columns of the map pass).  `next` issues the following chunk's copies.
template <int MODE, int NW, int NT>
__device__ __forceinline__ void state_chunk(const lds_u8* buf, f32x4 (&S)[8][NT], uint16_t* ob, int orow, int nvalid,
                                            int wave, int lane, int col0_wave, bool v_zero, uint32_t kt_lane,
                                            const Stager<MODE, NW, NT>& next) {
    using St = Stage<MODE, NW, NT>;
    const int n = lane & 15, g = lane >> 4;
    const lds_f32* G = reinterpret_cast<const lds_f32*>(buf + St::offG);
    const lds_u16* Vs = reinterpret_cast<const lds_u16*>(buf + St::offV + wave * St::vWave);

    next.issue();

    // (a) X = K S (and P = Q S for the output), in two k-halves so only half
    //     of the K and Q fragments is held at a time.
    f32x4 X[4][NT], P[4][NT];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) X[mt][nt] = P[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        bf16x8 kf[4][2], qf[St::out ? 4 : 1][2];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                const int f = 4 * mt + 2 * half + s2;
                kf[mt][s2] = kfrag(buf + St::offK, f, lane);
                if constexpr (St::out) qf[mt][s2] = frag(buf, St::offQ + f * kFragB, lane);
            }
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            const int s = 2 * half + s2;
            bf16x8 Bs[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) Bs[nt] = pack8(S[2 * s][nt], S[2 * s + 1][nt]);
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    X[mt][nt] = mfma16x16x32(kf[mt][s2], Bs[nt], X[mt][nt]);
                    if constexpr (St::out) P[mt][nt] = mfma16x16x32(Bs[nt], qf[mt][s2], P[mt][nt]);
                }
        }
    }
    bf16x8 tf[6], af[St::out ? 6 : 1], ktf[8][2];
    // With one wave per SIMD (NW <= 4) the Kt fragments are read here, while
    // (a) drains; with two (NW = 8) the other wave covers their latency, so
    // they are read just before (e) to keep this wave within 256 registers.
    constexpr bool kEarlyKt = NW <= 4;
    auto load_kt = [&]() {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            ktf[r][0] = ktfrag(buf + St::offK, kt_lane, r, 0);
            ktf[r][1] = ktfrag(buf + St::offK, kt_lane, r, 1);
        }
    };
#pragma unroll
    for (int f = 0; f < 6; ++f) tf[f] = frag(buf, St::offT + f * kFragB, lane);
    if constexpr (kEarlyKt) load_kt();
    // V in the accumulator layout (column n, rows 16 mt + 4 g + i): one
    // transposing read per (mt, nt) -- source lane 4 j + a of group g reads
    // row 16 mt + 4 g + j at columns 16 nt + 4 a .. + 3.  Kept as bf16 until use.
    i16x4 vv[NT][4];
    const lds_u8* vrow = reinterpret_cast<const lds_u8*>(Vs) + ((4 * g + ((lane >> 2) & 3)) * 16 * NT + 4 * (lane & 3)) * 2;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
            vv[nt][mt] = v_zero ? i16x4{0, 0, 0, 0}
                                : __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                      (lds_i16x4*)(vrow + (16 * mt * 16 * NT + 16 * nt) * 2));
    f32x4 gam[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) gam[mt] = *reinterpret_cast<const lds_f32x4*>(G + 16 * mt + 4 * g);
    const float gC = G[kC - 1];
    // (b) Y = V - gamma o X (in place in X).
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                X[mt][nt][i] = bf2f(static_cast<uint16_t>(vv[nt][mt][i])) - gam[mt][i] * X[mt][nt][i];
    // (c) dV = Tp Y.
    f32x4 D[4][NT];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) D[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Tp is lower triangular: fragments (0, 1) and (1, 1) are zero and absent.
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        bf16x8 BY[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) BY[nt] = pack8(X[2 * s][nt], X[2 * s + 1][nt]);
#pragma unroll
        for (int mt = 2 * s; mt < 4; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) D[mt][nt] = mfma16x16x32(tf[aq_index(mt, s)], BY[nt], D[mt][nt]);
    }
    if constexpr (St::out) {
#pragma unroll
        for (int i = 0; i < 6; ++i) af[i] = frag(buf, St::offA + i * kFragB, lane);
    }
    // The state update takes dV with its rows scaled by gamma_C / gamma_t
    // (the decay from token t to the chunk end); the output takes dV as is.
    f32x4 kd[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) kd[mt] = *reinterpret_cast<const lds_f32x4*>(G + 128 + 16 * mt + 4 * g);
    bf16x8 BS0[NT], BS1[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        BS0[nt] = pack8(kd[0] * D[0][nt], kd[1] * D[1][nt]);
        BS1[nt] = pack8(kd[2] * D[2][nt], kd[3] * D[3][nt]);
    }
    if constexpr (!kEarlyKt) load_kt();
    // (e) S <- gamma_C S + K^T (decay o dV)  (issued before (d): the recurrence's critical path).
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            S[r][nt] *= gC;
            S[r][nt] = mfma16x16x32(ktf[r][0], BS0[nt], S[r][nt]);
            S[r][nt] = mfma16x16x32(ktf[r][1], BS1[nt], S[r][nt]);
        }
    if constexpr (St::out) {
        bf16x8 BD0[NT], BD1[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            BD0[nt] = pack8(D[0][nt], D[1][nt]);
            BD1[nt] = pack8(D[2][nt], D[3][nt]);
        }
        // (d) O^T = (m scale gamma) o P^T + dV^T Aq^T, formed transposed so
        //     each lane holds 4 consecutive output columns of one token: the
        //     dV packs are the A operands and the Aq fragments the B operands
        //     as they stand (both carry their k in pi order), and P^T = S^T Q^T
        //     was accumulated with the operands of Q S swapped.  Lane (n, g) of
        //     tile mt stores out[token 16 mt + n][16 nt + 4 g .. + 3] as 8 bytes.
        float co[4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) co[mt] = G[64 + 16 * mt + n];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            f32x4 O[4];
            O[0] = mfma16x16x32(BD0[nt], af[0], co[0] * P[0][nt]);
            O[1] = mfma16x16x32(BD0[nt], af[1], co[1] * P[1][nt]);
            O[2] = mfma16x16x32(BD1[nt], af[3], mfma16x16x32(BD0[nt], af[2], co[2] * P[2][nt]));
            O[3] = mfma16x16x32(BD1[nt], af[5], mfma16x16x32(BD0[nt], af[4], co[3] * P[3][nt]));
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const int row = 16 * mt + n;
                if (row < nvalid)
                    *reinterpret_cast<u32x2*>(ob + row * orow + col0_wave + 16 * nt + 4 * g) = pack4_bf16(O[mt]);
            }
        }
    }
}

// Work decomposition of the state pass.
struct StateGrid {
    int nvg;         // workgroups per (head, group)
    int ngroups;     // chunk groups per sequence (G)
    int ngroups_run; // groups per sequence this launch covers (map pass: G - 1)
    int nheads;      // sequences x heads
    float* psi;      // [nheads][G][dv/16][8][64][4] fp32 (16-column tile, accumulator tile r,
                     // lane, slot): map pass zero-state results, then (scan) the initial
                     // state of group j + 1 in slot j
    uint16_t* phi;   // map pass: transitions as MFMA A fragments, [nheads][G][8][4][64][8]
                     // bf16 (row tile r, k-step, lane: row rho(r, n/4, n%4), columns 32ks + 8g..)
    // Packed sequences: per-sequence group counts planned on the device
    // (gdn_prefill_plan_kernel), or null for one group count G for all.
    // Table: [0] slots (sum of G_i), [1] map slots (sum of G_i - 1), then
    // (G_i, first slot of sequence i) for every sequence, then kPlanCap
    // entries (sequence << 8 | group) for every slot, then kPlanCap for every
    // map slot.  psi/phi of (sequence, head, group) sit at slot (first + group)
    // x H + head instead of ((sequence H + head) G + group).
    const int32_t* plan;
    int nseq;
};

constexpr int kPlanCap = 256;  // slot table capacity (slots per head never exceed 256 / H)
__device__ __forceinline__ int plan_groups(const StateGrid& sg, int sidx) { return sg.plan[2 + 2 * sidx]; }
__device__ __forceinline__ int plan_first(const StateGrid& sg, int sidx) { return sg.plan[3 + 2 * sidx]; }
// psi/phi unit of (sequence, head, group).
__device__ __forceinline__ size_t group_unit(const StateGrid& sg, int H, int sidx, int h, int grp) {
    return sg.plan ? static_cast<size_t>(plan_first(sg, sidx) + grp) * H + h
                   : static_cast<size_t>(sidx * H + h) * sg.ngroups + grp;
}

// State pass over one chunk group per workgroup (NW waves, NT 16-column tiles
// each, of one (sequence, head)).
//   kModeOut: from the group's initial state (state_in for group 0, else the
//             scan's result), writes the outputs; the last group writes
//             state_out.
//   kModeMap: columns [0, dv) start from zero (psi), columns [dv, dv + 128)
//             from the identity with V = 0 (phi = the group's transition).
//             The last group's map is never needed and is not computed.
// With one group (G = 1) only the output pass runs.  The chunk operands are
// shared by the waves and double-buffered in LDS: the copies for chunk c+1
// are in flight while chunk c is computed.
template <int MODE, int NW, int NT>
__global__ __launch_bounds__(64 * NW) void gdn_prefill_state_kernel(PrefillParams p, StateGrid sg) {
    using St = Stage<MODE, NW, NT>;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[2][St::bytes];
    lds_u8* const buf0 = (lds_u8*)&smem[0][0];
    lds_u8* const buf1 = (lds_u8*)&smem[1][0];

    const int wg = blockIdx.x;
    const int nunits = sg.nheads * sg.ngroups_run;
    int head, grp, vg, ngroups;
    if (sg.plan) {
        // ngroups_run = slots per head in the grid: (head, slot, column part)
        vg = wg % sg.nvg;
        const int hh = (wg / sg.nvg) / sg.ngroups_run, q = (wg / sg.nvg) % sg.ngroups_run;
        if (hh >= p.H || q >= sg.plan[MODE == kModeMap ? 1 : 0]) return;  // uniform over the workgroup
        const int e = sg.plan[2 + 2 * sg.nseq + (MODE == kModeMap ? kPlanCap : 0) + q];
        head = (e >> 8) * p.H + hh;
        grp = e & 255;
        ngroups = plan_groups(sg, e >> 8);
    } else {
        if (p.xcd_heads) {
            const HeadItem hi = head_major_xcd(wg, sg.ngroups_run * sg.nvg);
            head = hi.head;
            grp = hi.item / sg.nvg;
            vg = hi.item % sg.nvg;
        } else {
            vg = wg % sg.nvg;
            head = (wg / sg.nvg) / sg.ngroups_run;
            grp = (wg / sg.nvg) % sg.ngroups_run;
        }
        if (head * sg.ngroups_run + grp >= nunits) return;  // uniform over the workgroup
        ngroups = sg.ngroups;
    }
    const int sidx = head / p.H;
    const int h = head % p.H;
    const SeqInfo sq = seq_info(p, sidx);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int n = lane & 15, g = lane >> 4;
    const int dv = p.dv;
    const int col0_wave = (vg * NW + wave) * 16 * NT;  // map pass: >= dv means identity columns
    const bool phi_cols = MODE == kModeMap && col0_wave >= dv;
    const int nchunks = (sq.len + kC - 1) / kC;
    const int glen = (nchunks + ngroups - 1) / ngroups;
    const int c_begin = min(grp * glen, nchunks), c_end = min(c_begin + glen, nchunks);
    const StageLane L = {static_cast<uint32_t>(kslot_row(lane) * kDK * 2 + (lane >> 4) * 16),
                         static_cast<uint32_t>((lane & 15) * kDK * 2 + (lane >> 4) * 16),
                         static_cast<uint32_t>(16 * lane),
                         static_cast<uint32_t>((lane / (2 * NT)) * dv * 2 + (lane % (2 * NT)) * 16 +
                                               (phi_cols ? 0 : col0_wave) * 2)};

    const uint32_t kt_lane = kt_lane_offset(lane);

    // State tile: S[r][nt][i] = S[rho(r, g, i)][col0_wave + 16 nt + n].
    f32x4 S[8][NT];
    if constexpr (MODE == kModeMap) {
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    S[r][nt][i] = (phi_cols && rho_row(r, g, i) == col0_wave - dv + 16 * nt + n) ? 1.f : 0.f;
    } else if (grp > 0) {
        // Initial state of this group, left by the scan in psi slot grp - 1.
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f32x4* Ps = reinterpret_cast<const f32x4*>(
                sg.psi + (group_unit(sg, p.H, sidx, h, grp - 1) * (dv / 16) + col0_wave / 16 + nt) * 2048);
#pragma unroll
            for (int r = 0; r < 8; ++r) S[r][nt] = Ps[r * 64 + lane];
        }
    } else if (p.state_in) {
        const float* sin = p.state_in + static_cast<size_t>(sidx * p.H + h) * kDK * dv;
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) S[r][nt][i] = sin[rho_row(r, g, i) * dv + col0_wave + 16 * nt + n];
    } else {
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) S[r][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    const size_t head_row0 = static_cast<size_t>(sq.b * p.H + h) * p.T_stride + sq.tok0;
    auto rows = [&](int c) { return head_row0 + static_cast<size_t>(c) * kC; };
    // Output rows: head-major out[(sequence, head)][token][dv], or token-major
    // out[sequence][token][head][dv] (row stride H dv), as the caller asked.
    const int orow = p.out_tm ? p.H * dv : dv;
    auto obase = [&](int c) {
        const size_t tok = static_cast<size_t>(sq.b) * p.T_stride + sq.tok0 + static_cast<size_t>(c) * kC;
        return p.out_tm ? (tok * p.H + h) * dv : rows(c) * dv;
    };
    auto nval = [&](int c) { return min(kC, sq.len - c * kC); };
    auto wcof = [&](int c) { return static_cast<size_t>(sq.slot0 + c) * p.H + h; };
    auto step = [&](int c, lds_u8* cur, lds_u8* nxt) {
        // Chunk c's copies were issued before chunk c-1's output stores.
        if (c == c_begin)
            wait_vm<0>();
        else
            wait_vm<St::stores>();
        lds_barrier();  // chunk c staged by every wave; nobody still reads `nxt`
        const Stager<MODE, NW, NT> next = {&p,   nxt,  rows(c + 1), wcof(c + 1),     nval(c + 1), wave,
                                           lane, col0_wave, c + 1 < c_end, !phi_cols, &L};
        const int nv = nval(c);
        if (nv < kC) {
            zero_pad_rows<MODE, NW, NT>(cur, nv, wave, lane);
            lds_barrier();
        }
        state_chunk<MODE, NW, NT>(cur, S, p.out + obase(c), orow, nv, wave, lane, col0_wave, phi_cols, kt_lane,
                                  next);
    };

    {
        const Stager<MODE, NW, NT> first = {&p,   buf0, rows(c_begin), wcof(c_begin),   nval(c_begin), wave,
                                            lane, col0_wave, c_begin < c_end, !phi_cols, &L};
        first.issue();
    }
    for (int c = c_begin; c < c_end; c += 2) {
        step(c, buf0, buf1);
        if (c + 1 < c_end) step(c + 1, buf1, buf0);
    }

    if constexpr (MODE == kModeOut) {
        if (grp != ngroups - 1) return;
        float* so = p.state_out + static_cast<size_t>(sidx * p.H + h) * kDK * dv;
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) so[rho_row(r, g, i) * dv + col0_wave + 16 * nt + n] = S[r][nt][i];
    } else if (phi_cols) {
        // phi as A fragments: the accumulator holds 16-column tile T of phi
        // (a column per lane); a fragment lane needs 8 consecutive columns of
        // one row.  Transpose each 16x16 tile through this wave's own V area
        // (unused by identity columns), then store 512 contiguous bytes.
        uint16_t* Ph = sg.phi + group_unit(sg, p.H, sidx, h, grp) * kDK * kDK;
        lds_u16* tt = reinterpret_cast<lds_u16*>(buf0 + St::offV + wave * St::vWave);
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int T = (col0_wave - dv) / 16 + nt;
#pragma unroll
                for (int i = 0; i < 4; ++i) tt[(4 * g + i) * 16 + n] = f2bf_bits(S[r][nt][i]);
                if (lane < 32) {  // fragment lanes 16 (2 (T % 2) + h) + n: row n of the tile, columns 8h..
                    const int h = lane >> 4;
                    const u32x4 v = *reinterpret_cast<const lds_u32x4*>(tt + n * 16 + 8 * h);
                    *reinterpret_cast<u32x4*>(Ph + ((r * 4 + (T >> 1)) * 64 + 16 * (2 * (T & 1) + h) + n) * 8) = v;
                }
            }
    } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            f32x4* Ps = reinterpret_cast<f32x4*>(
                sg.psi + (group_unit(sg, p.H, sidx, h, grp) * (dv / 16) + col0_wave / 16 + nt) * 2048);
#pragma unroll
            for (int r = 0; r < 8; ++r) Ps[r * 64 + lane] = S[r][nt];
        }
    }
}

// ---------------------------------------------------------------------------
// Kernel 2b: the state pass for dv % 128 == 0 -- four compute waves of 32
// columns and one copy wave
// ---------------------------------------------------------------------------
// A workgroup owns 128 state columns of one (sequence, head, chunk group):
// compute wave w owns columns 32 w .. 32 w + 31 as two 16-column MFMA tiles,
// so every operand fragment it reads from LDS feeds two MFMAs (with 16-column
// waves, eight per CU, the LDS reads of a chunk step outlast its MFMAs).
// In the output pass three copy waves do all global memory traffic of the
// chunk loop: waves 4 and 5 stage chunk c + 1 (half of the copies each)
// while the compute waves work on chunk c, and wave 6 writes chunk c - 1's
// outputs, which the compute waves left in LDS, as whole 256-byte rows
// (77 KiB of memory traffic a chunk step): loads and stores from separate
// waves flow at the same time, and no compute wave stalls on a full memory
// queue.  (Staging chunk c + 2 through the loaders' registers, for two steps
// of copy latency instead of one, measured slower: the step is bound by its
// LDS traffic, not by the copies' latency.)  The output pass runs one workgroup per CU
// (one compute wave per SIMD), the map pass two.
// Per chunk, DMA-staged into one of two LDS buffers:
//   K   16 blocks of 8 rows x 64 columns (line_frag, line_ktfrag)
//   Q   the same (output pass)
//   record: Tp 6, Aq 6 (output pass), gate block 1
//   V   8 such blocks per 64 columns (not for phi columns)
// and in the output pass two output tiles [64 rows][128 columns] bf16 (row
// pitch 272 bytes: the compute waves' 8-byte writes then hit all 64 banks).
// Full chunks take a path without per-row checks; a sequence's partial last
// chunk clamps its copies to the sequence and predicates its output rows.
// Rows past the sequence end stay finite copies of the last row, and their Tp
// rows and columns are zero (beta m = 0 there), so they add exact zeros.
constexpr int kObPitch = 272;                // output tile row pitch (bytes)
constexpr int kObBytes = kC * kObPitch;      // one output tile
template <int MODE, int NT = 2>
struct Stage4 {
    static_assert(NT == 2 || (NT == 1 && MODE == kModeOut), "16-column tiles per compute wave");
    static constexpr bool out = MODE == kModeOut;
    static constexpr int cols = 64 * NT;  // state columns of a workgroup (4 compute waves x 16 NT)
    static constexpr int offK = 0;
    static constexpr int offQ = 16 * kFragB;
    static constexpr int offR = offQ + (out ? 16 : 0) * kFragB;
    // copied record fragments: Tp, the gate block and (output pass) the token block
    static constexpr int nRec = out ? kRecShort : kRecGShort + 1;
    static constexpr int offTp = offR;
    static constexpr int offG = offR + kRecGShort * kFragB;
    static constexpr int offH = offR + kRecH * kFragB;
    static constexpr int offAq = offR + nRec * kFragB;  // output pass: Aq, formed by the copy waves
    static constexpr int offV = offAq + (out ? 6 : 0) * kFragB;
    static constexpr int bytes = offV + 8 * NT * kFragB;  // V: [64 rows][32 columns] per 32 columns
    static constexpr int ob_bytes = out ? kObBytes : 0;
    // waves: 4 compute, then (output pass) 2 copying chunks in, a store wave
    // and the Aq wave
    static constexpr int loaders = out ? 2 : 0;
    static constexpr int nWaves = 4 + loaders + (out ? 2 : 0);
    static constexpr int nStores = out ? kC * 256 / kFragB : 0;  // output store instructions per chunk
};

// Per-lane byte offsets of the copies (fixed for the kernel).
struct Lane4 {
    uint32_t k, r, v;  // K and Q rows, record fragments, V rows
};

// Staged K, Q and V: 1 KiB blocks of 8 rows x 64 columns (one 128-byte line a
// row), block 2 rb + h of K and Q holding rows 8 rb .. and columns 64 h ..,
// block 8 h + rb of V likewise.  Chunk c (8 columns) of a row sits in slot
// c ^ (row % 8), so fragment reads (8 rows, one chunk each) and the
// transposing reads spread over the banks.  Copies of whole lines enter LDS
// faster than those of 64-byte row pieces (a fragment's shape): the L2 serves
// a request per line piece.
__device__ __forceinline__ uint32_t line_chunk(int lane) {  // byte offset of the lane's source chunk in its row
    return 16u * static_cast<uint32_t>((lane & 7) ^ (lane >> 3));
}
// Lane address of a fragment (row m, k group g) of a 16-row, 32-column tile in
// those blocks; odd 32-column steps XOR 64.
__device__ __forceinline__ uint32_t line_frag_lane(int lane) {
    const int m = lane & 15, g = lane >> 4;
    return static_cast<uint32_t>((m >> 3) * 2048 + (m & 7) * 128 + ((g ^ (m & 7)) << 4));
}
// Fragment (rows 16 mt .., columns 32 s ..) of staged K or Q.
__device__ __forceinline__ bf16x8 line_frag(const lds_u8* base, int mt, int s, uint32_t fl) {
    return *reinterpret_cast<const lds_bf16x8*>(base + mt * 4096 + (s >> 1) * 1024 + ((s & 1) ? fl ^ 64u : fl));
}
// K^T fragment (r, s) from those blocks (as ktfrag): source lane 4 j + a of
// group g reads row 32 s + 16 u + 4 g + j, columns 32 (r / 2) + 8 a + 4 (r % 2) ..
__device__ __forceinline__ uint32_t line_kt_lane(int lane) {
    const int g = lane >> 4, j = (lane >> 2) & 3, a = lane & 3, row = 4 * (g & 1) + j;
    return static_cast<uint32_t>((g >> 1) * 2048 + row * 128 + ((a ^ row) << 4));
}
__device__ __forceinline__ bf16x8 line_ktfrag(const lds_u8* base, uint32_t kl, int r, int s) {
    const lds_u8* q = base + s * 8192 + (r >> 2) * 1024 + 8 * (r & 1) + (((r >> 1) & 1) ? kl ^ 64u : kl);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)q));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(q + 4096)));
    return as_bf16x8(u32x4{lo[0], lo[1], hi[0], hi[1]});
}

// Issue chunk `c`'s copies into `buf`: jobs first, first + STRIDE, ... of
// each kind (the output pass's copy wave takes all of them, STRIDE 1; in the
// map pass each compute wave takes a quarter, STRIDE 4).  `row0`: q/k/v row
// of the chunk's first token; `rec`: the chunk's record; `vcol0`: the
// workgroup's first V column.
template <int MODE, int NT, bool FULL, int STRIDE>
__device__ __forceinline__ void stage4_issue(const PrefillParams& p, lds_u8* buf, size_t row0, const u32x4* rec,
                                             int vcol0, int nvalid, int first, int lane, const Lane4& L, bool v_on) {
    using St = Stage4<MODE, NT>;
    // Full chunks: uniform bases, fixed lane offsets.  The partial chunk:
    // base at the chunk's first row and each lane's row clamped to the
    // sequence, so every offset is non-negative and in range.
    // A copy of K, Q or V reads 8 rows of 128 bytes (whole lines).
    const unsigned char* kc = reinterpret_cast<const unsigned char*>(p.k + row0 * kDK);
    const unsigned char* qc = reinterpret_cast<const unsigned char*>(p.q + row0 * kDK);
    auto copy_rows = [&](const unsigned char* base, int f, lds_u8* dst) {  // f = 2 rb + h: rows 8 rb .., columns 64 h ..
        const int rb = f >> 1, h = f & 1;
        if (FULL)
            dma16(base + rb * 8 * kDK * 2 + 128 * h, L.k, dst + f * kFragB);
        else
            dma16(base, static_cast<uint32_t>(min(8 * rb + (lane >> 3), nvalid - 1) * kDK * 2 + 128 * h) + line_chunk(lane),
                  dst + f * kFragB);
    };
#pragma unroll
    for (int i = 0; i < 16 / STRIDE; ++i) copy_rows(kc, first + STRIDE * i, buf + St::offK);
    if constexpr (St::out) {
#pragma unroll
        for (int i = 0; i < 16 / STRIDE; ++i) copy_rows(qc, first + STRIDE * i, buf + St::offQ);
    }
    const unsigned char* rb = reinterpret_cast<const unsigned char*>(rec);
#pragma unroll
    for (int i = 0; i < (St::nRec + STRIDE - 1) / STRIDE; ++i) {
        const int j = first + STRIDE * i;
        if (j < St::nRec) {
            dma16(rb + j * kFragB, L.r, buf + St::offR + j * kFragB);
        }
    }
    if (v_on) {  // job u: columns 64 (u / 8) .., rows 8 (u % 8) ..
        const unsigned char* vb = reinterpret_cast<const unsigned char*>(p.v + row0 * p.dv + vcol0);
#pragma unroll
        for (int i = 0; i < 8 * NT / STRIDE; ++i) {
            const int u = first + STRIDE * i, hv = u >> 3, rv = u & 7;
            lds_u8* vd = buf + St::offV + u * kFragB;
            if (FULL)
                dma16(vb + static_cast<size_t>(8 * rv) * p.dv * 2 + 128 * hv, L.v, vd);
            else
                dma16(vb, static_cast<uint32_t>(min(8 * rv + (lane >> 3), nvalid - 1) * p.dv * 2 + 128 * hv) + line_chunk(lane),
                      vd);
        }
    }
}

// The output pass's copy waves form the six nonzero fragments of the staged
// chunk's causal Aq = (m scale) (Q K^T o Gamma) into the buffer's Aq area,
// from the staged Q and K and the token block, each wave the fragments of
// SLOTS (bit i: fragment i), so that the Aq products are spread over the four
// SIMDs instead of queueing behind one compute wave's products on one.
// Each 16x16 tile (t, s) is formed transposed, as K_s Q_t^T: its accumulator
// (lane (n, g): s rows 4 g + i of token column n) is then, packed, half of a
// fragment (mt, S) as the B operand of dV^T Aq^T reads it (lane (n, g): token
// 16 mt + n, s in pi order).  Rows past a sequence's end are clamped copies;
// their tokens have m scale = 0.
//   fragment: 0      1            2            3      4            5
//   tiles:    (0,0)  (1,0),(1,1)  (2,0),(2,1)  (2,2)  (3,0),(3,1)  (3,2),(3,3)
template <unsigned SLOTS>
__device__ __forceinline__ void stage4_aq(lds_u8* buf, int lane) {
    using St = Stage4<kModeOut>;
    constexpr int t_of[6] = {0, 1, 2, 2, 3, 3};
    constexpr int s_lo[6] = {0, 0, 0, 2, 0, 2};  // first tile's s (the second's is s + 1)
    constexpr bool two[6] = {false, true, true, false, true, true};
    auto needs_q = [](int t) {
        for (int i = 0; i < 6; ++i)
            if (((SLOTS >> i) & 1) && t_of[i] == t) return true;
        return false;
    };
    auto needs_k = [](int s) {
        for (int i = 0; i < 6; ++i)
            if (((SLOTS >> i) & 1) && (s_lo[i] == s || (two[i] && s_lo[i] + 1 == s))) return true;
        return false;
    };
    const int n = lane & 15, g = lane >> 4;
    const uint32_t fl = line_frag_lane(lane);
    const lds_f32* Hb = reinterpret_cast<const lds_f32*>(buf + St::offH);
    bf16x8 qf[4][4], kf[4][4];
    float lt[4], mt[4];
    f32x4 ls[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (needs_q(t)) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) qf[t][kk] = line_frag(buf + St::offQ, t, kk, fl);
            lt[t] = Hb[16 * t + n];
            mt[t] = Hb[64 + 16 * t + n];
        }
        if (needs_k(t)) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) kf[t][kk] = line_frag(buf + St::offK, t, kk, fl);
            ls[t] = *reinterpret_cast<const lds_f32x4*>(Hb + 16 * t + 4 * g);
        }
    }
    auto tile = [&](int ti, int si) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) acc = mfma16x16x32(kf[si][kk], qf[ti][kk], acc);
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = mt[ti] * acc[i] * __builtin_amdgcn_exp2f(lt[ti] - ls[si][i]);
            v[i] = (ti > si || 4 * g + i <= n) ? x : 0.f;
        }
        return pack4_bf16(v);
    };
    const u32x2 z = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        if ((SLOTS >> i) & 1) {
            const u32x2 lo = tile(t_of[i], s_lo[i]);
            const u32x2 hi = two[i] ? tile(t_of[i], s_lo[i] + 1) : z;
            *reinterpret_cast<lds_u32x4*>(buf + St::offAq + i * kFragB + 16 * lane) = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    }
}

// The copy wave: chunk c's output tile from LDS to `ob` (row 0, the
// workgroup's first column), rows of RB bytes (the workgroup's columns): 4
// rows of 256 bytes or 8 rows of 128 bytes per instruction.
template <bool FULL, int RB>
__device__ __forceinline__ void stage4_store(const lds_u8* obuf, uint16_t* ob, int orow, int nvalid, int lane) {
    constexpr int LPR = RB / 16;  // lanes per row
    static_assert(LPR == 16 || LPR == 8, "output row bytes");
    // Opaque per call: otherwise the per-lane row offsets are hoisted out of
    // the chunk loop and held in registers that every wave then pays for.
    asm volatile("" : "+s"(orow));
#pragma unroll
    for (int i = 0; i < kC * LPR / 64; ++i) {
        const int row = (64 / LPR) * i + lane / LPR;
        const u32x4 v = *reinterpret_cast<const lds_u32x4*>(obuf + row * kObPitch + (lane % LPR) * 16);
        if (FULL || row < nvalid)  // streamed out: nothing in this pass reads the outputs back
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(ob + static_cast<size_t>(row) * orow + (lane % LPR) * 8));
    }
}

// One chunk of the state recurrence for this wave's 128 x 32 state tile, the
// chunk's operands staged in `buf`; the output pass leaves the chunk's
// outputs in the LDS tile `obuf` for the copy wave.
// LDS reads run one phase ahead of the MFMAs that consume them: K S and
// S^T Q^T go in four k-groups, each group's MFMAs issued after the next
// group's fragment reads, and each later phase's operands (V and the gates,
// Tp, K^T, Aq) are read while the phase before it computes.  Phase fences
// (PHASE()) keep that order: the scheduler would otherwise sink reads to
// their first use (exposing the LDS latency at every one) or hoist all of
// them to the top (past the 256 VGPRs a wave has).
template <int MODE, int NT, typename Mid>
__device__ __forceinline__ void state4_step(const lds_u8* buf, f32x4 (&S)[8][NT], lds_u8* obuf, int wave, int lane,
                                            bool v_zero, uint32_t kt_lane, Mid mid) {
    using St = Stage4<MODE, NT>;
    constexpr bool OUT = St::out;
    const int n = lane & 15, g = lane >> 4;
    const lds_f32* G = reinterpret_cast<const lds_f32*>(buf + St::offG);
    // This wave's columns of the staged V: chunks vc0 .. of 64-column block
    // vh (a 32-column wave half of a block, a 16-column wave a quarter).
    const int vh = NT == 2 ? wave >> 1 : 0, vc0 = NT == 2 ? 4 * (wave & 1) : 2 * wave;
    const uint32_t fl = line_frag_lane(lane);
#define PHASE() __builtin_amdgcn_sched_barrier(0)

    // (a) X = K S and P^T = S^T Q^T.  The state's bf16 copy is the B operand
    //     of K S and the A operand of S^T Q^T as it stands (k = state rows
    //     32 s + 8 g + j in both).
    bf16x8 kf[2][4], qf[2][OUT ? 4 : 1];
    auto load_a = [&](int s, int slot) {
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            kf[slot][mt] = line_frag(buf + St::offK, mt, s, fl);
            if constexpr (OUT) qf[slot][mt] = line_frag(buf + St::offQ, mt, s, fl);
        }
    };
    i16x4 vv[NT][4];
    f32x4 gam[4], kd[4];
    float gC = 0.f;
    // (b)'s operands: V in the accumulator layout (column n, rows
    // 16 mt + 4 g + i) -- source lane 4 j + a of group g of a transposing read
    // fetches row 16 mt + 4 g + j, columns 16 nt + 4 a .. -- and the gates.
    auto load_b = [&]() {
        const int vr = 4 * (g & 1) + ((lane >> 2) & 3);  // row % 8
        const uint32_t vl = static_cast<uint32_t>(vh * 8192 + (g >> 1) * 1024 + vr * 128 +
                                                  (((vc0 + ((lane & 3) >> 1)) ^ vr) << 4) + 8 * (lane & 1));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
                vv[nt][mt] = v_zero ? i16x4{0, 0, 0, 0}
                                    : __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                          (lds_i16x4*)(buf + St::offV + mt * 2048 + (vl ^ (32u * nt))));
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            gam[mt] = *reinterpret_cast<const lds_f32x4*>(G + 16 * mt + 4 * g);
            kd[mt] = *reinterpret_cast<const lds_f32x4*>(G + 128 + 16 * mt + 4 * g);
        }
        gC = G[kC - 1];
    };
    f32x4 X[4][NT], P[4][NT];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) X[mt][nt] = P[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    load_a(0, 0);
    PHASE();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (s < 3)
            load_a(s + 1, (s + 1) & 1);
        else
            load_b();
        bf16x8 Bs[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) Bs[nt] = pack8(S[2 * s][nt], S[2 * s + 1][nt]);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                X[mt][nt] = mfma16x16x32(kf[s & 1][mt], Bs[nt], X[mt][nt]);
                if constexpr (OUT) P[mt][nt] = mfma16x16x32(Bs[nt], qf[s & 1][mt], P[mt][nt]);
            }
        PHASE();
    }
    // (b) Y = V - gamma o X (in place in X), while Tp is read.
    bf16x8 tf[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) tf[i] = frag(buf, St::offTp + i * kFragB, lane);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                X[mt][nt][i] = bf2f(static_cast<uint16_t>(vv[nt][mt][i])) - gam[mt][i] * X[mt][nt][i];
    bf16x8 BY[2][NT];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) BY[s][nt] = pack8(X[2 * s][nt], X[2 * s + 1][nt]);
    PHASE();
    // (c) dV = Tp Y (Tp lower triangular: six nonzero fragments), while the
    //     first half of K^T is read.
    bf16x8 ktf[8][2];
    auto load_kt = [&](int r0) {
#pragma unroll
        for (int r = r0; r < r0 + 4; ++r) {
            ktf[r][0] = line_ktfrag(buf + St::offK, kt_lane, r, 0);
            ktf[r][1] = line_ktfrag(buf + St::offK, kt_lane, r, 1);
        }
    };
    load_kt(0);
    f32x4 D[4][NT];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) D[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int mt = 2 * s; mt < 4; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) D[mt][nt] = mfma16x16x32(tf[aq_index(mt, s)], BY[s][nt], D[mt][nt]);
    PHASE();
    // (d) S <- gamma_C S + K^T ((gamma_C / gamma) o dV) in two halves of
    //     row tiles: the second half of K^T is read during the first, Aq
    //     during the second.
    bf16x8 af[OUT ? 6 : 1];
    float co[4];
    bf16x8 BS0[NT], BS1[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        BS0[nt] = pack8(kd[0] * D[0][nt], kd[1] * D[1][nt]);
        BS1[nt] = pack8(kd[2] * D[2][nt], kd[3] * D[3][nt]);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half == 0) {
            load_kt(4);
        } else if constexpr (OUT) {
            mid();  // the copy waves have formed Aq
#pragma unroll
            for (int i = 0; i < 6; ++i) af[i] = frag(buf, St::offAq + i * kFragB, lane);
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) co[mt] = G[64 + 16 * mt + n];
        }
#pragma unroll
        for (int r = 4 * half; r < 4 * half + 4; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                S[r][nt] *= gC;
                S[r][nt] = mfma16x16x32(ktf[r][0], BS0[nt], S[r][nt]);
                S[r][nt] = mfma16x16x32(ktf[r][1], BS1[nt], S[r][nt]);
            }
        PHASE();
    }
    // (e) O^T = (m scale gamma) o P^T + dV^T Aq^T: each lane holds 4
    //     consecutive output columns of token 16 mt + n, written to the
    //     output tile as 8 bytes.
    if constexpr (OUT) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const bf16x8 BD0 = pack8(D[0][nt], D[1][nt]), BD1 = pack8(D[2][nt], D[3][nt]);
            f32x4 O[4];
            O[0] = mfma16x16x32(BD0, af[0], co[0] * P[0][nt]);
            O[1] = mfma16x16x32(BD0, af[1], co[1] * P[1][nt]);
            O[2] = mfma16x16x32(BD1, af[3], mfma16x16x32(BD0, af[2], co[2] * P[2][nt]));
            O[3] = mfma16x16x32(BD1, af[5], mfma16x16x32(BD0, af[4], co[3] * P[3][nt]));
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
                *reinterpret_cast<lds_u32x2*>(obuf + (16 * mt + n) * kObPitch + (16 * NT * wave + 16 * nt + 4 * g) * 2) =
                    pack4_bf16(O[mt]);
        }
    }
#undef PHASE
}

// The state pass of one workgroup: 128 columns of one (sequence, head,
// chunk group) in the roles of gdn_prefill_state_kernel (output pass: from
// the group's initial state, outputs and the final state; map pass: psi
// columns from zero with V, phi columns from the identity without V).
// This file is compiled with MFMA results forced into VGPRs (the build's
// -amdgpu-mfma-vgpr-form): with one compute wave per SIMD the compiler would
// otherwise park the accumulators in AGPRs and copy them back for every VALU
// use, about 300 extra instructions per chunk.
// The output pass adds the copy waves.  In the map pass (two workgroups per
// CU, 39 KiB a chunk step each) the compute waves issue a quarter of the
// copies each: dedicated copy waves there measured slower.
template <int MODE, int NT>
__global__ __launch_bounds__((64 * Stage4<MODE, NT>::nWaves)) __attribute__((amdgpu_waves_per_eu(
    MODE == kModeOut ? 1 : 2, 2))) void gdn_prefill_state4_kernel(PrefillParams p, StateGrid sg) {
    using St = Stage4<MODE, NT>;
    constexpr bool OUT = St::out;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * St::bytes + 2 * St::ob_bytes];
    auto buf = [&](int i) { return (lds_u8*)&smem[0] + i * St::bytes; };
    auto obuf = [&](int i) { return (lds_u8*)&smem[0] + 2 * St::bytes + i * St::ob_bytes; };

    const int wg = blockIdx.x;
    int head, grp, vg, ngroups;
    if (sg.plan) {
        vg = wg % sg.nvg;
        const int hh = (wg / sg.nvg) / sg.ngroups_run, q = (wg / sg.nvg) % sg.ngroups_run;
        if (hh >= p.H || q >= sg.plan[MODE == kModeMap ? 1 : 0]) return;  // uniform over the workgroup
        const int e = sg.plan[2 + 2 * sg.nseq + (MODE == kModeMap ? kPlanCap : 0) + q];
        head = (e >> 8) * p.H + hh;
        grp = e & 255;
        ngroups = plan_groups(sg, e >> 8);
    } else {
        if (p.xcd_heads) {
            const HeadItem hi = head_major_xcd(wg, sg.ngroups_run * sg.nvg);
            head = hi.head;
            grp = hi.item / sg.nvg;
            vg = hi.item % sg.nvg;
        } else {
            vg = wg % sg.nvg;
            head = (wg / sg.nvg) / sg.ngroups_run;
            grp = (wg / sg.nvg) % sg.ngroups_run;
        }
        if (head * sg.ngroups_run + grp >= sg.nheads * sg.ngroups_run) return;  // uniform over the workgroup
        ngroups = sg.ngroups;
    }
    const int sidx = head / p.H;
    const int h = head % p.H;
    const SeqInfo sq = seq_info(p, sidx);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Copy waves (output pass): 4 and 5 copy chunk c + 1 in, 6 writes chunk
    // c - 1's outputs, and all four form chunk c's Aq.  In the map pass the
    // compute waves copy (`issuer`).
    const bool loader = OUT && wave >= 4 && wave < 4 + St::loaders;
    const bool storer = OUT && wave == 4 + St::loaders;
    const bool aqw = OUT && wave == 5 + St::loaders;
    const bool issuer = OUT ? loader : true;
    const bool copier = loader || storer || aqw;
    const int cw = copier ? 0 : wave;  // compute wave (column block)
    const int lane = threadIdx.x & 63;
    const int n = lane & 15, g = lane >> 4;
    const int dv = p.dv;
    const int col0_wave = vg * St::cols + 16 * NT * cw;  // map pass: >= dv means identity columns
    const bool phi_cols = MODE == kModeMap && vg * St::cols >= dv;
    const int vcol0 = phi_cols ? 0 : vg * St::cols;
    const int nchunks = (sq.len + kC - 1) / kC;
    const int glen = (nchunks + ngroups - 1) / ngroups;
    const int c_begin = min(grp * glen, nchunks), c_end = min(c_begin + glen, nchunks);
    const Lane4 L = {static_cast<uint32_t>((lane >> 3) * kDK * 2) + line_chunk(lane), static_cast<uint32_t>(16 * lane),
                     static_cast<uint32_t>((lane >> 3) * dv * 2) + line_chunk(lane)};
    const uint32_t kt_lane = line_kt_lane(lane);

    const size_t head_row0 = static_cast<size_t>(sq.b * p.H + h) * p.T_stride + sq.tok0;
    const int orow = p.out_tm ? p.H * dv : dv;
    auto rows = [&](int c) { return head_row0 + static_cast<size_t>(c) * kC; };
    auto obase = [&](int c) {  // out row of chunk c's first token, the workgroup's first column
        const size_t tok = static_cast<size_t>(sq.b) * p.T_stride + sq.tok0 + static_cast<size_t>(c) * kC;
        return p.out + (p.out_tm ? (tok * p.H + h) * dv : rows(c) * dv) + vg * St::cols;
    };
    auto nval = [&](int c) { return min(kC, sq.len - c * kC); };
    auto rec = [&](int c) { return p.wsR + (static_cast<size_t>(sq.slot0 + c) * p.H + h) * kRecShort * 64; };
    auto issue = [&](int c, int bi) {
        // Opaque per call: otherwise the copies' LDS addresses (buffer and
        // fragment constants) are hoisted out of the chunk loop and held in
        // SGPRs, which runs the kernel out of them.
        int first = OUT ? wave - 4 : wave;
        asm volatile("" : "+s"(first));
        lds_u8* b = buf(bi);
        constexpr int STRIDE = OUT ? St::loaders : 4;
        if (nval(c) == kC)
            stage4_issue<MODE, NT, true, STRIDE>(p, b, rows(c), rec(c), vcol0, kC, first, lane, L, !phi_cols);
        else
            stage4_issue<MODE, NT, false, STRIDE>(p, b, rows(c), rec(c), vcol0, nval(c), first, lane, L, !phi_cols);
    };

    // Chunk c = c_begin + k uses buffer k % 2 and output tile k % 2.  Barrier
    // k opens step k: chunk c is staged, nobody reads buffer (k + 1) % 2 any
    // more, and chunk c - 1's outputs are in tile (k - 1) % 2.  In the output
    // pass a second barrier per step, in the middle of the compute waves'
    // state update, publishes chunk c's Aq, formed meanwhile by the copy waves.
    // The copy waves run their own loop (with the same barriers), so the
    // compute waves' state is not live in it.
    if constexpr (OUT) {
        if (copier) {
            if (loader && c_begin < c_end) issue(c_begin, 0);
            for (int c = c_begin; c < c_end; ++c) {
                const int k = c - c_begin;
                if (loader) wait_vm<0>();  // chunk c staged
                lds_barrier();
                if (loader && c + 1 < c_end) issue(c + 1, (k + 1) & 1);
                // Chunk c's Aq: each copy wave (one a SIMD) forms 2 or 3 of its 10 tiles.
                static_assert(St::loaders == 2, "copy waves 4..7");
                if (wave == 4) stage4_aq<0x28>(buf(k & 1), lane);  // (2,2), (3,2), (3,3)
                if (wave == 5) stage4_aq<0x11>(buf(k & 1), lane);  // (0,0), (3,0), (3,1)
                if (wave == 6) stage4_aq<0x04>(buf(k & 1), lane);  // (2,0), (2,1)
                if (wave == 7) stage4_aq<0x02>(buf(k & 1), lane);  // (1,0), (1,1)
                // Chunk c - 1 is never a sequence's partial last chunk here.
                if (storer && k >= 1) stage4_store<true, 2 * St::cols>(obuf((k - 1) & 1), obase(c - 1), orow, kC, lane);
                lds_barrier();  // chunk c's Aq formed
            }
            lds_barrier();  // the last chunk's outputs are in LDS
            if (storer && c_end > c_begin) {
                const int c = c_end - 1, k = c - c_begin;
                if (nval(c) == kC)
                    stage4_store<true, 2 * St::cols>(obuf(k & 1), obase(c), orow, kC, lane);
                else
                    stage4_store<false, 2 * St::cols>(obuf(k & 1), obase(c), orow, nval(c), lane);
            }
            return;
        }
    }

    // State tile: S[r][nt][i] = S[rho(r, g, i)][col0_wave + 16 nt + n].
    f32x4 S[8][NT];
    if constexpr (MODE == kModeMap) {
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    S[r][nt][i] = (phi_cols && rho_row(r, g, i) == col0_wave - dv + 16 * nt + n) ? 1.f : 0.f;
    } else if (grp > 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f32x4* Ps = reinterpret_cast<const f32x4*>(
                sg.psi + (group_unit(sg, p.H, sidx, h, grp - 1) * (dv / 16) + col0_wave / 16 + nt) * 2048);
#pragma unroll
            for (int r = 0; r < 8; ++r) S[r][nt] = Ps[r * 64 + lane];
        }
    } else if (p.state_in) {
        const float* sin = p.state_in + static_cast<size_t>(sidx * p.H + h) * kDK * dv;
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) S[r][nt][i] = sin[rho_row(r, g, i) * dv + col0_wave + 16 * nt + n];
    } else {
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) S[r][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    if (!OUT && c_begin < c_end) issue(c_begin, 0);
    for (int c = c_begin; c < c_end; ++c) {
        const int k = c - c_begin;
        if (!OUT) wait_vm<0>();  // chunk c staged (the map pass's compute waves copy)
        lds_barrier();
        if (!OUT && c + 1 < c_end) issue(c + 1, (k + 1) & 1);
        state4_step<MODE, NT>(buf(k & 1), S, obuf(k & 1), cw, lane, phi_cols, kt_lane, [] { lds_barrier(); });
    }

    if constexpr (OUT) {
        lds_barrier();  // the last chunk's outputs are in LDS (matches the copy waves' final barrier)
        if (grp != ngroups - 1) return;
        float* so = p.state_out + static_cast<size_t>(sidx * p.H + h) * kDK * dv;
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) so[rho_row(r, g, i) * dv + col0_wave + 16 * nt + n] = S[r][nt][i];
    } else if (phi_cols) {
        // phi as A fragments, transposed 16x16 tile by tile through this
        // wave's V area of buffer 0 (unused by identity columns): no copy is
        // in flight any more, and no other wave reads that area.
        uint16_t* Ph = sg.phi + group_unit(sg, p.H, sidx, h, grp) * kDK * kDK;
        lds_u16* tt = reinterpret_cast<lds_u16*>(buf(0) + St::offV + cw * 4 * kFragB);
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int T = (col0_wave - dv) / 16 + nt;
#pragma unroll
                for (int i = 0; i < 4; ++i) tt[(4 * g + i) * 16 + n] = f2bf_bits(S[r][nt][i]);
                if (lane < 32) {  // fragment lanes 16 (2 (T % 2) + h2) + n: row n of the tile, columns 8 h2 ..
                    const int h2 = lane >> 4;
                    const u32x4 v = *reinterpret_cast<const lds_u32x4*>(tt + n * 16 + 8 * h2);
                    *reinterpret_cast<u32x4*>(Ph + ((r * 4 + (T >> 1)) * 64 + 16 * (2 * (T & 1) + h2) + n) * 8) = v;
                }
            }
    } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            f32x4* Ps = reinterpret_cast<f32x4*>(sg.psi +
                                                 (group_unit(sg, p.H, sidx, h, grp) * (dv / 16) + col0_wave / 16 + nt) * 2048);
#pragma unroll
            for (int r = 0; r < 8; ++r) Ps[r * 64 + lane] = S[r][nt];
        }
    }
}

// Initial states of the chunk groups: S_in(0) = state_in (or 0) and
// S_in(j + 1) = phi_j S_in(j) + psi_j, written over psi_j.  One workgroup of
// 8 waves per (sequence-head, 16-column tile); wave w owns accumulator row
// tile r = w (state rows rho(w, g, i)).  Row tiles 2s and 2s + 1 make up
// MFMA k-step s, so wave w publishes its rows as one 8-byte half of k-step
// w / 2's B operand (bf16 high and low parts of the fp32 state, which give
// two independent accumulation chains) and every wave reads all four k-steps
// back.  The steps are a dependent chain, so what bounds a step is latency:
// each wave holds its phi fragments and psi quad for the next kScanDepth
// steps in registers (20 VGPRs a step), loaded kScanDepth steps before use,
// which covers the memory latency that a shallower LDS ring (limited to 3
// steps by LDS capacity) did not.
constexpr int kScanDepth = 6;
constexpr int kMaxGroups = 16;  // chunk groups per sequence (plan_state caps G here)

__device__ __forceinline__ u32x2 pack4_hi(const f32x4 v) { return pack4_bf16(v); }
// bf16 of (x - bf16(x)): the low part of a two-term bf16 split.
__device__ __forceinline__ u32x2 pack4_lo(const f32x4 v, const u32x2 hi) {
    f32x4 d;
    d[0] = v[0] - __uint_as_float(hi[0] << 16);
    d[1] = v[1] - __uint_as_float(hi[0] & 0xffff0000u);
    d[2] = v[2] - __uint_as_float(hi[1] << 16);
    d[3] = v[3] - __uint_as_float(hi[1] & 0xffff0000u);
    return pack4_hi(d);
}

// STEPS = G - 1 is a template parameter so that the step loop unrolls
// completely with static register slots and exact wait counts (a rolled
// loop makes the compiler wait for every outstanding load at its header).
// PLANNED: per-sequence group counts (sg.plan); STEPS is then the most any
// sequence can have and each workgroup stops after its own G_i - 1 steps.
template <int STEPS, bool PLANNED>
__global__ __launch_bounds__(512) void gdn_prefill_scan_kernel(PrefillParams p, StateGrid sg) {
    static_assert(STEPS >= 1 && STEPS < kMaxGroups, "scan steps");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * 8 * kFragB];
    const int dv = p.dv, ntile = dv / 16;
    const int nunits = sg.nheads * ntile;
    if (static_cast<int>(blockIdx.x) >= nunits) return;  // uniform over the workgroup
    int head, tile;
    if (p.xcd_heads) {
        const HeadItem hi = head_major_xcd(blockIdx.x, ntile);
        head = hi.head;
        tile = hi.item;
    } else {
        head = blockIdx.x / ntile;
        tile = blockIdx.x % ntile;
    }
    const int sidx = head / p.H, h = head % p.H;
    const int nsteps = PLANNED ? plan_groups(sg, sidx) - 1 : STEPS;
    if (PLANNED && nsteps <= 0) return;  // one group: nothing to compose
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // = row tile r
    const int lane = threadIdx.x & 63;
    const int n = lane & 15, g = lane >> 4;
    const int col = 16 * tile + n;
    lds_u8* const sbuf = (lds_u8*)&smem[0];

    f32x4 S;
    if (p.state_in) {
        const float* sin = p.state_in + static_cast<size_t>(sidx * p.H + h) * kDK * dv;
#pragma unroll
        for (int i = 0; i < 4; ++i) S[i] = sin[rho_row(wave, g, i) * dv + col];
    } else {
        S = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // psi/phi unit of group j: unit0 + j ustride (group_unit, with the plan
    // table read once here: a table read inside the step loop would come with
    // a wait for every load in flight, the prefetched steps included).
    const size_t unit0 = PLANNED ? static_cast<size_t>(plan_first(sg, sidx)) * p.H + h
                                 : static_cast<size_t>(sidx * p.H + h) * sg.ngroups;
    const size_t ustride = PLANNED ? static_cast<size_t>(p.H) : 1;
    auto unit = [&](int j) { return unit0 + static_cast<size_t>(j) * ustride; };
    auto psi_at = [&](int j) {
        return reinterpret_cast<f32x4*>(sg.psi + (unit(j) * ntile + tile) * 2048) + wave * 64 + lane;
    };
    // This wave's phi fragments (row tile r, k-steps 0..3: 4 contiguous KiB)
    // and psi quad r of step j, into register slot j % kScanDepth.
    constexpr int D = STEPS < kScanDepth ? STEPS : kScanDepth;
    u32x4 ph[D][4];
    f32x4 ps[D];
    auto load = [&](int j) {
        const u32x4* src = reinterpret_cast<const u32x4*>(sg.phi + unit(j) * kDK * kDK) + 4 * wave * 64 + lane;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) ph[j % D][ks] = src[ks * 64];
        ps[j % D] = *psi_at(j);
        // Keep each step's loads together and in step order: the wait for
        // step j then only covers what was issued up to step j.
        __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < D; ++j)
        if (!PLANNED || j < nsteps) load(j);
    const int half = (wave & 1) * 8;  // this row tile's bytes in its k-step's B fragment
    auto publish = [&](lds_u8* buf) {
        const u32x2 hi = pack4_hi(S);
        *reinterpret_cast<lds_u32x2*>(buf + (2 * (wave >> 1)) * kFragB + 16 * lane + half) = hi;
        *reinterpret_cast<lds_u32x2*>(buf + (2 * (wave >> 1) + 1) * kFragB + 16 * lane + half) = pack4_lo(S, hi);
    };
    // From a zero initial state the first step is S_in(1) = psi_0 (phi_0 0 +
    // psi_0 adds exact zeros), which psi_0's slot already holds: it is taken
    // as is, one dependent step shorter.
    const bool zero_start = p.state_in == nullptr;
    if (!zero_start) publish(sbuf);
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        if (PLANNED && j >= nsteps) continue;  // uniform over the workgroup (the loop still unrolls)
        if (j == 0 && zero_start) {
            S = ps[0];
            if (D < STEPS && (!PLANNED || D < nsteps)) load(D);
            publish(sbuf + 8 * kFragB);
            continue;
        }
        lds_u8* const buf = sbuf + (j & 1) * 8 * kFragB;
        lds_barrier();
        f32x4 acc_h = ps[j % D];
        f32x4 acc_l = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const bf16x8 a = as_bf16x8(ph[j % D][ks]);
            acc_h = mfma16x16x32(a, frag(buf, (2 * ks) * kFragB, lane), acc_h);
            acc_l = mfma16x16x32(a, frag(buf, (2 * ks + 1) * kFragB, lane), acc_l);
        }
        if (j + D < STEPS && (!PLANNED || j + D < nsteps)) load(j + D);
        S = acc_h + acc_l;
        *psi_at(j) = S;
        publish(sbuf + ((j + 1) & 1) * 8 * kFragB);
    }
}

template <int STEPS>
int launch_scan(const PrefillParams& p, const StateGrid& sg, unsigned nblocks, hipStream_t stream, int steps) {
    if constexpr (STEPS < kMaxGroups) {
        if (steps == STEPS) {
            if (sg.plan)
                hipLaunchKernelGGL((gdn_prefill_scan_kernel<STEPS, true>), dim3(nblocks), dim3(512), 0, stream, p, sg);
            else
                hipLaunchKernelGGL((gdn_prefill_scan_kernel<STEPS, false>), dim3(nblocks), dim3(512), 0, stream, p, sg);
            return gdn_host::check_launch("gdn_prefill_scan_kernel");
        }
        return launch_scan<STEPS + 1>(p, sg, nblocks, stream, steps);
    } else {
        return gdn_host::fail(GDN_ERR_UNSUPPORTED, "prefill: %d chunk groups", steps + 1);
    }
}

// Chunk groups of packed sequences, balanced by length: the smallest group
// length L (at least 4 chunks) for which sum_i min(16, ceil(n_i / L)) groups
// fit `target` slots per head, n_i the chunks of sequence i (an empty
// sequence keeps one group, which passes its state through).  Every group of
// a sequence then has ceil(n_i / G_i) chunks (the last may have fewer), so the
// longest chain is about L wherever the long sequences sit, instead of the
// longest sequence over one group count shared by all.  One wave; writes the
// StateGrid::plan table.  Requires nseq <= target <= kPlanCap.
__global__ __launch_bounds__(64) void gdn_prefill_plan_kernel(const int32_t* __restrict__ cu, int nseq, int target,
                                                              int32_t* __restrict__ tab) {
    const int lane = threadIdx.x;
    auto nchunks = [&](int i) { return (cu[i + 1] - cu[i] + kC - 1) / kC; };
    auto gcount = [&](int n, int L) { return min(kMaxGroups, max(1, (n + L - 1) / L)); };
    // Chunk counts of sequences lane + 64 u (nseq <= target <= kPlanCap = 256).
    int nc[kPlanCap / 64];
    int nmax = 0;
#pragma unroll
    for (int u = 0; u < kPlanCap / 64; ++u) {
        const int i = lane + 64 * u;
        nc[u] = i < nseq ? nchunks(i) : -1;
        nmax = max(nmax, nc[u]);
    }
    for (int off = 32; off > 0; off >>= 1) nmax = max(nmax, __shfl_xor(nmax, off));
    auto total = [&](int L) {
        int t = 0;
#pragma unroll
        for (int u = 0; u < kPlanCap / 64; ++u) t += nc[u] >= 0 ? gcount(nc[u], L) : 0;
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off);
        return t;
    };
    int lo = 4, hi = max(4, nmax);  // total(hi) = nseq <= target
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (total(mid) <= target)
            hi = mid;
        else
            lo = mid + 1;
    }
    // Slots in sequence order: sequence i = lane + 64 u takes slots from the
    // sum of G over the sequences before it (exclusive wave scans per u).
    int base = 0, mbase = 0;
#pragma unroll
    for (int u = 0; u < kPlanCap / 64; ++u) {
        const int i = lane + 64 * u;
        const int G = nc[u] >= 0 ? gcount(nc[u], lo) : 0, M = G > 0 ? G - 1 : 0;
        int x = G, y = M;  // inclusive scans
        for (int off = 1; off < 64; off <<= 1) {
            const int xs = __shfl_up(x, off), ys = __shfl_up(y, off);
            if (lane >= off) {
                x += xs;
                y += ys;
            }
        }
        const int first = base + x - G, mfirst = mbase + y - M;
        if (i < nseq) {
            tab[2 + 2 * i] = G;
            tab[3 + 2 * i] = first;
            for (int g = 0; g < G; ++g) {
                tab[2 + 2 * nseq + first + g] = (i << 8) | g;
                if (g < M) tab[2 + 2 * nseq + kPlanCap + mfirst + g] = (i << 8) | g;
            }
        }
        base += __shfl(x, 63);
        mbase += __shfl(y, 63);
    }
    if (lane == 0) {
        tab[0] = base;
        tab[1] = mbase;
    }
}

// ---------------------------------------------------------------------------
// Zero fill used for the T == 0 state (a kernel rather than a memset node, so
// the call stays safe to capture in a HIP graph).
__global__ void gdn_fill_zero_kernel(float* __restrict__ p, size_t n) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        p[i] = 0.f;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
constexpr size_t kFragBytes = 64 * 16;  // one record fragment

size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

// How the state pass is split: NT 16-column tiles per wave; NW waves per
// workgroup; G chunk groups per sequence when (sequence, head) pairs alone
// cannot fill the chip (each group then runs its own chain of chunks, joined
// through the groups' affine maps).
struct StatePlan {
    int NT_out, NW_out, nvg_out, NT_map, NW_map, nvg_map, G;
    bool wide;  // dv % 128 == 0: gdn_prefill_state4_kernel (4 waves x 32 columns, 128 columns a workgroup)
    bool half;  // wide, output pass in 64-column workgroups (4 compute waves x 16): one group, few pairs
};

// `exact`: max_chunks is the exact chunk count of every sequence, so the
// group count is trimmed until no group is empty.  Workspace sizing uses the
// untrimmed count, which never decreases as sequences grow.
// `varlen`: packed sequences of unequal lengths.
StatePlan plan_state(long long nheads, int dv, long long max_chunks, bool exact, bool varlen) {
    StatePlan s;
    s.wide = dv % 128 == 0;
    s.half = false;
    if (s.wide) {
        s.NT_out = s.NT_map = 2;
        s.NW_out = s.NW_map = 4;
        s.nvg_out = dv / 128;
        s.nvg_map = (dv + kDK) / 128;
        // Chunk groups when the output pass alone would leave CUs idle: below
        // 256 output workgroups for packed sequences (groups also balance
        // their unequal lengths), below 128 for equal lengths (measured at
        // T = 8192: 128 (sequence, head) pairs run 1.2x faster as one group
        // each than as two, where the map pass and scan cost more than the
        // idle half of the chip).  Groups of at least 4 chunks; of 2 when
        // there are at most 16 (sequence, head) pairs and at most 16 chunks,
        // where the map pass's chain is most of the call (measured: B=1,
        // H=16, T=512 27.7 -> 23.9 us, T=1024 29.9 -> 28.4; H=4, T=900 34.6
        // -> 30.7; B=2, H=8, T=1024 30.1 -> 28.6; H=2, T=600 33.2 -> 27.4;
        // slower at 32 or more pairs, and at T=2048).
        const long long base = nheads * s.nvg_out;  // output-pass workgroups (one per CU) with one group
        long long G = 1;
        if (base < (varlen ? 256 : 128) && max_chunks >= 8) {
            const long long min_chunks = (!varlen && base <= 16 && max_chunks <= 16) ? 2 : 4;
            G = std::min<long long>(std::min<long long>(kMaxGroups, 256 / base), max_chunks / min_chunks);
        }
        if (exact && G > 1) G = (max_chunks + (max_chunks + G - 1) / G - 1) / ((max_chunks + G - 1) / G);
        s.G = G < 2 ? 1 : static_cast<int>(G);
        // At most half the CUs busy in the output pass (equal lengths, or
        // one group): split each head's 128 columns over two workgroups of
        // four 16-column compute waves (the state columns update
        // independently; the halves of a head share K and Q through the L2
        // of their XCD).  Packed sequences with planned groups keep whole
        // heads (their plan targets a full round of 128-column workgroups).
        s.half = (s.G == 1 || !varlen) && base * s.G <= 128;
        if (s.half) s.nvg_out = dv / 64;
        return s;
    }
    // dv not a multiple of 128: the 16-column state kernel.  Output pass:
    // 32-column waves where dv allows, as many waves (up to 4) as divide the
    // tiles.  Map pass (dv + 128 columns): two waves per SIMD (8-wave
    // workgroups of 32-column waves) where the tiling allows, so the waves
    // hide each other's LDS and copy latency; otherwise wider or fewer waves.
    s.NT_out = (dv % 32 == 0) ? 2 : 1;
    {
        const int tiles = dv / (16 * s.NT_out);
        s.NW_out = (tiles % 4 == 0) ? 4 : (tiles % 2 == 0) ? 2 : 1;
    }
    s.nvg_out = dv / (16 * s.NT_out * s.NW_out);
    if ((dv + kDK) % 256 == 0) {
        s.NT_map = 2;
        s.NW_map = 8;
        s.nvg_map = (dv + kDK) / 256;
    } else if ((dv + kDK) % 64 == 0 && (dv + kDK) / 64 <= 4) {
        // One workgroup of 64-column waves for all dv + 128 columns (dv = 64).
        s.NT_map = 4;
        s.NW_map = (dv + kDK) / 64;
        s.nvg_map = 1;
    } else {
        s.NT_map = (dv % 32 == 0) ? 2 : 1;
        const int mtiles = (dv + kDK) / (16 * s.NT_map);
        s.NW_map = (mtiles % 4 == 0) ? 4 : (mtiles % 2 == 0) ? 2 : 1;
        s.nvg_map = mtiles / s.NW_map;
    }
    const long long base = nheads * s.nvg_out;  // output-pass workgroups with one group
    long long G = 1;
    if (base < 256 && max_chunks >= 8)
        G = std::min<long long>(std::min<long long>(kMaxGroups, 256 / base), max_chunks / 4);
    if (exact && G > 1) G = (max_chunks + (max_chunks + G - 1) / G - 1) / ((max_chunks + G - 1) / G);
    s.G = G < 2 ? 1 : static_cast<int>(G);
    // A map pass that would fill at most half the CUs (few groups, e.g. G = 2
    // at 128 (sequence, head) pairs) splits each group's dv + 128 columns over
    // workgroups of 8 waves x 16 columns instead (psi and phi apart).
    if (s.G > 1 && s.NT_map == 2 && s.NW_map == 8 && nheads * (s.G - 1) * s.nvg_map * 2 <= 256) {
        s.NT_map = 1;
        s.nvg_map = (dv + kDK) / 128;
    }
    return s;
}

// The plan a launch runs: `s` (plan_state's, which sizes the workspace) or,
// where it is estimated to end sooner, every (sequence, head) as one chain of
// chunks with the output pass alone, its columns over one (full) or two (half)
// workgroups.  Estimates in us, fitted at H = 16: a chunk step of the output
// pass takes 2.9 full width and 1.46 half width, 1.75 with every CU busy; of
// the map pass 1.3 to 2.2 as its workgroups fill the 512 slots; a scan step
// 0.75; the two launches more and the passes' prologues 10 to 14 (20 with the
// device's plan).  A workgroup's own start and end take 3.  Where there are more
// workgroups than CUs the call ends after the longest one, or after the CUs'
// share of all workgroups and half the longest.  (Without their starts and ends
// in that share, packed sequences of a few chunks each ran half width, more
// workgroups than CUs, at 129 to 255 pairs: 12 of one token 14.6 us, full width
// 12.6; 20 of up to 130, H = 8, 19.6, 16.8.)  Over 200 packs of 129 to 700 full-width
// workgroups, H = 4 to 32, the choice between the widths is within 3% of the better
// one for 193 (169 so), 9% from it at worst (22%).  Against groups wherever
// plan_state has them, 244 shapes of equal lengths (H = 1 to 32, B = 1 to 16, T = 192
// to 8192, dv = 64 to 256) take 0.71 to 1.03 of the time.
// State phase at B = 4, T = 1024 37.0 -> 26.4 us, T = 2048 55.6 -> 49.0, T = 4096
// 96.0 -> 94.3 and at B = 1, T = 512 17.5 -> 14.2; grouped stays at B = 1, T = 1024
// (21.6 against 25.1) and T = 8192 (65 against 184).  Packed calls: 8 sequences of 709
// to 4688 tokens 196 -> 168 us, 8 x 3000 176 -> 129, 11 of 8 to 5013 205 -> 168;
// 6 + 2690 + 7579 stays grouped (113 against 196).
// `total_chunks`: of all sequences (estimated for packed ones).
StatePlan choose_plan(const StatePlan& s, long long nheads, int H, int dv, long long max_chunks,
                      long long total_chunks, bool varlen) {
    if (!s.wide) return s;
    constexpr double kCUs = 256, kFull = 2.9, kHalf = 1.46, kHalfBusy = 1.75;
    const int nvg = dv / 128;
    const long long base = nheads * nvg;  // output-pass workgroups, full width, one group
    const double C = static_cast<double>(max_chunks);
    const double steps = static_cast<double>(total_chunks) * H * nvg;  // full-width chunk steps in all
    auto ends = [&](double wgs, double all, double step) {
        const double longest = 3 + step * C;
        return wgs <= kCUs ? longest : std::max(longest, (3 * wgs + step * all) / kCUs + longest / 2);
    };
    const double full = ends(static_cast<double>(base), steps, kFull);
    const double half = ends(2.0 * base, 2 * steps, 2 * base > kCUs / 2 ? kHalfBusy : kHalf);
    StatePlan one = s;
    one.G = 1;
    one.half = varlen ? half < 0.95 * full : base <= 128;
    one.nvg_out = one.half ? dv / 64 : nvg;
    if (s.G > 1) {
        double glen, G = s.G, fixed;
        if (varlen) {  // the device's plan: at most `target` groups a head
            const double target = kCUs / (H * nvg), nseq = static_cast<double>(nheads) / H;
            glen = std::min(C, std::ceil(static_cast<double>(total_chunks) / (target - nseq / 2)));
            G = std::ceil(C / glen);
            fixed = 20;
        } else {
            glen = static_cast<double>((max_chunks + s.G - 1) / s.G);
            fixed = s.half ? 10 : 14;
        }
        const double map_wgs = static_cast<double>(nheads) * (G - 1) * s.nvg_map;
        const double map = 1.3 + 0.9 * std::min(1.0, map_wgs / 512);
        const double grouped = fixed + glen * ((s.half ? kHalf : kFull) + map) + 0.75 * (G - 1);
        if (grouped < (one.half ? half : full)) return s;
    }
    return one;
}

// Record length: the 32-column state kernel forms Aq itself.
int rec_frags(const StatePlan& sp) { return sp.wide ? kRecShort : kRecFull; }

struct WsLayout {
    size_t offR, offPsi, offPhi, offPlan, total;
};

// Packed sequences with chunk groups plan them per sequence on the device
// (gdn_prefill_plan_kernel): target slots per head, at most 256 / (H nvg_out)
// (one round of the output pass), which also bounds the group maps.
bool planned_groups(const StatePlan& sp, bool varlen) { return varlen && sp.G > 1; }
int plan_target(const StatePlan& sp, int H) { return std::max(1, 256 / (H * sp.nvg_out)); }

WsLayout ws_layout(long long slots, int H, long long nheads, int dv, const StatePlan& sp, bool varlen, int nseq) {
    const size_t ch = static_cast<size_t>(slots) * H;
    const bool planned = planned_groups(sp, varlen);
    WsLayout L;
    L.offR = 0;
    L.offPsi = align256(L.offR + ch * rec_frags(sp) * kFragBytes);
    const size_t units = planned      ? static_cast<size_t>(H) * plan_target(sp, H)
                         : sp.G > 1 ? static_cast<size_t>(nheads) * sp.G
                                    : 0;
    L.offPhi = align256(L.offPsi + units * kDK * dv * 4);
    L.offPlan = align256(L.offPhi + units * kDK * kDK * 2);
    L.total = align256(L.offPlan + (planned ? (2 + 2 * static_cast<size_t>(nseq) + 2 * kPlanCap) * 4 : 0));
    return L;
}

int check_common(const char* who, int H, int dk, int dv) {
    using gdn_host::fail;
    if (H <= 0) return fail(GDN_ERR_INVALID_ARGUMENT, "%s: H=%d", who, H);
    if (dk != kDK) return fail(GDN_ERR_UNSUPPORTED, "%s: dk=%d, only dk=128 is built", who, dk);
    if (dv < 16 || dv > 512 || dv % 16 != 0)
        return fail(GDN_ERR_UNSUPPORTED, "%s: dv=%d must be a multiple of 16 in [16, 512]", who, dv);
    return GDN_OK;
}

template <int MODE, int NT>
int launch_state4(const PrefillParams& p, const StateGrid& sg, hipStream_t stream) {
    const long long nwg = static_cast<long long>(sg.nheads) * sg.ngroups_run * sg.nvg;
    if (nwg > 0x7fffffffLL) return gdn_host::fail(GDN_ERR_UNSUPPORTED, "prefill: grid too large");
    hipLaunchKernelGGL((gdn_prefill_state4_kernel<MODE, NT>), dim3(static_cast<unsigned>(nwg)),
                       dim3(64 * Stage4<MODE, NT>::nWaves), 0, stream, p, sg);
    return gdn_host::check_launch(MODE == kModeMap ? "gdn_prefill_state4_kernel<map>" : "gdn_prefill_state4_kernel");
}

template <int MODE>
int launch_state_plan(const PrefillParams& p, const StateGrid& sg, const StatePlan& sp, hipStream_t stream);

template <int MODE, int NT>
int launch_state(const PrefillParams& p, const StateGrid& sg, int NW, hipStream_t stream) {
    const long long nwg = static_cast<long long>(sg.nheads) * sg.ngroups_run * sg.nvg;
    if (nwg > 0x7fffffffLL) return gdn_host::fail(GDN_ERR_UNSUPPORTED, "prefill: grid too large");
    const dim3 grid(static_cast<unsigned>(nwg));
    switch (NW) {
        case 1: hipLaunchKernelGGL((gdn_prefill_state_kernel<MODE, 1, NT>), grid, dim3(64), 0, stream, p, sg); break;
        case 2: hipLaunchKernelGGL((gdn_prefill_state_kernel<MODE, 2, NT>), grid, dim3(128), 0, stream, p, sg); break;
        case 4: hipLaunchKernelGGL((gdn_prefill_state_kernel<MODE, 4, NT>), grid, dim3(256), 0, stream, p, sg); break;
        case 3:
            if constexpr (MODE == kModeMap && NT == 4) {
                hipLaunchKernelGGL((gdn_prefill_state_kernel<MODE, 3, NT>), grid, dim3(192), 0, stream, p, sg);
                break;
            }
            return gdn_host::fail(GDN_ERR_UNSUPPORTED, "prefill: no state kernel for %d waves", NW);
        case 8:
            if constexpr (MODE == kModeMap && NT <= 2) {
                hipLaunchKernelGGL((gdn_prefill_state_kernel<MODE, 8, NT>), grid, dim3(512), 0, stream, p, sg);
                break;
            }
            return gdn_host::fail(GDN_ERR_UNSUPPORTED, "prefill: no state kernel for %d waves", NW);
        default:
            return gdn_host::fail(GDN_ERR_UNSUPPORTED, "prefill: no state kernel for %d waves", NW);
    }
    return gdn_host::check_launch(MODE == kModeMap ? "gdn_prefill_state_kernel<map>" : "gdn_prefill_state_kernel");
}

template <int MODE>
int launch_state_plan(const PrefillParams& p, const StateGrid& sg, const StatePlan& sp, hipStream_t stream) {
    if (sp.wide) {
        if constexpr (MODE == kModeOut)
            if (sp.half) return launch_state4<MODE, 1>(p, sg, stream);
        return launch_state4<MODE, 2>(p, sg, stream);
    }
    if (MODE == kModeMap)
        return sp.NT_map == 4   ? launch_state<MODE, 4>(p, sg, sp.NW_map, stream)
               : sp.NT_map == 2 ? launch_state<MODE, 2>(p, sg, sp.NW_map, stream)
                                : launch_state<MODE, 1>(p, sg, sp.NW_map, stream);
    return sp.NT_out == 2 ? launch_state<MODE, 2>(p, sg, sp.NW_out, stream)
                          : launch_state<MODE, 1>(p, sg, sp.NW_out, stream);
}

// phases: bit 0 = chunk-parallel intra kernel, bit 1 = state pass (map pass
// and scan when chunk groups are used, then the output pass).
// total_chunks: chunks of all sequences (an estimate for packed ones).
int launch(PrefillParams& p, int nseq, int nchunk_grid, long long total_chunks, bool exact, void* workspace,
           size_t ws_bytes, long long slots, hipStream_t stream, int phases) {
    using gdn_host::fail;
    const long long nheads = static_cast<long long>(nseq) * p.H;
    const bool varlen = p.cu != nullptr;
    const StatePlan sized = plan_state(nheads, p.dv, nchunk_grid, exact, varlen);
    const size_t need = ws_layout(slots, p.H, nheads, p.dv, sized, varlen, nseq).total;
    const StatePlan sp = choose_plan(sized, nheads, p.H, p.dv, nchunk_grid, total_chunks, varlen);
    const WsLayout L = ws_layout(slots, p.H, nheads, p.dv, sp, varlen, nseq);
    if (!workspace || ws_bytes < need)
        return fail(GDN_ERR_WORKSPACE, "prefill: workspace of %zu bytes given, %zu needed", ws_bytes, need);
    if (!gdn_host::aligned(workspace, 256))
        return fail(GDN_ERR_INVALID_ARGUMENT, "prefill: workspace must be 256-byte aligned");
    char* ws = static_cast<char*>(workspace);
    p.wsR = reinterpret_cast<u32x4*>(ws + L.offR);
    p.nseq = nseq;
    p.xcd_heads = (nheads % 8 == 0) ? 1 : 0;
    if ((phases & 1) && nchunk_grid > 0) {
        // One wave per (sequence, head) chunk.  Packed sequences: the longest
        // one's chunks of each where those are no more than the chunk slots,
        // which hold up to num_seqs empty ones a head and take a search (32
        // sequences of up to 64 tokens, H = 16: dv = 64 26.0 us a call by slots,
        // 24.3 so; dv = 128 23.5, 21.8).
        PrefillParams pi = p;
        const long long heads = varlen ? p.H : nheads;
        const long long each = static_cast<long long>(nseq) * nchunk_grid;
        const bool by_chunk = !varlen || each <= slots - 1;
        const long long items = !varlen ? nchunk_grid : by_chunk ? each : slots - 1;
        if (heads * items > 0x7fffffffLL) return fail(GDN_ERR_UNSUPPORTED, "prefill: grid too large");
        pi.intra_items = static_cast<int>(items);
        pi.intra_chunks = varlen && by_chunk ? nchunk_grid : 0;
        pi.xcd_heads = heads % 8 == 0 ? 1 : 0;
        const dim3 grid(static_cast<unsigned>(heads * items));
        if (sp.wide)
            hipLaunchKernelGGL(gdn_prefill_intra_kernel<false>, grid, dim3(64), 0, stream, pi);
        else
            hipLaunchKernelGGL(gdn_prefill_intra_kernel<true>, grid, dim3(64), 0, stream, pi);
        const int st = gdn_host::check_launch("gdn_prefill_intra_kernel");
        if (st != GDN_OK) return st;
    }
    if (!(phases & 2)) return GDN_OK;
    StateGrid sg = {};
    sg.ngroups = sp.G;
    sg.nheads = static_cast<int>(nheads);
    sg.psi = reinterpret_cast<float*>(ws + L.offPsi);
    sg.phi = reinterpret_cast<uint16_t*>(ws + L.offPhi);
    sg.nseq = nseq;
    int st;
    if (planned_groups(sp, varlen)) {
        // Per-sequence group counts, planned on the device from cu_seqlens.
        const int target = plan_target(sp, p.H);
        if (target > kPlanCap || nseq > target) return fail(GDN_ERR_UNSUPPORTED, "prefill: group plan");
        int32_t* tab = reinterpret_cast<int32_t*>(ws + L.offPlan);
        hipLaunchKernelGGL(gdn_prefill_plan_kernel, dim3(1), dim3(64), 0, stream, p.cu, nseq, target, tab);
        st = gdn_host::check_launch("gdn_prefill_plan_kernel");
        if (st != GDN_OK) return st;
        sg.plan = tab;
        const int map_cap = target - nseq;  // sum of G_i - 1
        if (map_cap > 0) {
            StateGrid sm = sg;
            sm.nheads = p.H;  // grid: (head, map slot, column part)
            sm.nvg = sp.nvg_map;
            sm.ngroups_run = map_cap;
            st = launch_state_plan<kModeMap>(p, sm, sp, stream);
            if (st != GDN_OK) return st;
            const long long nscan = nheads * (p.dv / 16);
            if (nscan > 0x7fffffffLL) return fail(GDN_ERR_UNSUPPORTED, "prefill: grid too large");
            st = launch_scan<1>(p, sg, static_cast<unsigned>(nscan), stream, std::min(kMaxGroups - 1, map_cap));
            if (st != GDN_OK) return st;
        }
        StateGrid so = sg;
        so.nheads = p.H;  // grid: (head, slot, column part)
        so.nvg = sp.nvg_out;
        so.ngroups_run = target;
        return launch_state_plan<kModeOut>(p, so, sp, stream);
    }
    if (sp.G > 1) {
        sg.nvg = sp.nvg_map;
        sg.ngroups_run = sp.G - 1;
        st = launch_state_plan<kModeMap>(p, sg, sp, stream);
        if (st != GDN_OK) return st;
        const long long nscan = nheads * (p.dv / 16);
        if (nscan > 0x7fffffffLL) return fail(GDN_ERR_UNSUPPORTED, "prefill: grid too large");
        st = launch_scan<1>(p, sg, static_cast<unsigned>(nscan), stream, sp.G - 1);
        if (st != GDN_OK) return st;
    }
    sg.nvg = sp.nvg_out;
    sg.ngroups_run = sp.G;
    return launch_state_plan<kModeOut>(p, sg, sp, stream);
}

}  // namespace

extern "C" {

size_t gdn_prefill_workspace_bytes(int B, int H, int T, int dk, int dv) {
    (void)dk;
    if (B <= 0 || H <= 0 || T <= 0 || dv <= 0) return 0;
    const long long nch = (T + kC - 1) / kC;
    const long long slots = static_cast<long long>(B) * nch;
    const long long nheads = static_cast<long long>(B) * H;
    return ws_layout(slots, H, nheads, dv, plan_state(nheads, dv, nch, false, false), false, B).total;
}

size_t gdn_prefill_varlen_workspace_bytes(int num_seqs, int H, int T_total, int dk, int dv) {
    (void)dk;
    if (num_seqs <= 0 || H <= 0 || T_total < 0 || dv <= 0) return 0;
    const long long slots = static_cast<long long>(T_total) / kC + num_seqs + 1;
    const long long nheads = static_cast<long long>(num_seqs) * H;
    // Whether chunk groups are used only grows with the longest sequence: size
    // for T_total (the per-sequence plan then fits in H x 256 / (H nvg) maps).
    return ws_layout(slots, H, nheads, dv, plan_state(nheads, dv, (T_total + kC - 1) / kC, false, true), true, num_seqs)
        .total;
}

}  // extern "C"

namespace {

int prefill_batch(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                  const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                  const float* state_in, float scale, gdn_bf16_t* out, float* state_out, int B, int H, int T,
                  int dk, int dv, void* workspace, size_t workspace_bytes, void* stream, int phases,
                  int out_tm = 0) {
    using gdn_host::aligned;
    using gdn_host::fail;
    int st = check_common("prefill", H, dk, dv);
    if (st != GDN_OK) return st;
    if (B < 0 || T < 0) return fail(GDN_ERR_INVALID_ARGUMENT, "prefill: B=%d T=%d", B, T);
    if (B == 0) return GDN_OK;
    if (!q || !k || !v || !A_log || !a || !b_logits || !state_out || (T > 0 && !out))
        return fail(GDN_ERR_INVALID_ARGUMENT, "prefill: null pointer argument");
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || (out && !aligned(out, 16)) ||
        !aligned(state_out, 4) || (state_in && !aligned(state_in, 4)))
        return fail(GDN_ERR_INVALID_ARGUMENT, "prefill: q/k/v/out need 16-byte alignment");
    if (static_cast<long long>(B) * H * T * dv >= (1LL << 40))
        return fail(GDN_ERR_UNSUPPORTED, "prefill: problem too large");
    PrefillParams p = {};
    p.q = q;
    p.k = k;
    p.v = v;
    p.a = a;
    p.b = b_logits;
    p.A_log = A_log;
    p.mask = mask;
    p.state_in = state_in;
    p.out = out;
    p.state_out = state_out;
    p.cu = nullptr;
    p.out_tm = out_tm;
    p.dt_bias = dt_bias;
    p.scale = scale == 0.f ? 1.f / sqrtf(static_cast<float>(dk)) : scale;
    p.H = H;
    p.dv = dv;
    p.T_stride = T;
    p.T_len = T;
    p.chunks_per_seq = (T + kC - 1) / kC;
    const long long slots = static_cast<long long>(B) * p.chunks_per_seq;
    if (slots == 0) {
        // T == 0: the state passes through unchanged.
        if (!(phases & 2)) return GDN_OK;
        if (state_in)
            return hipMemcpyAsync(state_out, state_in, static_cast<size_t>(B) * H * dk * dv * 4,
                                  hipMemcpyDeviceToDevice, static_cast<hipStream_t>(stream)) == hipSuccess
                       ? GDN_OK
                       : fail(GDN_ERR_HIP, "prefill: state copy failed");
        hipLaunchKernelGGL(gdn_fill_zero_kernel, dim3(1024), dim3(256), 0, static_cast<hipStream_t>(stream),
                           state_out, static_cast<size_t>(B) * H * dk * dv);
        return gdn_host::check_launch("gdn_fill_zero_kernel");
    }
    return launch(p, B, p.chunks_per_seq, slots, true, workspace, workspace_bytes, slots, static_cast<hipStream_t>(stream),
                  phases);
}

}  // namespace

extern "C" {

int gdn_prefill_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                    const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                    const float* state_in, float scale, gdn_bf16_t* out, float* state_out, int B, int H,
                    int T, int dk, int dv, void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_batch(q, k, v, A_log, a, dt_bias, b_logits, mask, state_in, scale, out, state_out, B, H, T, dk,
                         dv, workspace, workspace_bytes, stream, 3);
}

int gdn_prefill_tm_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                       const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                       const float* state_in, float scale, gdn_bf16_t* out, float* state_out, int B, int H,
                       int T, int dk, int dv, void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_batch(q, k, v, A_log, a, dt_bias, b_logits, mask, state_in, scale, out, state_out, B, H, T, dk,
                         dv, workspace, workspace_bytes, stream, 3, 1);
}

int gdn_prefill_intra_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                          const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                          const float* state_in, float scale, gdn_bf16_t* out, float* state_out, int B, int H,
                          int T, int dk, int dv, void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_batch(q, k, v, A_log, a, dt_bias, b_logits, mask, state_in, scale, out, state_out, B, H, T, dk,
                         dv, workspace, workspace_bytes, stream, 1);
}

int gdn_prefill_state_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                          const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                          const float* state_in, float scale, gdn_bf16_t* out, float* state_out, int B, int H,
                          int T, int dk, int dv, void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_batch(q, k, v, A_log, a, dt_bias, b_logits, mask, state_in, scale, out, state_out, B, H, T, dk,
                         dv, workspace, workspace_bytes, stream, 2);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// No-allocation prefill: the workspace is a static device array, one copy per
// GPU (each device that loads this code object holds it until the process
// ends).  Its device address is looked up once per device, with that device
// current, on the first call there; host code uses only that address (the
// array's own name is a host-side stand-in, not a device pointer); the
// stream must belong to the current device.  Nothing in
// the workspace has to start zeroed: every chunk slot and group map that a
// kernel reads was written earlier in the same call.  Calls that overlap on
// one GPU (e.g. on two streams) share the array and race.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kScratchBytes = static_cast<size_t>(GDN_PREFILL_NOALLOC_MAX_BYTES);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
// Device address of `scratch` per device, set once a lookup has succeeded (a
// failed lookup is not cached: the next call on that device tries again).
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {};

// `scratch`'s address on the current device `dev`, or null with *err set.
void* scratch_ptr(int dev, hipError_t* err) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* ptr = nullptr;
        *err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (*err != hipSuccess) return nullptr;
        g_scratch[dev] = ptr;
    }
    return g_scratch[dev];
}

}  // namespace

extern "C" {

int gdn_prefill_noalloc_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                            const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                            const float* state_in, float scale, gdn_bf16_t* out, float* state_out, int B, int H,
                            int T, int dk, int dv, void* stream) {
    using gdn_host::fail;
    // Sizes first: a request that cannot fit is refused before any HIP call.
    const int st = check_common("prefill_noalloc", H, dk, dv);
    if (st != GDN_OK) return st;
    if (B < 0 || T < 0) return fail(GDN_ERR_INVALID_ARGUMENT, "prefill_noalloc: B=%d T=%d", B, T);
    const size_t need = gdn_prefill_workspace_bytes(B, H, T, dk, dv);
    if (need > kScratchBytes)
        return fail(GDN_ERR_WORKSPACE,
                    "prefill_noalloc: B=%d H=%d T=%d dv=%d needs %zu bytes of scratch, the static buffer holds %zu "
                    "(use gdn_prefill_hip with a caller workspace)",
                    B, H, T, dv, need, kScratchBytes);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail(GDN_ERR_HIP, "prefill_noalloc: hipGetDevice failed");
    if (dev < 0 || dev >= kMaxDevices) return fail(GDN_ERR_UNSUPPORTED, "prefill_noalloc: device %d", dev);
    // The buffer is the current device's: a stream of another device would
    // run the kernels there against this device's address.
    if (stream) {
        int sdev = -1;
        if (hipStreamGetDevice(static_cast<hipStream_t>(stream), &sdev) != hipSuccess)
            return fail(GDN_ERR_HIP, "prefill_noalloc: hipStreamGetDevice failed");
        if (sdev != dev)
            return fail(GDN_ERR_INVALID_ARGUMENT, "prefill_noalloc: stream is on device %d, the current device is %d",
                        sdev, dev);
    }
    hipError_t err = hipSuccess;
    void* const ws = scratch_ptr(dev, &err);
    if (!ws) return fail(GDN_ERR_HIP, "prefill_noalloc: scratch address lookup failed: %s", hipGetErrorString(err));
    return prefill_batch(q, k, v, A_log, a, dt_bias, b_logits, mask, state_in, scale, out, state_out, B, H, T, dk,
                         dv, ws, kScratchBytes, stream, 3);
}

}  // extern "C"

namespace {

int prefill_varlen(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                   const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                   const int32_t* cu_seqlens, int num_seqs, int max_seqlen, const float* state_in, float scale,
                   gdn_bf16_t* out, float* state_out, int H, int T_total, int dk, int dv, void* workspace,
                   size_t workspace_bytes, void* stream, int out_tm) {
    using gdn_host::aligned;
    using gdn_host::fail;
    int st = check_common("prefill_varlen", H, dk, dv);
    if (st != GDN_OK) return st;
    if (num_seqs < 0 || T_total < 0)
        return fail(GDN_ERR_INVALID_ARGUMENT, "prefill_varlen: num_seqs=%d T_total=%d", num_seqs, T_total);
    if (num_seqs == 0) return GDN_OK;
    if (!q || !k || !v || !A_log || !a || !b_logits || !cu_seqlens || !state_out || (T_total > 0 && !out))
        return fail(GDN_ERR_INVALID_ARGUMENT, "prefill_varlen: null pointer argument");
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || (out && !aligned(out, 16)))
        return fail(GDN_ERR_INVALID_ARGUMENT, "prefill_varlen: q/k/v/out need 16-byte alignment");
    if (static_cast<long long>(H) * T_total * dv >= (1LL << 40))
        return fail(GDN_ERR_UNSUPPORTED, "prefill_varlen: problem too large");
    PrefillParams p = {};
    p.q = q;
    p.k = k;
    p.v = v;
    p.a = a;
    p.b = b_logits;
    p.A_log = A_log;
    p.mask = mask;
    p.state_in = state_in;
    p.out = out;
    p.state_out = state_out;
    p.cu = cu_seqlens;
    p.out_tm = out_tm;
    p.dt_bias = dt_bias;
    p.scale = scale == 0.f ? 1.f / sqrtf(static_cast<float>(dk)) : scale;
    p.H = H;
    p.dv = dv;
    p.T_stride = T_total;
    p.T_len = 0;
    p.chunks_per_seq = 0;
    const int maxlen = (max_seqlen > 0 && max_seqlen < T_total) ? max_seqlen : T_total;
    const int nchunk_grid = (maxlen + kC - 1) / kC;
    const long long slots = static_cast<long long>(T_total) / kC + num_seqs + 1;
    const long long total_chunks = static_cast<long long>(T_total) / kC + (num_seqs + 1) / 2;
    return launch(p, num_seqs, nchunk_grid, total_chunks, false, workspace, workspace_bytes, slots,
                  static_cast<hipStream_t>(stream), 3);
}

}  // namespace

extern "C" {

int gdn_prefill_varlen_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                           const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                           const int32_t* cu_seqlens, int num_seqs, int max_seqlen, const float* state_in,
                           float scale, gdn_bf16_t* out, float* state_out, int H, int T_total, int dk, int dv,
                           void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_varlen(q, k, v, A_log, a, dt_bias, b_logits, mask, cu_seqlens, num_seqs, max_seqlen, state_in,
                          scale, out, state_out, H, T_total, dk, dv, workspace, workspace_bytes, stream, 0);
}

int gdn_prefill_varlen_tm_hip(const gdn_bf16_t* q, const gdn_bf16_t* k, const gdn_bf16_t* v, const float* A_log,
                              const gdn_bf16_t* a, float dt_bias, const gdn_bf16_t* b_logits, const float* mask,
                              const int32_t* cu_seqlens, int num_seqs, int max_seqlen, const float* state_in,
                              float scale, gdn_bf16_t* out, float* state_out, int H, int T_total, int dk, int dv,
                              void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_varlen(q, k, v, A_log, a, dt_bias, b_logits, mask, cu_seqlens, num_seqs, max_seqlen, state_in,
                          scale, out, state_out, H, T_total, dk, dv, workspace, workspace_bytes, stream, 1);
}

}  // extern "C"
