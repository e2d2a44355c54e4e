// prompt_gemm.hip -- the GEMMs of prompt chunks and ragged batches,
// Y[n, m] = sum_k W[m, k] X[n, k]: a tiled one, and one for up to 64 rows.
//
// A prompt's tokens (crates/atlas-model/src/lib.rs:1612-1618 feeds them one by
// one) go through a layer together, so every weight read feeds N rows and the
// work is a contraction on the matrix cores: v_mfma_f32_16x16x32_bf16 with the
// f32 activations split into a bf16 "hi" (truncation) and "lo" (RNE of the
// exact remainder) part, two MFMAs per product, f32 sums (~2^-16 relative; the
// recipe of the 2..16-row kernels).
//
// MFMA operands (lane = 16 g + i): A = activations, lane (g, i) has k = 8g ..
// 8g+7 of row i of a 16-row tile; B = weights, the same k of weight row i, as
// stored (bf16) or made bf16 exactly (int8 q; int4 16 q, see below); D: lane
// (g, i) has rows 4g .. 4g+3 of weight row i.
//
// What bounds it: with N in the hundreds the matrix cores (a bare loop of these
// MFMAs on random operands runs at 1.9-2.0 PFLOP/s of the 2.5 on this card, its
// clock falling under the load), up to ~100 rows the weights' stream.  So:
//  * Tiles of 256, 192 or 128 weight rows x 128 (or 64) activation rows.  Eight
//    waves, two per SIMD, so that one wave's LDS reads and conversions run
//    behind the other's MFMAs; a wave owns 4..8 weight tiles x 2 activation
//    tiles.  (One wave per SIMD with 128 x 64 each reads a third less LDS but
//    stalls on every barrier: 12288 x 4096 at 1024 rows 246 against 212 us.)
//  * Everything reaches LDS by direct loads (16 bytes per lane), raw: weights as
//    stored in units of one 128-byte line per row (2 k steps of bf16, 4 of int8;
//    4 of int4, 64 bytes), activations in f32, 128 bytes per row and k step.  Two
//    rings (2-3 units, 4-5 steps), refilled right after a barrier, keep 2-4 steps
//    in flight; a barrier waits only for the loads that the next step reads.
//    Lines loaded in halves (64-byte rows) cost 6% more.
//  * Fragments are read one step ahead, into the registers that the MFMAs have
//    just used; the split of an activation tile and the conversion of the next
//    weights sit between the MFMAs.  Each instance fits 256 registers: beyond
//    that the compiler moves accumulators to and fro (1.4x slower).
//  * 16-byte chunk c of row r sits in LDS slot c ^ (r & 7) (the loads permute
//    their global addresses), so that fragment reads hit distinct banks.
//  * The blocks of one weight tile run side by side on one XCD (its L2 then
//    serves the weights to all but the first).
//  * int4: the nibbles become 16 q exactly (each at the top of a byte, converted
//    as int8 is), a step's products start from zero and are multiplied by the
//    block's scale (K % 32 == 0: a step is within one block), the 1/16 by the
//    epilogue.  (Masks alone give q + 24, whose -24 sum(x) has to be taken off
//    again: nothing faster, 505 against 514 us at 22016 x 4096 and 1001 rows and
//    310 against 288 at 12288 x 4096, but the larger sums cost every other element
//    of a row with an outlier its low bits.  The sums of 16 q x fit f32 for |x| up
//    to 8e34.)
//
// Measured (us; 7B shapes, the same weights call after call, against the
// one-launch-per-128-rows kernel before it):
//   1024 rows          bf16          int8          int4
//   22016 x 4096       595 -> 335    613 -> 409    1158 -> 526    (+ SwiGLU)
//   12288 x 4096       431 -> 191    450 -> 235     821 -> 309
//   4096 x 4096        201 ->  75    214 ->  93     270 -> 113
//   4096 x 11008       342 -> 175    357 -> 211     482 -> 263
//   127 rows
//   22016 x 4096        75 ->  56     77 ->  66     143 ->  88
//   12288 x 4096        55 ->  37     57 ->  41     102 ->  52
//   4096 x 4096         25 ->  22     27 ->  20      34 ->  24
//   4096 x 11008        43 ->  36     45 ->  36      59 ->  43
// Counters at 1024 rows (22016 x 4096; SIMD cycles): MFMAs 47% of them in bf16,
// 36 in int8, 27 in int4; vector instructions (4 cycles each) 38, 55 and 63: two
// MFMAs per product bound bf16, making the weights bf16 the other two.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemv.hpp"
#include "mfma.hpp"

namespace atlas {

// 16 (or 4) bytes per lane from global memory straight into LDS: lane l's
// bytes land at lds + l * VW (lds, soff wave-uniform)
template <int VW>
__device__ __forceinline__ void load_lds(__amdgpu_buffer_rsrc_t src, uint32_t voff, uint32_t soff, void* lds) {
    const auto dst = (__attribute__((address_space(3))) void*)lds;
    if constexpr (VW == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(src, dst, 16, voff, soff, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(src, dst, 4, voff, soff, 0, 0);
}

// all but this wave's newest N loads have landed; then the block meets
template <int N>
__device__ __forceinline__ void sync_stage() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(N) : "memory");
}

constexpr float kI4Unit = 16.0f;

template <int FMT>
using PgRaw = std::conditional_t<FMT == WF_BF16, u32x4, std::conditional_t<FMT == WF_I8, u32x2, uint32_t>>;

// the bf16 parts of 8 activations.
// NS = 2: hi (truncation) and the rounded remainder; NS = 3: two truncations and
// the rest, x exactly (8 + 8 + 8 bits).
// The matrix cores round an f32 sum down, which shifts every result by about
// -1e-7 of their size: little beside the 5e-6 of two parts, but at three the
// same in every row, so that it adds up through a model (3.3e-6 of a 1000-token
// prompt's logits against 1.5e-6).  So with three parts every other k step
// multiplies -x and its sum is subtracted (flip, the sign bit): what one rounds
// down the next rounds up.
template <int NS>
__device__ __forceinline__ void pg_split(const f32x4 p, const f32x4 q, uint32_t flip, bf16x8 (&part)[NS]) {
    float e[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
    if constexpr (NS == 3)
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = __uint_as_float(__float_as_uint(e[i]) ^ flip);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        u32x4 h;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            h[i] = s + 1 < NS ? bf16_hi2(e[2 * i], e[2 * i + 1]) : bf16_rne2(e[2 * i], e[2 * i + 1]);
        if (s + 1 < NS)
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] -= __uint_as_float(__float_as_uint(e[i]) & 0xFFFF0000u);
        part[s] = __builtin_bit_cast(bf16x8, h);
    }
}

// 8 weights as a bf16 operand (int4: times kI4Unit)
template <int FMT>
__device__ __forceinline__ bf16x8 pg_operand(const PgRaw<FMT> v) {
    u32x4 b;
    if constexpr (FMT == WF_BF16) {
        b = v;
    } else if constexpr (FMT == WF_I8) {
        b = u32x4{pack_f32_pair(s8_at(v.x, 0), s8_at(v.x, 1)), pack_f32_pair(s8_at(v.x, 2), s8_at(v.x, 3)),
                  pack_f32_pair(s8_at(v.y, 0), s8_at(v.y, 1)), pack_f32_pair(s8_at(v.y, 2), s8_at(v.y, 3))};
    } else {
        // element 2b in the high nibble of byte b: each nibble at the top of a
        // byte is 16 q there
        const uint32_t h = v & 0xF0F0F0F0u, l = (v << 4) & 0xF0F0F0F0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = pack_f32_pair(s8_at(h, i), s8_at(l, i));
    }
    return __builtin_bit_cast(bf16x8, b);
}

// SwiGLU of one D tile: rows (2i, 2i+1) = (gate_i, up_i) sit in adjacent lanes;
// the even lane finishes activation rows nb, nb + 1 of both, the odd one the
// other two
__device__ __forceinline__ void pg_store_swiglu(const GemvArgs& a, const f32x4 v, int m, int nb) {
    const bool odd = m & 1;
    float* y = a.y + (long)(m >> 1) * a.y_stride_m;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float mine0 = v[r], mine1 = v[r + 2];
        const float give = odd ? mine0 : mine1;
        const float got = __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(give), 0xB1, 0xF, 0xF, false));
        const float gate = odd ? got : mine0, up = odd ? mine1 : got;
        const int n = nb + r + (odd ? 2 : 0);
        if (n < a.N && m < a.M) y[n * a.y_stride_n] = gate / (1.0f + expf(-gate)) * up;
    }
}

template <int FMT, int WM, int WN, int MF, int NF, int VW>
struct PgShape {
    static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
    static constexpr int BM = WM * MF * 16, BN = WN * NF * 16;
    static constexpr int KU = FMT == WF_BF16 ? 2 : 4;                // k steps per weight unit
    static constexpr int WR = FMT == WF_BF16 ? 3 : 2;                // weight units in the ring
    static constexpr bool W_FIRST = WR == 2;                         // the next unit is due within the unit
    static constexpr int XR = FMT == WF_BF16 ? 4 : 5;                // activation steps in the ring
    static constexpr int RB = FMT == WF_BF16 ? 128 : FMT == WF_I8 ? 128 : 64;   // bytes of a weight row per unit
    static constexpr int CH = RB / 16;                               // 16-byte chunks of it
    static constexpr int W_BYTES = BM * RB, X_BYTES = BN * 128;
    static constexpr int S_BYTES = FMT == WF_I4 ? BM * 16 : 0;       // int4 scales of a unit (one per step)
    static constexpr int W_LD = (W_BYTES / (64 * VW) + WAVES - 1) / WAVES;     // loads per wave
    static constexpr int X_LD = (X_BYTES / 1024 + WAVES - 1) / WAVES;
    static constexpr int S_LD = FMT == WF_I4 ? (S_BYTES / 256 + WAVES - 1) / WAVES : 0;
    static constexpr int U_LD = W_LD + S_LD, U_BYTES = W_BYTES + S_BYTES;
    static constexpr int X_OFS = WR * U_BYTES;
    static constexpr int BYTES = X_OFS + XR * X_BYTES;
};

template <int FMT, int WM, int WN, int MF, int NF, int VW, int NS>
__global__ __launch_bounds__(64 * WM * WN) void prompt_gemm_kernel(GemvArgs a, float* __restrict__ partial,
                                                                  int steps_per_split, int cpb_shift,
                                                                  int m_tiles, int n_tiles) {
    using S = PgShape<FMT, WM, WN, MF, NF, VW>;
    extern __shared__ __align__(1024) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, li = lane & 15;
    const int wm = wave % WM, wn = wave / WM;
    const int M = a.M, N = a.N;
    // block -> tile: the tiles of one weight row block run on one XCD, side by side
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int nt = idx % n_tiles, mt = (idx / n_tiles) * 8 + xcd;
    if (mt >= m_tiles) return;
    const int m0 = mt * S::BM, n0 = nt * S::BN;
    const int s0 = blockIdx.y * steps_per_split;
    const int nsteps = min(a.K / 32, s0 + steps_per_split) - s0;

    // ---- this lane's global sources, as offsets from block-uniform bases that advance per k step
    const long ldw = a.ldw > 0 ? a.ldw : (long)(FMT == WF_BF16 ? 2L * a.K : FMT == WF_I8 ? (long)a.K : a.K / 2);
    const uint8_t* wbase = uniform_ptr(reinterpret_cast<const uint8_t*>(a.w) + (long)m0 * ldw + (long)(s0 / S::KU) * S::RB);
    const uint8_t* xbase = uniform_ptr(reinterpret_cast<const uint8_t*>(a.x + (long)n0 * a.x_stride_n + (long)s0 * 32));
    const uint8_t* sbase = FMT == WF_I4 ? uniform_ptr(reinterpret_cast<const uint8_t*>(a.scales + (long)m0 * a.bpr)) : nullptr;
    uint32_t woff[S::W_LD], xoff[S::X_LD], soff[S::S_LD > 0 ? S::S_LD : 1];
    constexpr int WI = S::W_BYTES / (64 * VW), XI = S::X_BYTES / 1024, SI = S::S_BYTES / 256;
#pragma unroll
    for (int j = 0; j < S::W_LD; ++j) {
        const int inst = min(wave + S::WAVES * j, WI - 1);
        const int p = (inst * 64 + lane) * VW;                   // byte of the unit's weight tile
        const int r = p / S::RB, c = (p % S::RB) >> 4;
        const int sw = S::CH == 8 ? r & 7 : (r >> 1) & 3;
        woff[j] = (uint32_t)((long)min(r, M - 1 - m0) * ldw + ((c ^ sw) << 4) + (p & 15));
    }
#pragma unroll
    for (int j = 0; j < S::X_LD; ++j) {
        const int inst = min(wave + S::WAVES * j, XI - 1);
        const int r = inst * 8 + (lane >> 3), c = (lane & 7) ^ (r & 7);
        xoff[j] = (uint32_t)((long)min(r, N - 1 - n0) * a.x_stride_n * 4 + c * 16);
    }
    if constexpr (FMT == WF_I4) {
        // (step q of the unit, row r): the scale of the step's block
#pragma unroll
        for (int j = 0; j < S::S_LD; ++j) {
            const int p = min(wave + S::WAVES * j, SI - 1) * 64 + lane, q = p / S::BM, r = p % S::BM;
            soff[j] = (uint32_t)((long)min(r, M - 1 - m0) * a.bpr * 4 + ((q >> cpb_shift) << 2));
        }
    }
    const auto wsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wbase), 0, 0xFFFFFFFFu, 0x00020000);
    const auto xsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(xbase), 0, 0xFFFFFFFFu, 0x00020000);
    auto issue_w = [&](int u) {                                  // weight unit u into ring slot u % WR
        uint8_t* st = lds + (u % S::WR) * S::U_BYTES;
#pragma unroll
        for (int j = 0; j < S::W_LD; ++j)
            load_lds<VW>(wsrc, woff[j], u * S::RB, st + min(wave + S::WAVES * j, WI - 1) * 64 * VW);
        if constexpr (FMT == WF_I4) {
            const auto ssrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(sbase), 0, 0xFFFFFFFFu, 0x00020000);
            const uint32_t so = (uint32_t)((s0 + u * S::KU) >> cpb_shift) * 4;
#pragma unroll
            for (int j = 0; j < S::S_LD; ++j)
                load_lds<4>(ssrc, soff[j], so, st + S::W_BYTES + min(wave + S::WAVES * j, SI - 1) * 256);
        }
    };
    auto issue_x = [&](int s) {                                  // activations of step s into slot s % XR
        uint8_t* st = lds + S::X_OFS + (s % S::XR) * S::X_BYTES;
#pragma unroll
        for (int j = 0; j < S::X_LD; ++j)
            load_lds<16>(xsrc, xoff[j], s * 128, st + min(wave + S::WAVES * j, XI - 1) * 1024);
    };

    // ---- fragments
    PgRaw<FMT> w[MF];                                                  // (bf16: the operands)
    bf16x8 b[FMT == WF_BF16 ? 1 : MF];
    f32x4 x0[NF], x1[NF];
    float sc[FMT == WF_I4 ? MF : 1], scn[FMT == WF_I4 ? MF : 1];
    const int wrow = wm * MF * 16 + li, xrow = wn * NF * 16 + li;
    // lane (g, li) reads k = 8g..8g+7 of row li of each 16-row tile; 16-byte
    // chunk c of row r sits in slot c ^ (r & 7) (or (r >> 1) & 3 of four)
    const int wsw = S::CH == 8 ? wrow & 7 : (wrow >> 1) & 3;
    const int xofs0 = xrow * 128 + (((2 * g) ^ (xrow & 7)) << 4);
    const int xofs1 = xrow * 128 + (((2 * g + 1) ^ (xrow & 7)) << 4);
    auto w_unit = [&](int s) { return (const uint8_t*)lds + ((s / S::KU) % S::WR) * S::U_BYTES; };
    auto x_slot = [&](int s) { return (const uint8_t*)lds + S::X_OFS + (s % S::XR) * S::X_BYTES; };
    auto read_w = [&](const uint8_t* st, int q, int i) {         // q: step of the unit
        const int r = (wrow + 16 * i) * S::RB;
        if constexpr (FMT == WF_BF16)
            w[i] = *reinterpret_cast<const PgRaw<FMT>*>(st + r + (((4 * q + g) ^ wsw) << 4));
        else if constexpr (FMT == WF_I8)
            w[i] = *reinterpret_cast<const PgRaw<FMT>*>(st + r + (((2 * q + (g >> 1)) ^ wsw) << 4) + (g & 1) * 8);
        else {
            w[i] = *reinterpret_cast<const PgRaw<FMT>*>(st + r + ((q ^ wsw) << 4) + g * 4);
            scn[i] = *reinterpret_cast<const float*>(st + S::W_BYTES + (q * S::BM + wrow + 16 * i) * 4);
        }
    };
    auto read_x = [&](const uint8_t* st, int j) {
        x0[j] = *reinterpret_cast<const f32x4*>(st + xofs0 + j * 2048);
        x1[j] = *reinterpret_cast<const f32x4*>(st + xofs1 + j * 2048);
    };
    // (three parts: odd steps with the sign turned)
    auto flip = [&](int s) { return (uint32_t)(s & 1) << 31; };
    auto split_x = [&](int j, uint32_t f, bf16x8 (&part)[NS]) { pg_split<NS>(x0[j], x1[j], f, part); };
    auto conv_w = [&](int i) {
        if constexpr (FMT != WF_BF16) b[i] = pg_operand<FMT>(w[i]);
    };
    auto w_op = [&](int i) -> bf16x8 {
        if constexpr (FMT == WF_BF16) return __builtin_bit_cast(bf16x8, w[i]);
        else return b[i];
    };

    f32x4 acc[NF][MF];
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
        for (int i = 0; i < MF; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // activation tile j against every weight tile; last: each weight tile's
    // registers take the next step's tile as soon as it is done
    auto mfma_group = [&](const bf16x8 (&xp)[NS], int j, float sgn, const uint8_t* wst, int q, bool last) {
        if constexpr (FMT == WF_I4) {
            constexpr int H = MF / 2;
#pragma unroll
            for (int h = 0; h < MF; h += H) {
                f32x4 d[H];
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int i = 0; i < H; ++i) {
                        d[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            xp[s], w_op(h + i), s ? d[i] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        if (last && s + 1 == NS) conv_w(h + i);
                    }
#pragma unroll
                for (int i = 0; i < H; ++i) acc[j][h + i] += d[i] * sc[h + i];
            }
            if (last)
#pragma unroll
                for (int i = 0; i < MF; ++i) sc[i] = scn[i];
        } else if constexpr (NS == 3) {
            // small parts first; each step's sum joins the running one by a
            // rounded addition
            constexpr int H = MF / 2;
#pragma unroll
            for (int h = 0; h < MF; h += H) {
                f32x4 d[H];
#pragma unroll
                for (int s = NS - 1; s >= 0; --s)
#pragma unroll
                    for (int i = 0; i < H; ++i) {
                        d[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            xp[s], w_op(h + i), s == NS - 1 ? f32x4{0.f, 0.f, 0.f, 0.f} : d[i], 0, 0, 0);
                        if (last && s == 0) {
                            if constexpr (FMT == WF_BF16) read_w(wst, q, h + i);
                            else conv_w(h + i);
                        }
                    }
#pragma unroll
                for (int i = 0; i < H; ++i) acc[j][h + i] += d[i] * sgn;
            }
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int i = 0; i < MF; ++i) {
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xp[s], w_op(i), acc[j][i], 0, 0, 0);
                    if (last && s + 1 == NS) {
                        if constexpr (FMT == WF_BF16) read_w(wst, q, i);
                        else conv_w(i);
                    }
                }
        }
    };

    // ---- pipeline: rings of WR weight units and XR activation steps;
    // fragments are read one step ahead
    const int nunits = nsteps / S::KU;
    // what step t issues: the activations of step t + XR - 1 and, at step 0 of
    // unit u, weight unit u + WR - 1 (before them when the next unit needs it)
    auto issue = [&](int t, bool guard) {
        const bool wu = t % S::KU == 0;
        const int u = t / S::KU + S::WR - 1;
        if (S::W_FIRST && wu && (!guard || u < nunits)) issue_w(u);
        if (!guard || t + S::XR - 1 < nsteps) issue_x(t + S::XR - 1);
        if (!S::W_FIRST && wu && (!guard || u < nunits)) issue_w(u);
    };
#pragma unroll
    for (int u = 0; S::KU * (u - S::WR + 1) < 1 - S::XR; ++u)
        if (u < nunits) issue_w(u);
#pragma unroll
    for (int t = 1 - S::XR; t < 0; ++t) issue(t, true);
    // steps 1 - XR .. -1 behind step 0's own loads
    constexpr int W_BEHIND = (S::XR - 1) / S::KU - (S::W_FIRST && (S::XR - 1) % S::KU == 0 ? 1 : 0);
    if (nsteps >= S::XR - 1 && nunits >= S::WR - 1) sync_stage<(S::XR - 2) * S::X_LD + W_BEHIND * S::U_LD>();
    else sync_stage<0>();
    const uint8_t *wst = w_unit(0), *xst = x_slot(0);
#pragma unroll
    for (int j = 0; j < NF; ++j) read_x(xst, j);
#pragma unroll
    for (int i = 0; i < MF; ++i) read_w(wst, 0, i);
#pragma unroll
    for (int i = 0; i < MF; ++i) conv_w(i);
    if constexpr (FMT == WF_I4) {
#pragma unroll
        for (int i = 0; i < MF; ++i) sc[i] = scn[i];
    }
    bf16x8 xp[NS];
    split_x(0, 0, xp);

    // One k step s (step q of its weight unit): its fragments are in registers
    // (tile 0's split done), and step s + 1 has landed at the barrier.
    constexpr int WG = NF > 1 ? NF - 1 : 1, WPG = (MF + WG - 1) / WG;
    auto compute = [&](int s, int q) {
        const uint8_t *wst = w_unit(s + 1), *xst = x_slot(s + 1);
        const int qn = (q + 1) % S::KU;
        bf16x8 yp[NS];
        __builtin_amdgcn_sched_barrier(0);
        read_x(xst, 0);
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            if constexpr (FMT != WF_BF16) {
#pragma unroll
                for (int i = j * WPG; i < min(MF, (j + 1) * WPG); ++i) read_w(wst, qn, i);
            }
            if (j + 1 < NF) {
                split_x(j + 1, flip(s), yp);
                read_x(xst, j + 1);
            } else {
                split_x(0, flip(s + 1), yp);
            }
            mfma_group(xp, j, (s & 1) ? -1.0f : 1.0f, wst, qn, j + 1 == NF);
#pragma unroll
            for (int s = 0; s < NS; ++s) xp[s] = yp[s];
        }
    };
    // At the barrier of step s the slots of step s - 1 are free (every wave
    // has used its reads).  It leaves in flight what was issued behind the
    // activations of step s + 1: those of XR - 3 steps, and the weight unit
    // of a step in [s - XR + 2 (+ 1 if weights go first), s - 1].
    int s = 0;
    for (; s + S::XR - 1 + S::KU - 1 < nsteps && s / S::KU + S::WR - 1 < nunits; s += S::KU) {
        auto one = [&](auto qc) {
            constexpr int q = decltype(qc)::value, lo = q - S::XR + 2 + (S::W_FIRST ? 1 : 0);
            constexpr int nw = (q > 0 && lo <= 0 ? 1 : 0) + (lo <= -S::KU ? 1 : 0);
            sync_stage<(S::XR - 3) * S::X_LD + nw * S::U_LD>();
            issue(s + q, false);
            compute(s + q, q);
        };
        if constexpr (FMT == WF_I4) {
#pragma unroll 1
            for (int q = 0; q < S::KU; ++q) {
                sync_stage<(S::XR - 3) * S::X_LD>();
                issue(s + q, false);
                compute(s + q, q);
            }
            continue;
        }
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        if constexpr (S::KU == 4) {
            one(std::integral_constant<int, 2>{});
            one(std::integral_constant<int, 3>{});
        }
    }
    for (; s < nsteps; s += S::KU) {
#pragma unroll 1
        for (int q = 0; q < S::KU; ++q) {
            sync_stage<0>();
            issue(s + q, true);
            compute(s + q, q);                 // (past the last step it reads spent slots)
        }
    }

    // ---- epilogue: lane (g, li) holds D[4 g + v][li] of tile (j, i)
    const int mb = m0 + wm * MF * 16 + li, nb = n0 + wn * NF * 16 + 4 * g;
    if constexpr (FMT == WF_I8) {
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            const float rs = a.scales[min(mb + 16 * i, M - 1)];
#pragma unroll
            for (int j = 0; j < NF; ++j) acc[j][i] *= rs;
        }
    } else if constexpr (FMT == WF_I4) {
#pragma unroll
        for (int j = 0; j < NF; ++j)
#pragma unroll
            for (int i = 0; i < MF; ++i) acc[j][i] *= 1.0f / kI4Unit;
    }
    const bool split_out = gridDim.y > 1;
    if (!split_out && a.epi == EPI_SILU_MUL) {
#pragma unroll
        for (int j = 0; j < NF; ++j)
#pragma unroll
            for (int i = 0; i < MF; ++i) pg_store_swiglu(a, acc[j][i], mb + 16 * i, nb + 16 * j);
        return;
    }
    float* y0 = split_out ? partial + (long)blockIdx.y * N * M + mb : a.y + (long)mb * a.y_stride_m;
    const long sn = split_out ? M : a.y_stride_n, sm = split_out ? 16 : 16 * a.y_stride_m;
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int n = nb + 16 * j + v;
            if (n < N) {
                float* yr = y0 + n * sn;
#pragma unroll
                for (int i = 0; i < MF; ++i)
                    if (mb + 16 * i < M) yr[i * sm] = acc[j][i][v];
            }
        }
}

// ---- few rows ------------------------------------------------------------------
// Up to 64 rows the weights' stream bounds the product and a k step is too
// little work for a barrier of its own (0.4 us whatever it computes).  Here the
// eight waves of a block split K as well: wave (wm, kg) owns MF weight tiles x
// all NF activation tiles and step kg of every unit of KG steps, so a barrier
// covers 128 k, no two waves convert the same weights, and the partial sums of
// the KG waves meet in LDS once, at the end.
template <int FMT, int MF, int NF, int VW>
struct FrShape {
    static constexpr int WM = 2, KG = 4, WAVES = WM * KG, THREADS = 64 * WAVES;
    static constexpr int BM = WM * MF * 16, BN = NF * 16;
    static constexpr int RB = FMT == WF_BF16 ? 256 : FMT == WF_I8 ? 128 : 64;  // bytes of a weight row per unit
    static constexpr int W_BYTES = BM * RB, X_BYTES = BN * 512;
    static constexpr int S_BYTES = FMT == WF_I4 ? BM * 16 : 0;
    static constexpr int WI = W_BYTES / (64 * VW), XI = X_BYTES / 1024, SI = S_BYTES / 256;
    static constexpr int W_LD = (WI + WAVES - 1) / WAVES, X_LD = (XI + WAVES - 1) / WAVES;
    static constexpr int S_LD = (SI + WAVES - 1) / WAVES, LD = W_LD + X_LD + S_LD;
    static constexpr int UNIT = W_BYTES + X_BYTES + S_BYTES;
    // units in the ring: up to six in half of the LDS, three or at least two in all of it
    static constexpr int UR0 = 80 * 1024 / UNIT, UR = UR0 > 6 ? 6 : UR0 >= 3 ? UR0 : 3 * UNIT <= 160 * 1024 ? 3 : 2;
    static constexpr int RED = WAVES * MF * NF * 1024;
    static constexpr int BYTES = UR * UNIT > RED ? UR * UNIT : RED;
};

template <int FMT, int MF, int NF, int VW, int NS>
__global__ __launch_bounds__(512) void few_rows_gemm_kernel(GemvArgs a, float* __restrict__ partial,
                                                             int units_per_split, int cpb_shift) {
    using S = FrShape<FMT, MF, NF, VW>;
    extern __shared__ __align__(1024) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, li = lane & 15;
    const int wm = wave % S::WM, kg = wave / S::WM;
    const int M = a.M, N = a.N;
    const int m0 = blockIdx.x * S::BM, n0 = blockIdx.z * S::BN;
    const int u0 = blockIdx.y * units_per_split;
    const int nunits = min(a.K / 128, u0 + units_per_split) - u0;

    const long ldw = a.ldw > 0 ? a.ldw : (long)(FMT == WF_BF16 ? 2L * a.K : FMT == WF_I8 ? (long)a.K : a.K / 2);
    const uint8_t* wbase = uniform_ptr(reinterpret_cast<const uint8_t*>(a.w) + (long)m0 * ldw + (long)u0 * S::RB);
    const uint8_t* xbase = uniform_ptr(reinterpret_cast<const uint8_t*>(a.x + (long)n0 * a.x_stride_n + (long)u0 * 128));
    const uint8_t* sbase = FMT == WF_I4 ? uniform_ptr(reinterpret_cast<const uint8_t*>(a.scales + (long)m0 * a.bpr)) : nullptr;
    uint32_t woff[S::W_LD], xoff[S::X_LD], soff[S::S_LD > 0 ? S::S_LD : 1];
#pragma unroll
    for (int j = 0; j < S::W_LD; ++j) {
        const int p = (min(wave + S::WAVES * j, S::WI - 1) * 64 + lane) * VW;
        const int r = p / S::RB, c = (p % S::RB) >> 4;
        const int sw = S::RB >= 128 ? r & 7 : (r >> 1) & 3;
        woff[j] = (uint32_t)((long)min(r, M - 1 - m0) * ldw + ((c ^ sw) << 4) + (p & 15));
    }
#pragma unroll
    for (int j = 0; j < S::X_LD; ++j) {
        const int p = min(wave + S::WAVES * j, S::XI - 1) * 64 + lane;       // 16-byte piece: 32 per row
        const int r = p >> 5, c = (p & 31) ^ (r & 7);
        xoff[j] = (uint32_t)((long)min(r, N - 1 - n0) * a.x_stride_n * 4 + c * 16);
    }
    if constexpr (FMT == WF_I4) {
#pragma unroll
        for (int j = 0; j < S::S_LD; ++j) {
            const int p = min(wave + S::WAVES * j, S::SI - 1) * 64 + lane, q = p / S::BM, r = p % S::BM;
            soff[j] = (uint32_t)((long)min(r, M - 1 - m0) * a.bpr * 4 + ((q >> cpb_shift) << 2));
        }
    }
    const auto wsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wbase), 0, 0xFFFFFFFFu, 0x00020000);
    const auto xsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(xbase), 0, 0xFFFFFFFFu, 0x00020000);
    auto issue = [&](int u) {
        uint8_t* st = lds + (u % S::UR) * S::UNIT;
#pragma unroll
        for (int j = 0; j < S::W_LD; ++j)
            load_lds<VW>(wsrc, woff[j], u * S::RB, st + min(wave + S::WAVES * j, S::WI - 1) * 64 * VW);
#pragma unroll
        for (int j = 0; j < S::X_LD; ++j)
            load_lds<16>(xsrc, xoff[j], u * 512, st + S::W_BYTES + min(wave + S::WAVES * j, S::XI - 1) * 1024);
        if constexpr (FMT == WF_I4) {
            const auto ssrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(sbase), 0, 0xFFFFFFFFu, 0x00020000);
            const uint32_t so = (uint32_t)((u0 + u) * S::KG >> cpb_shift) * 4;
#pragma unroll
            for (int j = 0; j < S::S_LD; ++j)
                load_lds<4>(ssrc, soff[j], so,
                            st + S::W_BYTES + S::X_BYTES + min(wave + S::WAVES * j, S::SI - 1) * 256);
        }
    };

    const int wrow = wm * MF * 16 + li;
    const int wsw = S::RB >= 128 ? wrow & 7 : (wrow >> 1) & 3;
    const int wofs = wrow * S::RB + (FMT == WF_BF16 ? ((4 * kg + g) ^ wsw) << 4
                                     : FMT == WF_I8 ? (((2 * kg + (g >> 1)) ^ wsw) << 4) + (g & 1) * 8
                                                    : ((kg ^ wsw) << 4) + g * 4);
    const int xofs0 = S::W_BYTES + li * 512 + (((8 * kg + 2 * g) ^ (li & 7)) << 4);
    const int xofs1 = S::W_BYTES + li * 512 + (((8 * kg + 2 * g + 1) ^ (li & 7)) << 4);
    const int sofs = S::W_BYTES + S::X_BYTES + (kg * S::BM + wrow) * 4;

    f32x4 acc[NF][MF];
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
        for (int i = 0; i < MF; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](int u) {
        const uint8_t* st = lds + (u % S::UR) * S::UNIT;
        f32x4 x0[NF], x1[NF];
        PgRaw<FMT> w[MF];
        float sc[FMT == WF_I4 ? MF : 1];
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            x0[j] = *reinterpret_cast<const f32x4*>(st + xofs0 + j * 16 * 512);
            x1[j] = *reinterpret_cast<const f32x4*>(st + xofs1 + j * 16 * 512);
        }
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            w[i] = *reinterpret_cast<const PgRaw<FMT>*>(st + wofs + i * 16 * S::RB);
            if constexpr (FMT == WF_I4) sc[i] = *reinterpret_cast<const float*>(st + sofs + i * 64);
        }
        bf16x8 xp[NF][NS];
        const uint32_t flip = (uint32_t)(kg & 1) << 31;             // the step is KG u + kg
        const float sgn = (kg & 1) ? -1.0f : 1.0f;
#pragma unroll
        for (int j = 0; j < NF; ++j) pg_split<NS>(x0[j], x1[j], flip, xp[j]);
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            const bf16x8 b = pg_operand<FMT>(w[i]);
            f32x4 d[NF];
#pragma unroll
            for (int j = 0; j < NF; ++j)
                d[j] = FMT == WF_I4 || NS == 3 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[j][i];
#pragma unroll
            for (int s = 0; s < NS; ++s)                       // (three parts: the small ones first)
#pragma unroll
                for (int j = 0; j < NF; ++j)
                    d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xp[j][NS == 3 ? 2 - s : s], b, d[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                if constexpr (FMT == WF_I4) acc[j][i] += d[j] * sc[i];
                else if constexpr (NS == 3) acc[j][i] += d[j] * sgn;
                else acc[j][i] = d[j];
            }
        }
    };

    // ring: at the barrier of unit u its loads have landed and the slot of unit
    // u - 1, whose reads every wave has used, takes unit u + UR - 1
#pragma unroll
    for (int u = 0; u < S::UR - 1; ++u)
        if (u < nunits) issue(u);
    int u = 0;
    for (; u + S::UR - 1 < nunits; ++u) {
        sync_stage<(S::UR - 2) * S::LD>();
        issue(u + S::UR - 1);
        compute(u);
    }
    for (; u < nunits; ++u) {
        sync_stage<0>();
        compute(u);
    }

    // ---- the KG partial sums meet: each wave finishes every WAVES-th tile
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(lds);               // [kg][wm][j][i][lane]
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
        for (int i = 0; i < MF; ++i) red[(((kg * S::WM + wm) * NF + j) * MF + i) * 64 + lane] = acc[j][i];
    __syncthreads();
    constexpr int TILES = S::WM * NF * MF;
    const bool split_out = gridDim.y > 1;
    for (int t = wave; t < TILES; t += S::WAVES) {
        f32x4 v = red[t * 64 + lane];
#pragma unroll
        for (int k = 1; k < S::KG; ++k) v += red[(k * TILES + t) * 64 + lane];
        const int twm = t / (NF * MF), j = t / MF % NF, i = t % MF;
        const int m = m0 + (twm * MF + i) * 16 + li, nb = n0 + 16 * j + 4 * g;
        if constexpr (FMT == WF_I8) v *= a.scales[min(m, M - 1)];
        if constexpr (FMT == WF_I4) v *= 1.0f / kI4Unit;
        if (!split_out && a.epi == EPI_SILU_MUL) {
            pg_store_swiglu(a, v, m, nb);
        } else if (m < M) {
            float* y = split_out ? partial + (long)blockIdx.y * N * M + m : a.y + (long)m * a.y_stride_m;
            const long sn = split_out ? M : a.y_stride_n;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (nb + r < N) y[(nb + r) * sn] = v[r];
        }
    }
}

// ---- tile and K split ------------------------------------------------------------
enum { PG_256x128, PG_192x128, PG_128x128, PG_256x64, PG_TILES };
struct PgTile { int bm, bn; float step[3]; };      // us per k step of a block (bf16, int8, int4)
// From the 7B shapes at 1024 rows (rounds of 256 blocks x 128 or 344 steps).
static constexpr PgTile kPgTiles[PG_TILES] = {{256, 128, {0.83f, 1.02f, 1.30f}},
                                              {192, 128, {0.71f, 0.86f, 1.14f}},
                                              {128, 128, {0.54f, 0.66f, 0.85f}},
                                              {256, 64, {0.60f, 0.66f, 0.85f}}};
// us per unit (128 k) of a few-rows block of 64 or 128 weight rows x 16, 32 or 64
// activation rows, from the 7B gate/up and the 16384 x 2048 shapes
static constexpr float kFrUnit[3][3][2] = {{{0.50f, 0.95f}, {0.62f, 1.00f}, {0.94f, 1.50f}},
                                           {{0.36f, 0.63f}, {0.45f, 0.79f}, {0.80f, 1.20f}},
                                           {{0.47f, 0.70f}, {0.59f, 0.94f}, {1.10f, 1.54f}}};
constexpr int kFewRows = 64, kMaxSplits = 32;
// few: the few-rows kernel, tile = weight tiles per wave (2, 4), steps = units of 128 k
struct PgPlan { bool few; int tile, splits, steps; };

static int pg_fmt(int fmt) { return fmt == WF_BF16 ? 0 : fmt == WF_I8 ? 1 : 2; }
static int fr_nf(int N) { return N <= 16 ? 1 : N <= 32 ? 2 : 4; }

// The tile and K split of least estimated time: rounds of one block per CU, each
// 4 us (first loads, stores) plus its k steps, and for a split the partials'
// write and read at ~5 TB/s and the sum's launch.  Counted with N rounded up to
// a tile, so that sizing at those N covers every N.  Measured against the
// neighbours in this order (us, bf16): 127 rows gate/up 192 rows x 2 splits 64,
// 256 x 2 68, 128 x 1 69; QKV 192 x 4 39, 256 x 4 42, 128 x 2 44; W_down
// 128 x 8 37, 192 x 8 42; 24 rows gate/up 128 x 1 40, 64 x 1 48; W_down 64 x 4
// 24, 128 x 8 25.
static PgPlan pg_plan(int fmt, int M, int N, int K, int max_splits = kMaxSplits) {
    const int f = pg_fmt(fmt), cus = device_cu_count();
    PgPlan best{};
    float best_us = 0.f;
    auto consider = [&](bool few, int tile, int bm, int bn, float step) {
        const int total = few ? K / 128 : K / 32, unit = few ? 1 : 4;
        const int nn = N <= kFewRows ? bn : (N + 63) / 64 * 64;
        const long tiles = (long)((M + bm - 1) / bm) * ((nn + bn - 1) / bn);
        const float stream_us = few ? (float)M * gemv_row_bytes(fmt, K) / 5.5e6f : 0.f;
        for (int want = 1; want <= max_splits; ++want) {
            const int steps = ((total + want - 1) / want + unit - 1) / unit * unit;
            const int splits = (total + steps - 1) / steps;
            if (splits != want) continue;
            const long rounds = (tiles * splits + cus - 1) / cus;
            float us = few ? 4.f + std::max(rounds * steps * step, stream_us) : rounds * (4.f + steps * step);
            if (splits > 1) us += 3.f + (float)splits * nn * M * 8.f / 5e6f;
            if (best_us == 0.f || us < best_us) {
                best = PgPlan{few, tile, splits, steps};
                best_us = us;
            }
        }
    };
    if (N <= 2 * kFewRows)
        for (int mf = 2; mf <= 4; mf += 2)
            consider(true, mf, 32 * mf, 16 * fr_nf(N), kFrUnit[f][fr_nf(N) >> 1][mf >> 2]);
    if (N > kFewRows)
        for (int t = 0; t < PG_TILES; ++t)
            consider(false, t, kPgTiles[t].bm, kPgTiles[t].bn, kPgTiles[t].step[f]);
    return best;
}

template <int FMT, int WM, int WN, int MF, int NF, int VW = 16>
static void pg_go(const GemvArgs& a, const PgPlan& p, float* partial, int cpb_shift, hipStream_t st) {
    using S = PgShape<FMT, WM, WN, MF, NF, VW>;
    static_assert(S::BYTES <= 160 * 1024, "LDS of a CU");
    const int mt = (a.M + S::BM - 1) / S::BM, nt = (a.N + S::BN - 1) / S::BN;
    const dim3 grid((mt + 7) / 8 * 8 * nt, p.splits);
    if constexpr (FMT != WF_I4) {
        if (a.f32x) {
            hipLaunchKernelGGL((prompt_gemm_kernel<FMT, WM, WN, MF, NF, VW, 3>), grid, dim3(S::THREADS), S::BYTES,
                               st, a, partial, p.steps, cpb_shift, mt, nt);
            return;
        }
    }
    hipLaunchKernelGGL((prompt_gemm_kernel<FMT, WM, WN, MF, NF, VW, 2>), grid, dim3(S::THREADS), S::BYTES, st, a,
                       partial, p.steps, cpb_shift, mt, nt);
}

template <int FMT, int MF, int NF, int VW = 16>
static void fr_go(const GemvArgs& a, const PgPlan& p, float* partial, int cpb_shift, hipStream_t st) {
    using S = FrShape<FMT, MF, NF, VW>;
    static_assert(S::BYTES <= 160 * 1024, "LDS of a CU");
    const dim3 grid((a.M + S::BM - 1) / S::BM, p.splits, (a.N + S::BN - 1) / S::BN);
    if constexpr (FMT != WF_I4) {
        if (a.f32x) {
            hipLaunchKernelGGL((few_rows_gemm_kernel<FMT, MF, NF, VW, 3>), grid, dim3(S::THREADS), S::BYTES, st, a,
                               partial, p.steps, cpb_shift);
            return;
        }
    }
    hipLaunchKernelGGL((few_rows_gemm_kernel<FMT, MF, NF, VW, 2>), grid, dim3(S::THREADS), S::BYTES, st, a, partial,
                       p.steps, cpb_shift);
}

// 16-byte loads need 16-byte aligned weight rows; others (int8 from 8, int4
// from 4 bytes up) load 4 bytes per lane, in one tile of each kind
template <int FMT>
static void pg_launch(const GemvArgs& a, const PgPlan& p, float* partial, int sh, hipStream_t st) {
    const int nf = fr_nf(a.N);
    if constexpr (FMT != WF_BF16) {
        if (((uintptr_t)a.w | (uintptr_t)a.ldw) & 15) {
            if (!p.few) pg_go<FMT, 2, 4, 4, 2, 4>(a, p, partial, sh, st);
            else if (nf == 1) fr_go<FMT, 2, 1, 4>(a, p, partial, sh, st);
            else if (nf == 2) fr_go<FMT, 2, 2, 4>(a, p, partial, sh, st);
            else fr_go<FMT, 2, 4, 4>(a, p, partial, sh, st);
            return;
        }
    }
    if (p.few && p.tile == 2) {
        if (nf == 1) fr_go<FMT, 2, 1>(a, p, partial, sh, st);
        else if (nf == 2) fr_go<FMT, 2, 2>(a, p, partial, sh, st);
        else fr_go<FMT, 2, 4>(a, p, partial, sh, st);
    } else if (p.few) {
        if (nf == 1) fr_go<FMT, 4, 1>(a, p, partial, sh, st);
        else if (nf == 2) fr_go<FMT, 4, 2>(a, p, partial, sh, st);
        else fr_go<FMT, 4, 4>(a, p, partial, sh, st);
    } else {
        switch (p.tile) {
        case PG_256x128: pg_go<FMT, 2, 4, 8, 2>(a, p, partial, sh, st); break;
        case PG_192x128: pg_go<FMT, 2, 4, 6, 2>(a, p, partial, sh, st); break;
        case PG_128x128: pg_go<FMT, 2, 4, 4, 2>(a, p, partial, sh, st); break;
        default: pg_go<FMT, 4, 2, 4, 2>(a, p, partial, sh, st); break;
        }
    }
}

// a: after gemv_fill_int4_index (int4 bpr / cpb); any N
bool gemm_rows_ok(const GemvArgs& a) {
    const uintptr_t wa = (uintptr_t)a.w;
    const bool fmt_ok =
        a.fmt == WF_BF16 ? (wa & 15) == 0 && (a.ldw == 0 || a.ldw % 16 == 0)
        : a.fmt == WF_I8 ? a.scales && (wa & 7) == 0 && (a.ldw == 0 || a.ldw % 8 == 0)
        : a.fmt == WF_I4 ? a.scales && (wa & 3) == 0 && a.ldw == 0 && a.block % 32 == 0 &&
                               a.bpr > 0 && (a.cpb & (a.cpb - 1)) == 0
                         : false;
    return fmt_ok && a.K % 128 == 0 && a.K > 0 && a.M > 0 &&
           a.x_stride_k == 1 && a.x_stride_n % 4 == 0 && ((uintptr_t)a.x & 15) == 0 &&
           (a.epi == EPI_STORE || (a.epi == EPI_SILU_MUL && a.M % 2 == 0));
}

// a tile's rows are addressed with 32-bit offsets from its first
bool gemm_rows_fit(const GemvArgs& a) {
    const long ldw = a.ldw > 0 ? a.ldw : gemv_row_bytes(a.fmt, a.K);
    return 256 * ldw < (1L << 32) && 128 * 4L * a.x_stride_n < (1L << 32) && a.K <= (1 << 23);
}

// the row counts that pg_plan tells apart: 16, 32, 64 and every 64 from there
static int pg_next_rows(int n) { return n < 16 ? 16 : n < kFewRows ? 2 * n : n + 64; }

size_t gemm_rows_partial_bytes(int fmt, int M, int N, int K) {
    size_t need = 0;
    for (int n = 0; n < N;) {
        n = pg_next_rows(n);
        const int sp = pg_plan(fmt, M, n, K).splits;
        if (sp > 1) need = std::max(need, (size_t)sp * std::min(n, N) * M * sizeof(float));
    }
    return need;
}

// What an eager call on the thread's scratch leaves there: enough for any
// smaller N of the same weights (up to kHoldRows), so that such a call is
// captured as it would run.  Fewer rows split K more: 4096 x 4096 not at all at
// 1024 rows (76 us), eight times at 127 (21 us; 73 unsplit).  The plans are
// looked at once per shape and thread (~1 us each).
constexpr int kHoldRows = 1024;
static size_t scratch_to_hold(const GemvArgs& a) {
    struct Shape { int fmt, M, K, rows; size_t bytes; };
    static thread_local Shape shapes[64] = {};
    Shape& s = shapes[((unsigned)a.M * 31u + (unsigned)a.K * 7u + (unsigned)a.fmt) % 64u];
    if (s.fmt != a.fmt || s.M != a.M || s.K != a.K)
        s = Shape{a.fmt, a.M, a.K, 0, skinny_partial_bytes(a.M, 16, a.K)};
    while (s.rows < std::min(a.N, kHoldRows)) {
        s.rows = pg_next_rows(s.rows);
        const int sp = pg_plan(a.fmt, a.M, s.rows, a.K).splits;
        if (sp > 1) s.bytes = std::max(s.bytes, (size_t)sp * s.rows * a.M * sizeof(float));
    }
    return s.bytes;
}

int gemm_rows_launch(const GemvArgs& a, hipStream_t st) {
    ATLAS_REQUIRE(gemm_rows_ok(a) && gemm_rows_fit(a), "gemm rows: unsupported shape (fmt %d, n %d, k %d)",
                  a.fmt, a.N, a.K);
    PgPlan p = pg_plan(a.fmt, a.M, a.N, a.K);
    float* partial = nullptr;
    const size_t split = (size_t)a.N * a.M * sizeof(float);
    const size_t need = p.splits > 1 ? p.splits * split : 0;
    const size_t hold = a.partial ? need : std::max(need, scratch_to_hold(a));
    // (an unsplit call touches the scratch only to make it large enough)
    const bool ask = need > 0 || (hold > 0 && hold > thread_scratch_held(SCR_GEMM));
    if (ask && skinny_partial_for(a, hold, &partial)) {
        // Not to be had (no memory, or a capture on a thread that made no such
        // call before it): what there is takes fewer splits, or none.
        clear_error();
        const size_t have = a.partial ? a.partial_bytes : thread_scratch_held(SCR_GEMM);
        if (need > have) p = pg_plan(a.fmt, a.M, a.N, a.K, std::max(1, (int)(have / split)));
        if (p.splits > 1) {
            const int rc = skinny_partial_for(a, p.splits * split, &partial);
            if (rc) return rc;
        }
    }
    int sh = 0;
    while ((1 << sh) < a.cpb) ++sh;
    if (a.fmt == WF_BF16) pg_launch<WF_BF16>(a, p, partial, sh, st);
    else if (a.fmt == WF_I8) pg_launch<WF_I8>(a, p, partial, sh, st);
    else pg_launch<WF_I4>(a, p, partial, sh, st);
    ATLAS_LAUNCH_CHECK("prompt_gemm");
    if (p.splits > 1 && skinny_defer_ok(a)) {
        *a.defer_splits = p.splits;           // the consumer sums the partials
        return ATLAS_OK;
    }
    return p.splits > 1 ? skinny_reduce_launch(a, partial, p.splits, st) : ATLAS_OK;
}

}  // namespace atlas
