// What the kernels with a first layer on four-channel pixels share (conv_p16.hip: conv_p16c4_kernel; conv_a16.hip): the tile's
// geometry, its staging and the schedule of its matrix instructions on rows of sixteen positions.  The including file is
// compiled twice: for fp32 tensors (operands split into fp16 hi and lo planes, three MFMA passes) and, with
// -DFYN_P16_HALF=1, for fp16 tensors (one plane, one pass).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "kernels.h"
#include "p16_common.h"
#include "range.h"

#ifndef FYN_P16_HALF
#define FYN_P16_HALF 0
#endif

namespace fynhip {
namespace {
constexpr int NT = 9;         // taps
constexpr int PD = 6;         // depth of the weight-fragment ring (steps)
constexpr bool HSTORE = FYN_P16_HALF != 0;   // fp16 tensors
constexpr int NPL = HSTORE ? 1 : 2;          // staged planes (hi, lo)
constexpr int NPASS = HSTORE ? 1 : 3;        // MFMAs per fragment pair (hi*hi, lo*hi, hi*lo)
// fp32 tensors, weight planes per fragment (launch_conv_p16, launch_tconv_p16): fp16 hi, fp16 lo, and the fp8 operands of
// the correction terms, [8 x fp8(hi / 32) | 8 x fp8(lo * 64)] per lane; a kernel reads plane 0 and one of the other two
constexpr int NPLW = HSTORE ? 1 : 3;
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
constexpr int ESZ = HSTORE ? 2 : 4;          // bytes per stored element
typedef std::conditional<HSTORE, _Float16, float>::type store_t;
// Output channel, inside a wave's 32, of accumulator element e of channel fragment fm in the lanes kq = lane / 16:
// kq * CHK + fm * CHF + e.  fp32 tensors: fragment rows are channels in order (a fragment's store is 64 contiguous bytes
// from the four lanes of a position).  fp16 tensors: the weights are packed so that a lane's eight values are eight
// consecutive channels (one 16-byte store per lane and position instead of two of 8 bytes; with fp32 tensors the same
// layout -- two 16-byte stores per lane, interleaved between lanes -- measured slower).
constexpr int CHK = HSTORE ? 8 : 4, CHF = HSTORE ? 4 : 16;
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// f(0), f(1), ... f(N - 1) with the index as a type (the loops of a stage are expanded ahead of the optimiser, which takes
// arrays indexed in loops this long to memory)
template <class F, int... I>
__device__ __forceinline__ void expand(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>()), ...);
}
template <class G>
__device__ __forceinline__ void rows_load_b8(i32x8_t& dst, int half, const unsigned char* at) {
    const i32x4_t v = *reinterpret_cast<const i32x4_t*>(at);
    if (half == 0) { dst[0] = v[0]; dst[1] = v[1]; dst[2] = v[2]; dst[3] = v[3]; }
    else { dst[4] = v[0]; dst[5] = v[1]; dst[6] = v[2]; dst[7] = v[3]; }
}
__device__ __forceinline__ void rows_put_w(half8_t (&a0)[2][2], i32x8_t (&a2)[2], int k, const i32x4_t v) {
    const int step = (k / 2) % 2, fm = k % 2;
    if (k < 4) a0[step][fm] = __builtin_bit_cast(half8_t, v);
    else if (step == 0) { a2[fm][0] = v[0]; a2[fm][1] = v[1]; a2[fm][2] = v[2]; a2[fm][3] = v[3]; }
    else { a2[fm][4] = v[0]; a2[fm][5] = v[1]; a2[fm][6] = v[2]; a2[fm][7] = v[3]; }
}
template <int K, int TH_, int TW>
struct GeoC4 {
    static constexpr int TH = TH_, STEP = 1, WN = 4, TWG = 4 * TW;
    static constexpr int PPR = (K + 1) / 2, NPAIR = K * PPR;          // tap pairs per kernel row, in all
    // (the staged width covers the empty tap that pads an odd kernel row to whole pairs: its weight is zero, but the
    // pixel it is multiplied with must be a number)
    static constexpr int HW = TWG + 2 * PPR - 1, HH = TH + K - 1;
    static constexpr int NS = ((NPAIR + 3) / 4 + 2) / 3 * 3;          // steps per stage (two stages are whole turns of the weight ring)
    static constexpr int PIX = 8;                                     // bytes per staged pixel and plane
    static constexpr int ROW_PITCH = (HW * PIX + 15) / 16 * 16 + 16;
    // A plane is staged twice, the second copy eight bytes further on: the two pixels of a tap pair are then 16 aligned
    // bytes in one of the copies whatever the parity of the pair's first pixel, and a B fragment is one 16-byte LDS read
    // (with 8-byte reads the four tap pairs of a step meet in the same banks and the reads, not the MFMAs, set the pace:
    // 59 % MFMA issue inside the step loop).  The copies lie 64 bytes apart modulo the 128 of the banks: of eight
    // neighbouring positions the even ones read the first copy and the odd ones the second, all banks once.
    static constexpr int COPY = HH * ROW_PITCH;
    static constexpr int COPY2 = (COPY + 127) / 128 * 128 + 48;        // offset of the second copy (its pixel x at COPY2 + 8 + 8 x)
    static constexpr int PLANE = COPY2 + COPY + 16;
    static constexpr int BUF = NPL * PLANE;
    static constexpr int NPOS = TH * TW, FN = NPOS / 16;
    static constexpr int NITEMS = HH * HW;                            // staging items: pixels
    static constexpr int NB = (NITEMS + 255) / 256;
    static constexpr int CPB = 32, FM = 2;                            // output channels, fragments of them
    // tiles whose fragments are rows of sixteen positions take the tap pairs in another order: c4_rows
    static constexpr bool ROWS = TW == 16;
    static_assert(!ROWS || K == 9, "rows: eight taps of a kernel row and one more");
    static_assert(NPOS % 16 == 0 && (2 * NS) % PD == 0, "whole position fragments; whole ring turns");
    static_assert((ROWS ? BUF : 2 * BUF + PLANE) < 65536, "offsets fit the LDS instructions' immediate field");
};

template <class G, bool C8>
__device__ __forceinline__ void c4_stager(const ConvP16Params& p, unsigned char* lds, int stid, int cb, int group, int ntiles, unsigned range_bits) {
    constexpr int sb_off = 2 * G::BUF;
    const store_t* in = reinterpret_cast<const store_t*>(p.in);
    int i_y[G::NB], i_x[G::NB], l_off[G::NB];
#pragma unroll
    for (int i = 0; i < G::NB; i++) {
        const int idx = stid + i * 256;
        l_off[i] = -1; i_y[i] = 1 << 20; i_x[i] = 0;
        if (idx < G::NITEMS) {
            const int py = idx / G::HW, px = idx - py * G::HW;
            i_y[i] = py; i_x[i] = px;
            l_off[i] = py * G::ROW_PITCH + px * G::PIX;
        }
    }
    int g_off[2][G::NB];
    typedef typename std::conditional<HSTORE, half4_t, float4>::type raw_t;   // a pixel as it comes from memory
    raw_t raw[2][G::NB];
    float in_scale = 1.f, inv_unused;
    auto fetch = [&](auto set_, int tile) {
        constexpr int SET = decltype(set_)::value;
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        const int y0 = tyi * G::TH + p.in_y0, x0 = txi * G::TWG + p.in_x0;
#pragma unroll
        for (int i = 0; i < G::NB; i++) {
            int gy = y0 + i_y[i], gx = x0 + i_x[i];
            if (p.in_clamp && l_off[i] >= 0) {
                gy = min(max(gy, 0), p.in_hp - 1);
                gx = min(max(gx, 0), p.in_wp - 1);
            }
            g_off[SET][i] = ((unsigned)gy < (unsigned)p.in_hp && (unsigned)gx < (unsigned)p.in_wp) ? (gy * p.in_wp + gx) * 4 : -1;
            raw[SET][i] = *reinterpret_cast<const raw_t*>(in + (g_off[SET][i] >= 0 ? g_off[SET][i] : 0));
        }
    };
    const bool plain_act = p.act.kind == ACT_NONE;   // (a first layer reads its input as it is)
    auto store = [&](auto set_, unsigned char* buf) {
        constexpr int SET = decltype(set_)::value;
#pragma unroll
        for (int i = 0; i < G::NB; i++) {
            if (l_off[i] < 0) continue;
            const bool ok = g_off[SET][i] >= 0;
            if constexpr (HSTORE) {
                half4_t v;
                _Float16 hlo, hhi;
                if (act_half_exact(p.act, hlo, hhi)) {   // (on the packed halves, as in p16_stager)
                    v = ok ? act_half4(raw[SET][i], hlo, hhi) : (half4_t)((_Float16)0.f);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = ok ? (_Float16)act_p16((float)raw[SET][i][e], p.act) : (_Float16)0.f;
                }
                *reinterpret_cast<half4_t*>(buf + l_off[i]) = v;
                *reinterpret_cast<half4_t*>(buf + G::COPY2 + 8 + l_off[i]) = v;
            } else {
                // (the hi/lo split of a pair of values in four instructions, as in split8)
                const float r[4] = {raw[SET][i].x, raw[SET][i].y, raw[SET][i].z, raw[SET][i].w};
                float x[4];
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = ok ? (plain_act ? r[e] : act_p16(r[e], p.act)) : 0.f;
                unsigned h0, l0, h1, l1;
                split_pair(x[0], x[1], in_scale, h0, l0);
                split_pair(x[2], x[3], in_scale, h1, l1);
                const half4_t hi = __builtin_bit_cast(half4_t, uint2{h0, h1}), lo = __builtin_bit_cast(half4_t, uint2{l0, l1});
                *reinterpret_cast<half4_t*>(buf + l_off[i]) = hi;
                *reinterpret_cast<half4_t*>(buf + G::COPY2 + 8 + l_off[i]) = hi;
                if constexpr (C8) {
                    // the pixel's fp8 operands of the correction terms: [4 x fp8(32 lo) | 4 x fp8(hi / 64)]
                    const int2 c8 = int2{(int)c8_quad(lo[0], lo[1], lo[2], lo[3], 0.03125f), (int)c8_quad(hi[0], hi[1], hi[2], hi[3], 64.f)};
                    *reinterpret_cast<int2*>(buf + G::PLANE + l_off[i]) = c8;
                    *reinterpret_cast<int2*>(buf + G::PLANE + G::COPY2 + 8 + l_off[i]) = c8;
                } else {
                    *reinterpret_cast<half4_t*>(buf + G::PLANE + l_off[i]) = lo;
                    *reinterpret_cast<half4_t*>(buf + G::PLANE + G::COPY2 + 8 + l_off[i]) = lo;
                }
            }
        }
    };
    typedef std::integral_constant<int, 0> Set0;
    typedef std::integral_constant<int, 1> Set1;
    int tile = group;                       // the stage the MFMA waves are on
    int t1 = tile + p.pos_groups, t2 = t1 + p.pos_groups;
    fetch(Set0(), tile);
    if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act), &inv_unused);
    if (stid < 32) {   // (scale and bias have one entry per channel of the output tensor's pitch)
        const bool have = cb * 32 + stid < p.out_cp;
        reinterpret_cast<float*>(lds + sb_off)[stid] = have ? p.scale[cb * 32 + stid] : 0.f;
        reinterpret_cast<float*>(lds + sb_off)[32 + stid] = have ? p.bias[cb * 32 + stid] : 0.f;
    }
    store(Set0(), lds);
    lds_barrier();
    if (t1 < ntiles) fetch(Set1(), t1);
    auto iteration = [&](auto next_set, auto free_set, unsigned char* next_buf) {
        if (t1 < ntiles) store(next_set, next_buf);
        if (t2 < ntiles) fetch(free_set, t2);
        lds_barrier();
        const bool go_on = t1 < ntiles;
        tile = t1; t1 = t2; t2 += p.pos_groups;
        return go_on;
    };
    for (;;) {
        if (!iteration(Set1(), Set0(), lds + G::BUF)) break;
        if (!iteration(Set0(), Set1(), lds)) break;
    }
}

// The stage on tiles whose fragments are rows of sixteen positions (9x9; fp16 tensors, or fp32 with the fp8 form).  Steps
// 0 .. 8 take the first eight taps of kernel row ky (a lane group's pair: taps 2 kq and 2 kq + 1), steps 9 .. 11 the ninth
// tap of four rows each (a pair with an empty partner).  In the first nine the fragment of output row r at ky is that of
// row r + 1 at ky - 1, and so are the fp8 operands of a pair of steps (ky, ky + 1) -- rows r + ky and r + ky + 1 -- for row
// r + 2 at the pair before: both move through registers, and a tile of TH rows reads 4 TH + 8 + 6 TH + 12 fragments from
// LDS instead of 24 TH (TH = 5: 70 against 120).  That leaves room for the weights there (48 KB, or 24 with fp16 tensors):
// the MFMA waves then load nothing from memory, and what they store need not have arrived before they go on -- loads and
// stores of a wave are counted in one order, so weights requested behind a tile's stores waited for the burst that all
// workgroups store at the same time.  Schedule
// and lifetimes as in p16_rows_c8: a slot is one output row of a pair of steps, what it takes is requested LA slots ahead,
// the weights of a pair one pair ahead; the barrier that hands over the next tile lies in front of the first request for it.
// 9x9 3 -> 32: 512x624 fp32 18.8 -> 17.3 us (19.2 with the weights from memory), 1920x1080 fp32 112 -> 102 (104), 1524x1856
// fp16 78 -> 65 (68).  Bound there: the stores (265 MB in 102 us beside 33 read).
template <class G>
struct C4Ring {
    // slots (64 or 128 matrix-pipe cycles; half of them with one fragment of output channels) from an LDS read to its use
    static constexpr int LA = (HSTORE ? 4 : 2) * (G::FM == 1 ? 2 : 1);
    static constexpr int LW = 1;                       // pairs of steps from the request of weights to their use
    half8_t a0[LW][2][2];
    i32x8_t a2[LW][2];
    half8_t b0[LA + 1];                                // rows 0 ..
    i32x8_t b8[LA];                                    // pairs of rows 0 ..
};
// (NEXT: false where the next tile is staged only when this one is through: its operands are not requested here)
template <class G, bool NEXT = true>
__device__ __forceinline__ void c4_rows(f32x4_t (&acc)[G::FM][G::FN], C4Ring<G>& ring, const unsigned char* at_rows, const unsigned char* at_ninth,
                                        const unsigned char* at_last, const unsigned char* next_rows, const unsigned char* weights) {
    constexpr int TH = G::FN, LA = C4Ring<G>::LA, LW = C4Ring<G>::LW, NP = 6, RP = G::ROW_PITCH;
    constexpr bool C8 = !HSTORE;
    static_assert(TH >= 4 && TH > LA - 1 && G::NS == 2 * NP, "a slot has room for its share of the requests");
    half8_t a0[NP + LW][2][2], b0[TH + 8], n0[LA + 1], l0[3][TH];
    i32x8_t a2[NP + LW][2], b8[TH + 6], n8[LA], u8[2][TH];   // (b8[s]: rows s and s + 1; u8: the pairs that hold a step of the ninth tap; n0, n8: the next tile's)
#pragma unroll
    for (int d = 0; d < LW; d++)
#pragma unroll
        for (int fm = 0; fm < G::FM; fm++) {
            a0[d][0][fm] = ring.a0[d][0][fm]; a0[d][1][fm] = ring.a0[d][1][fm];
            if constexpr (C8) a2[d][fm] = ring.a2[d][fm];
        }
#pragma unroll
    for (int r = 0; r <= LA; r++) b0[r] = ring.b0[r];
    if constexpr (C8) {
#pragma unroll
        for (int r = 0; r < LA; r++) b8[r] = ring.b8[r];
    }
    auto half_of = [](const unsigned char* at) { return *reinterpret_cast<const half8_t*>(at); };
    // the ninth tap of rows 4 j + kq and output row r (the last step: only row 8 of the first lane group counts)
    auto ninth = [&](int j, int r) { return j < 2 ? at_ninth + (4 * j + r) * RP : at_last + r * RP; };
    // the n-th read for row r of pair p (p = NP: the next tile's first pair)
    auto request = [&](auto p_, auto r_, auto n_) __attribute__((always_inline)) {
        constexpr int p = decltype(p_)::value, r = decltype(r_)::value, n = decltype(n_)::value;
        if constexpr (p == 0) {
            if constexpr (C8 && n < 2) rows_load_b8<G>(b8[r], n, at_rows + (r + n) * RP + G::PLANE);
            if constexpr (n == 2) b0[r + 1] = half_of(at_rows + (r + 1) * RP);
        } else if constexpr (p < 4) {
            if constexpr (C8 && n < 2 && r >= TH - 2) rows_load_b8<G>(b8[r + 2 * p], n, at_rows + (r + 2 * p + n) * RP + G::PLANE);
            if constexpr (n >= 2 && n < 4 && r == TH - 1) b0[TH + 2 * p + n - 3] = half_of(at_rows + (TH + 2 * p + n - 3) * RP);
        } else if constexpr (p == 4) {
            if constexpr (C8 && n == 0) rows_load_b8<G>(u8[0][r], 0, at_rows + (r + 8) * RP + G::PLANE);
            if constexpr (C8 && n == 1) rows_load_b8<G>(u8[0][r], 1, ninth(0, r) + G::PLANE);
            if constexpr (n == 2) l0[0][r] = half_of(ninth(0, r));
            if constexpr (n == 3 && r == TH - 1) b0[TH + 7] = half_of(at_rows + (TH + 7) * RP);
        } else if constexpr (p == 5) {
            if constexpr (C8 && n < 2) rows_load_b8<G>(u8[1][r], n, ninth(1 + n, r) + G::PLANE);
            if constexpr (n == 2) l0[1][r] = half_of(ninth(1, r));
            if constexpr (n == 3) l0[2][r] = half_of(ninth(2, r));
        } else if constexpr (NEXT) {
            if constexpr (C8 && n < 2) rows_load_b8<G>(n8[r], n, next_rows + (r + n) * RP + G::PLANE);
            if constexpr (n == 2) n0[r + 1] = half_of(next_rows + (r + 1) * RP);
            if constexpr (n == 3 && r == 0) n0[0] = half_of(next_rows);
        }
    };
    auto slot = [&](auto index) __attribute__((always_inline)) {
        constexpr int g = decltype(index)::value, p = g / TH, r = g % TH, u = g + LA;
        if constexpr (NEXT && g == NP * TH - LA) lds_barrier();
        auto issue = [&](auto index_m) __attribute__((always_inline)) {
            constexpr int m = decltype(index_m)::value, fm = m % 2;
            if constexpr (!(HSTORE && (m == 2 || m == 3))) {
                if constexpr (fm >= G::FM) {   // (a slot keeps its places for the reads)
                } else if constexpr (m < 2) {
                    const half8_t b = p < 4 ? b0[p < 4 ? r + 2 * p : 0] : p == 4 ? b0[r + 8 < TH + 8 ? r + 8 : 0] : l0[1][r];
                    acc[fm][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0[p][0][fm], b, acc[fm][r], 0, 0, 0);
                } else if constexpr (m < 4) {
                    acc[fm][r] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a2[p][fm], p < 4 ? b8[p < 4 ? r + 2 * p : 0] : u8[p < 4 ? 0 : p - 4][r], acc[fm][r], 0, 0, 0, 0, 0, 0);
                } else {
                    const half8_t b = p < 4 ? b0[p < 4 ? r + 2 * p + 1 : 0] : p == 4 ? l0[0][r] : l0[2][r];
                    acc[fm][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0[p][1][fm], b, acc[fm][r], 0, 0, 0);
                }
                // (fp16 tensors issue four matrix instructions a slot: their reads are the last two kinds)
                constexpr int n = HSTORE ? (m < 2 ? m + 2 : -1) : m;
                if constexpr (n >= 0 && n < 4) request(std::integral_constant<int, u / TH>(), std::integral_constant<int, u % TH>(), std::integral_constant<int, n>());
                // a share of the weights of pair p + LW
                constexpr int NW = HSTORE ? 4 : 8, k = (r * NW + TH - 1) / TH + m - (HSTORE ? 4 : 2);
                if constexpr (m >= (HSTORE ? 4 : 2) && k < NW && k * TH / NW == r && k % 2 < G::FM)
                    rows_put_w(a0[p + LW], a2[p + LW], k, *reinterpret_cast<const i32x4_t*>(weights + ((p + LW) % NP * NW + k) * 1024));
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        expand(issue, std::make_integer_sequence<int, 6>());
    };
    expand(slot, std::make_integer_sequence<int, NP * TH>());
#pragma unroll
    for (int d = 0; d < LW; d++)
#pragma unroll
        for (int fm = 0; fm < G::FM; fm++) {
            ring.a0[d][0][fm] = a0[NP + d][0][fm]; ring.a0[d][1][fm] = a0[NP + d][1][fm];
            if constexpr (C8) ring.a2[d][fm] = a2[NP + d][fm];
        }
    if constexpr (NEXT) {
#pragma unroll
        for (int r = 0; r <= LA; r++) ring.b0[r] = n0[r];
        if constexpr (C8) {
#pragma unroll
            for (int r = 0; r < LA; r++) ring.b8[r] = n8[r];
        }
    }
}

}  // namespace
}  // namespace fynhip
