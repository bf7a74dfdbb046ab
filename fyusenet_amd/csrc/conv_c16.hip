// Two 3x3 convolutions, one behind the other, between tensors of few channels as one launch (a residual block of a small
// style net, the middle of a light decoder) on gfx950 matrix cores (v_mfma_f32_16x16x32_f16, fp32 accumulate).
//
// Replaces, for such a pair, two passes of ConvLayerNxN::forward (fyusenet/gpu/vanilla/convlayerNxN_vanilla.cpp) or
// DeepConvLayerNxN::forward (fyusenet/gpu/deep/deepconvlayerNxN.cpp:129-211), with the residual input of the second.
//
// Bound: a launch's fixed cost, then the matrix pipes.  Apart, the two layers are launches of 4 us at 12x16 positions and of
// 8 us at 156x128, of which a microsecond is matrix work.  A workgroup owns TH rows of sixteen positions; it stages the
// input under them, two pixels wider on every side, computes the first layer one pixel wider into its LDS -- 1.5 times the
// positions for TH = 6 -- and the second from there.  As in conv_p16n.hip a step is four groups of eight channels wherever
// they lie in the window.  Waves: one per fragment of 16 output channels, share of the reduction and share of the positions
// (halves of both, twelve waves for three fragments; quarters of the reduction on tiles of two rows), so that all weights
// come through the L1 twice (once) and a wave's share of a layer stays in registers; the second layer's steps replace the
// first one's as those are through.
// Measured, one launch / apart: 40 to 40 to 40 at 156x128 fp32 12.0 / 16.3 us, fp16 8.7 / 11.0 (6.5k and 2.2k clocks of them
// matrix instructions); 48 to 48 to 48 at 161x121 12.9 / 17.1 and 9.2 / 11.1; at 256x256, where the tiles take three rounds,
// 32.0 / 29.2.  The samples' 9x9 style net at 512x624 167 -> 149 us a frame, fp16 117 -> 104.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"
#include "p16_common.h"
#include "range.h"

namespace fynhip {
namespace {
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// HS: fp16 tensors, G: groups of 8 channels of the input and of the tensor in between, FR: fragments of 16 output channels
// of either layer, TH: rows of a tile
template <bool HS_, int G_, int FR_, int TH_>
struct GeoC {
    static constexpr bool HS = HS_;
    static constexpr int G = G_, FR = FR_, TH = TH_;
    static constexpr int NPL = HS ? 1 : 2, NPASS = HS ? 1 : 3;
    // shares of the reduction and of the positions: few positions, and the weights are worth reading only once
    static constexpr int KS = TH <= 2 ? 4 : 2, NH = 4 / KS, WAVES = FR * KS * NH, NT = WAVES * 64;
    static constexpr int NS = (9 * G + 3) / 4, SPW = (NS + KS - 1) / KS;       // steps of a layer, of a wave
    static constexpr int PXB = (G | 1) * 16;                                   // bytes of a pixel and plane: an odd number of 16-byte pieces
    static constexpr int IW = 20, IH = TH + 4, MW = 18, MH = TH + 2;           // the staged input, the first layer's positions
    static constexpr int IN_PLANE = IW * IH * PXB, MID_PLANE = MW * MH * PXB;
    static constexpr int NITEMS = IW * IH * G, NB = (NITEMS + NT - 1) / NT;    // staging items: (pixel, 8 channels)
    static constexpr int NF1 = (MW * MH + 15) / 16, NF2 = TH;                  // fragments of positions
    static constexpr int NW1 = (NF1 + NH - 1) / NH, NW2 = (NF2 + NH - 1) / NH; // of a wave
    static constexpr int OWN1 = (NW1 + KS - 1) / KS, OWN2 = (NW2 + KS - 1) / KS;   // that it finishes
    static constexpr bool EARLY = SPW * NPL <= 8;                              // the second layer's weights are requested at the start as well
    static constexpr int MID = NPL * IN_PLANE, RED = MID + NPL * MID_PLANE;
    static constexpr int LDS = RED + WAVES * NW1 * 1024;
    static_assert(NT <= 1024 && LDS <= 160 * 1024 - 64, "a workgroup fits a CU");
};

template <class N>
__global__ __launch_bounds__(N::NT) void conv_c16_kernel(const ConvC16Params p) {
    constexpr bool HS = N::HS;
    constexpr int G = N::G, FR = N::FR, TH = N::TH, NPL = N::NPL, NPASS = N::NPASS, KS = N::KS, SPW = N::SPW, NT = N::NT;
    typedef typename std::conditional<HS, _Float16, float>::type store_t;
    typedef float f32x8_t __attribute__((ext_vector_type(8)));
    typedef typename std::conditional<HS, half8_t, f32x8_t>::type raw_t;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ unsigned box[4];   // largest magnitude of the tensor in between (bits), and what range_publish_waves takes
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mq = lane & 15, kq = lane >> 4;
    const unsigned range_bits = p.in_amax ? range_load(p.in_amax) : 0u;
    // (neighbouring tiles, whose windows overlap, meet in one XCD's L2)
    int bid = blockIdx.x;
    {
        const int per = (int)gridDim.x >> 3;
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const int tyi = (int)(((float)bid + 0.5f) * p.rcp_tiles_x), txi = bid - tyi * p.tiles_x;
    const int y0 = tyi * TH, x0 = txi * 16;

    // ---- everything the workgroup reads is requested here ----
    raw_t raw[N::NB];
    unsigned inside = 0u;   // one bit an item
    const store_t* const in = reinterpret_cast<const store_t*>(p.in);
#pragma unroll
    for (int i = 0; i < N::NB; i++) {
        const int item = tid + i * NT, pix = item / G, g = item - pix * G, wy = pix / N::IW, wx = pix - wy * N::IW;
        int y = y0 - 2 + wy, x = x0 - 2 + wx;
        if (p.clamp) {
            y = min(max(y, 0), p.h - 1);
            x = min(max(x, 0), p.w - 1);
        }
        const bool ok = item < N::NITEMS && (unsigned)y < (unsigned)p.h && (unsigned)x < (unsigned)p.w;
        inside |= ok ? 1u << i : 0u;
        raw[i] = *reinterpret_cast<const raw_t*>(in + (ok ? ((y + p.in_off) * p.in_wp + x + p.in_off) * p.in_cp + g * 8 : 0));
    }
    const int mf = wave % FR, share = (wave / FR) % KS, part = wave / (FR * KS);
    const unsigned char* const w1 = reinterpret_cast<const unsigned char*>(p.wpack) + (size_t)((mf * KS + share) * SPW * NPL) * 1024 + lane * 16;
    const unsigned char* const w2 = w1 + (size_t)(FR * KS * SPW * NPL) * 1024;
    half8_t a[SPW][NPL];
#pragma unroll
    for (int s = 0; s < SPW; s++)
#pragma unroll
        for (int pl = 0; pl < NPL; pl++) a[s][pl] = *reinterpret_cast<const half8_t*>(w1 + (s * NPL + pl) * 1024);
    const int ch = mf * 16 + kq * 4;
    const f32x4_t sc1 = *reinterpret_cast<const f32x4_t*>(p.scale[0] + ch), bi1 = *reinterpret_cast<const f32x4_t*>(p.bias[0] + ch);
    const f32x4_t sc2 = *reinterpret_cast<const f32x4_t*>(p.scale[1] + ch), bi2 = *reinterpret_cast<const f32x4_t*>(p.bias[1] + ch);
    half8_t a2[N::EARLY ? SPW : 1][NPL];
    if constexpr (N::EARLY) {
#pragma unroll
        for (int s = 0; s < SPW; s++)
#pragma unroll
            for (int pl = 0; pl < NPL; pl++) a2[s][pl] = *reinterpret_cast<const half8_t*>(w2 + (s * NPL + pl) * 1024);
    }
    // (the shares of a fragment of positions finish every KS-th one each)
    typedef typename std::conditional<HS, half4_t, f32x4_t>::type res_t;
    res_t rv[N::OWN2];
    if (p.res) {
#pragma unroll
        for (int j = 0; j < N::OWN2; j++) {
            const int oy = y0 + part * N::NW2 + share + KS * j, ox = x0 + mq;
            const bool ok = share + KS * j < N::NW2 && part * N::NW2 + share + KS * j < TH && oy < p.h && ox < p.w && ch + 4 <= p.out_cp;
            rv[j] = *reinterpret_cast<const res_t*>(reinterpret_cast<const store_t*>(p.res) + (ok ? ((size_t)(p.res_off + oy) * p.res_wp + p.res_off + ox) * p.res_cp + ch : 0));
        }
    }
    // where a lane's group of each step lies: in the staged input, in the tensor in between
    int off1[SPW], off2[SPW];
#pragma unroll
    for (int s = 0; s < SPW; s++) {
        const int g = min(4 * (share + KS * s) + kq, 9 * G - 1), t = g / G, ty = (t * 11) >> 5, tx = t - 3 * ty;   // (t / 3)
        off1[s] = (ty * N::IW + tx) * N::PXB + (g - t * G) * 16;
        off2[s] = (ty * N::MW + tx) * N::PXB + (g - t * G) * 16;
    }
    if (tid < 4) box[tid] = 0u;
    if (blockIdx.x == 0) range_clear(p.reset[0], p.reset[1], p.reset[2], p.reset[3], p.nreset);

    // ---- activation and operand conversion ----
    float in_scale = 1.f, inv_in = 1.f;
    if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act[0]), &inv_in);
    auto convert = [&](auto kind_) __attribute__((always_inline)) {
        constexpr int KIND = decltype(kind_)::value;
        _Float16 hlo, hhi;
        const bool packed = act_half_exact(p.act[0], hlo, hhi);
#pragma unroll
        for (int i = 0; i < N::NB; i++) {
            const int item = tid + i * NT, pix = item / G, g = item - pix * G, at = pix * N::PXB + g * 16;
            const bool ok = (inside >> i) & 1u;
            if constexpr (HS) {
                half8_t v = raw[i];
                if (packed) {
                    v = ok ? act_half(v, hlo, hhi) : (half8_t)((_Float16)0.f);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = ok ? (_Float16)act_p16((float)v[e], p.act[0]) : (_Float16)0.f;
                }
                if (item < N::NITEMS) *reinterpret_cast<half8_t*>(lds + at) = v;
            } else {
                const float x[8] = {raw[i][0], raw[i][1], raw[i][2], raw[i][3], raw[i][4], raw[i][5], raw[i][6], raw[i][7]};
                half8_t hi, lo;
                split8<KIND>(x, ok, p.act[0], in_scale, hi, lo);
                if (item < N::NITEMS) {
                    *reinterpret_cast<half8_t*>(lds + at) = hi;
                    *reinterpret_cast<half8_t*>(lds + N::IN_PLANE + at) = lo;
                }
            }
        }
    };
    if (HS || p.act[0].kind == ACT_LEAKY || p.act[0].kind == ACT_CLIP) convert(std::integral_constant<int, ACT_LEAKY>());
    else if (p.act[0].kind == ACT_RELU) convert(std::integral_constant<int, ACT_RELU>());
    else convert(std::integral_constant<int, ACT_NONE>());
    lds_barrier();   // the input is staged

    // A wave's steps on its NF fragments of positions: base(n) + off[step] is the lane's place.  Positions are requested
    // LA fragments ahead.
    auto steps = [&](auto nf_, auto& acc, auto&& base, const int (&off)[SPW], int plane, auto&& done) __attribute__((always_inline)) {
        constexpr int NF = decltype(nf_)::value, LA = 3, Q = SPW * NF;
        half8_t b[LA + 1][NPL];
        auto request = [&](int q) __attribute__((always_inline)) {
            const unsigned char* at = lds + base(q % NF) + off[q / NF];
#pragma unroll
            for (int pl = 0; pl < NPL; pl++) b[q % (LA + 1)][pl] = *reinterpret_cast<const half8_t*>(at + pl * plane);
        };
#pragma unroll
        for (int q = 0; q < LA && q < Q; q++) request(q);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int s = q / NF, n = q % NF;
            if (q + LA < Q) request(q + LA);
#pragma unroll
            for (int i = 0; i < NPASS; i++)
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[s][i == 1 ? NPL - 1 : 0], b[q % (LA + 1)][i == 2 ? NPL - 1 : 0], acc[n], 0, 0, 0);
            if (n == NF - 1) done(s);
        }
    };
    // The shares of a fragment meet: each wave leaves what the others finish and adds what they left.
    auto meet = [&](auto nf_, auto own_, auto& acc, auto& sum) __attribute__((always_inline)) {
        constexpr int NF = decltype(nf_)::value, OWN = decltype(own_)::value;
        unsigned char* const red = lds + N::RED;
#pragma unroll
        for (int n = 0; n < NF; n++)
            if (n % KS != share) *reinterpret_cast<f32x4_t*>(red + (wave * NF + n) * 1024 + lane * 16) = acc[n];
#pragma unroll
        for (int j = 0; j < OWN; j++) {
            sum[j] = acc[KS * j];
#pragma unroll
            for (int k = 1; k < KS; k++)
                if (share == k) sum[j] = KS * j + k < NF ? acc[KS * j + k < NF ? KS * j + k : 0] : (f32x4_t)(0.f);
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < OWN; j++) {
            const int n = min(share + KS * j, NF - 1);
#pragma unroll
            for (int k = 1; k < KS; k++) {
                const int other = wave + (((share + k) & (KS - 1)) - share) * FR;
                sum[j] += *reinterpret_cast<const f32x4_t*>(red + (other * NF + n) * 1024 + lane * 16);
            }
        }
    };

    // ---- first layer, on the tile and one position around it ----
    f32x4_t sum1[N::OWN1];
    {
        f32x4_t acc[N::NW1];
        int base[N::NW1];
#pragma unroll
        for (int n = 0; n < N::NW1; n++) {
            acc[n] = (f32x4_t)(0.f);
            const int idx = min((part * N::NW1 + n) * 16 + mq, N::MW * N::MH - 1), wy = idx / N::MW, wx = idx - wy * N::MW;
            base[n] = (wy * N::IW + wx) * N::PXB;
        }
        steps(std::integral_constant<int, N::NW1>(), acc, [&](int n) { return base[n]; }, off1, N::IN_PLANE, [&](int s) {
#pragma unroll
            for (int pl = 0; pl < NPL; pl++) {
                if constexpr (N::EARLY) a[s][pl] = a2[s][pl];
                else a[s][pl] = *reinterpret_cast<const half8_t*>(w2 + (s * NPL + pl) * 1024);
            }
        });
        meet(std::integral_constant<int, N::NW1>(), std::integral_constant<int, N::OWN1>(), acc, sum1);
    }
    float inv_mid = 1.f;
    {
        const float lo = p.act[1].kind == ACT_NONE ? -3.0e38f : p.act[1].kind == ACT_RELU ? 0.f : p.act[1].lo;
        const float hi = p.act[1].kind == ACT_NONE || p.act[1].kind == ACT_RELU ? 3.0e38f : p.act[1].hi;
        const float leak = p.act[1].kind == ACT_NONE || p.act[1].kind == ACT_RELU ? 0.f : p.act[1].leak;
        _Float16 hlo, hhi;
        const bool packed = act_half_exact(p.act[1], hlo, hhi);
        const float mul = p.acc_mul[0] * inv_in;
        float top = 0.f;
        half4_t hv[N::OWN1];
#pragma unroll
        for (int j = 0; j < N::OWN1; j++) {
            const int n = share + KS * j, idx = (part * N::NW1 + n) * 16 + mq, wy = idx / N::MW, wx = idx - wy * N::MW;
            const bool ok = n < N::NW1 && idx < N::MW * N::MH && (unsigned)(y0 - 1 + wy) < (unsigned)p.h && (unsigned)(x0 - 1 + wx) < (unsigned)p.w;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float v = sum1[j][e] * (sc1[e] * mul) + bi1[e];
                if constexpr (HS) {
                    hv[j][e] = (_Float16)v;   // (as the layer would have stored it)
                } else {
                    float x = __builtin_amdgcn_fmed3f(v, lo, hi);
                    if (leak != 0.f) x += leak * fminf(v, 0.f);
                    sum1[j][e] = ok ? x : 0.f;
                    top = fmaxf(top, ok ? fabsf(v) : 0.f);   // (in front of the activation, whose clamp makes a number of a NaN)
                }
            }
            if constexpr (HS) {
                if (packed) {
                    hv[j] = act_half4(hv[j], hlo, hhi);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) hv[j][e] = (_Float16)act_p16((float)hv[j][e], p.act[1]);
                }
                if (!ok) hv[j] = (half4_t)((_Float16)0.f);
            }
        }
        float s = 1.f;
        if constexpr (!HS) {   // the operand split needs the window's largest magnitude (range.h), as the layer's word would give the tensor's
            top = range_wave_max(top);
            if (lane == 0) atomicMax(&box[0], __float_as_uint(top));
            lds_barrier();
            s = range_scale(range_after_act(__uint_as_float(box[0]), p.act[1]), &inv_mid);
        }
#pragma unroll
        for (int j = 0; j < N::OWN1; j++) {
            const int n = share + KS * j, idx = (part * N::NW1 + n) * 16 + mq;
            if (n >= N::NW1 || idx >= N::MW * N::MH || ch >= G * 8) continue;
            unsigned char* const to = lds + N::MID + idx * N::PXB + ch * 2;
            if constexpr (HS) {
                *reinterpret_cast<half4_t*>(to) = hv[j];
            } else {
                uint2 h, l;
                split_pair(sum1[j][0], sum1[j][1], s, h.x, l.x);
                split_pair(sum1[j][2], sum1[j][3], s, h.y, l.y);
                *reinterpret_cast<uint2*>(to) = h;
                *reinterpret_cast<uint2*>(to + N::MID_PLANE) = l;
            }
        }
    }
    lds_barrier();   // the first layer's result is there
    if (p.clamp && (y0 == 0 || x0 == 0 || y0 + TH >= p.h || x0 + 16 >= p.w)) {   // positions outside the frame repeat its edge
        for (int item = tid; item < N::MW * N::MH * G; item += NT) {
            const int idx = item / G, g = item - idx * G, wy = idx / N::MW, wx = idx - wy * N::MW;
            const int y = y0 - 1 + wy, x = x0 - 1 + wx, cy = min(max(y, 0), p.h - 1), cx = min(max(x, 0), p.w - 1);
            const int from = (cy - y0 + 1) * N::MW + cx - x0 + 1;
            // (the tile's own positions are inside the frame or read by nobody who stores)
            if ((cy == y && cx == x) || cy < y0 - 1 || cx < x0 - 1) continue;
#pragma unroll
            for (int pl = 0; pl < NPL; pl++)
                *reinterpret_cast<half8_t*>(lds + N::MID + pl * N::MID_PLANE + idx * N::PXB + g * 16) =
                    *reinterpret_cast<const half8_t*>(lds + N::MID + pl * N::MID_PLANE + from * N::PXB + g * 16);
        }
        lds_barrier();
    }

    // ---- second layer ----
    f32x4_t sum2[N::OWN2];
    {
        f32x4_t acc[N::NW2];
#pragma unroll
        for (int n = 0; n < N::NW2; n++) acc[n] = (f32x4_t)(0.f);
        const int base = N::MID + (part * N::NW2 * N::MW + mq) * N::PXB;
        steps(std::integral_constant<int, N::NW2>(), acc, [&](int n) { return base + (N::NW2 * N::NH > TH ? min(n, TH - 1 - part * N::NW2) : n) * N::MW * N::PXB; }, off2, N::MID_PLANE, [](int) {});
        meet(std::integral_constant<int, N::NW2>(), std::integral_constant<int, N::OWN2>(), acc, sum2);
    }
    float vmax = 0.f;
    {
        const float mul = p.acc_mul[1] * inv_mid;
        store_t* const out = reinterpret_cast<store_t*>(p.out);
#pragma unroll
        for (int j = 0; j < N::OWN2; j++) {
            const int n = share + KS * j, row = part * N::NW2 + n, oy = y0 + row, ox = x0 + mq;
            const bool ok = n < N::NW2 && row < TH && oy < p.h && ox < p.w && ch + 4 <= p.out_cp;
            f32x4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = sum2[j][e] * (sc2[e] * mul) + bi2[e];
            if (p.res) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float r = (float)rv[j][e];
                    if (p.res_relu) r = fmaxf(r, 0.f);
                    if (p.res_scale) r *= sc2[e];
                    v[e] += r;
                }
            }
            store_t* const to = out + ((size_t)(p.out_off + oy) * p.out_wp + p.out_off + ox) * p.out_cp + ch;
            if constexpr (HS) {
                half4_t hv;
#pragma unroll
                for (int e = 0; e < 4; e++) hv[e] = (_Float16)v[e];
                if (ok) *reinterpret_cast<half4_t*>(to) = hv;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) vmax = fmaxf(vmax, ok ? fabsf(v[e]) : 0.f);
                if (ok) *reinterpret_cast<f32x4_t*>(to) = v;
            }
        }
    }
    if (p.out_amax) range_publish_waves(p.out_amax, vmax, &box[2], N::WAVES);
}

typedef void (*c16_fn)(const ConvC16Params);
struct C16Entry {
    int f16, groups, frags, th, waves, shares;
    size_t steps, lds;
    c16_fn fn;
};
template <bool HS, int G, int FR, int TH>
constexpr C16Entry c16_entry() {
    using N = GeoC<HS, G, FR, TH>;
    return C16Entry{HS, G, FR, TH, N::WAVES, N::KS, (size_t)N::SPW, (size_t)N::LDS, conv_c16_kernel<N>};
}
#define C16_BOTH(G, FR, TH) c16_entry<false, G, FR, TH>(), c16_entry<true, G, FR, TH>()
const C16Entry kC16[] = {
    C16_BOTH(5, 3, 2), C16_BOTH(5, 3, 4), C16_BOTH(5, 3, 6),
    C16_BOTH(6, 3, 2), C16_BOTH(6, 3, 4), C16_BOTH(6, 3, 6),
};
const C16Entry* find_c16(const ConvC16Params& p) {
    for (const C16Entry& e : kC16)
        if (e.f16 == (p.f16 ? 1 : 0) && e.groups == p.groups && e.th == p.th) return &e;
    return nullptr;
}
}  // namespace

int conv_c16_count() { return (int)(sizeof(kC16) / sizeof(kC16[0])); }
void conv_c16_variant(int index, int* f16, int* groups, int* frags, int* th) {
    const C16Entry& e = kC16[index];
    *f16 = e.f16; *groups = e.groups; *frags = e.frags; *th = e.th;
}
int conv_c16_steps(const ConvC16Params& p, int* shares) {
    const C16Entry* e = find_c16(p);
    *shares = e ? e->shares : 0;
    return e ? (int)e->steps : 0;
}
size_t conv_c16_lds_bytes(const ConvC16Params& p) {
    const C16Entry* e = find_c16(p);
    return e ? e->lds : 0;
}
int launch_conv_c16(const ConvC16Params& p, hipStream_t s) {
    const C16Entry* e = find_c16(p);
    if (!e) return -1;
    const long long tiles = (long long)p.tiles_x * p.tiles_y;
    if (!p.in || !p.out || !p.wpack || p.in_cp != 8 * e->groups || p.h < 1 || p.w < 1 || p.in_off < 0 || p.h + p.in_off > p.in_hp || p.w + p.in_off > p.in_wp ||
        (long long)p.in_hp * p.in_wp * p.in_cp > (1ll << 30) || p.out_cp % 4 != 0 || p.out_cp < 4 || p.out_cp > 16 * e->frags || (p.res && (p.res_cp < p.out_cp || p.res_cp % 4 != 0)) ||
        p.tiles_x != (p.w + 15) / 16 || p.tiles_y != (p.h + e->th - 1) / e->th || tiles > (1 << 22) || p.nreset < 0 || p.nreset > 4)
        return -5;
    if (ensure_lds(reinterpret_cast<const void*>(e->fn), e->lds) != 0) return -2;
    hipLaunchKernelGGL(e->fn, dim3((unsigned)tiles), dim3(64 * e->waves), e->lds, s, p);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace fynhip
