// A 1x1 convolution, the 3x3 convolution behind it and the 1x1 convolution behind that as one launch (a bottleneck block of
// a classification net) on gfx950 matrix cores with 16-position fragments (v_mfma_f32_16x16x32_f16, fp32 accumulate).
//
// Replaces, for such a block, DeepConvLayer1x1::forward (fyusenet/gpu/deep/deepconvlayer1x1.cpp:67-117), the render passes
// of DeepConvLayerNxN::forward (deepconvlayerNxN.cpp:129-211) and DeepConvLayer1x1::forward again, with the residual input
// of the last one.
//
// Bound: a launch's fixed cost and the weights through a CU's L1.  At batch 1 each of the three layers is a launch of 4 to
// 5.5 us with less than half a microsecond of matrix work.  A workgroup owns 4x4 positions of the block's output and keeps
// everything between input and output in its LDS: the 6x6 window of the input (all channels, converted once), the first
// layer's result on that window, the second layer's on the tile.  The 20 positions around the tile are computed by up to
// nine workgroups (2.25 times the first layer's arithmetic), and every workgroup reads all weights of the block: 278 KB for
// 256 -> 64 -> 64 -> 256 channels on fp32 tensors, 139 KB on fp16 tensors, at 64 bytes per clock and CU.  The eight waves
// split a layer's output fragments, and where there are fewer of those than waves its reduction too; a wave's weights for
// the three layers lie one behind the other, and the first of a layer's are requested in front of the barrier that its
// operands wait for.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"
#include "p16_common.h"
#include "range.h"

namespace fynhip {
namespace {
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
constexpr int TILE = 4, WIN = TILE + 2, NWIN = WIN * WIN, NPF = (NWIN + 15) / 16;
constexpr int WAVES = 8;

// What the second and third layer take of the layer in front: its activation on a value that is not in memory.
struct MidAct {
    float lo, hi, leak;
    _Float16 hlo, hhi;
    bool packed;
    __device__ __forceinline__ MidAct(const Act& a) {
        lo = a.kind == ACT_NONE ? -3.0e38f : a.kind == ACT_RELU ? 0.f : a.lo;
        hi = a.kind == ACT_NONE || a.kind == ACT_RELU ? 3.0e38f : a.hi;
        leak = a.kind == ACT_NONE || a.kind == ACT_RELU ? 0.f : a.leak;
        packed = act_half_exact(a, hlo, hhi);
    }
    __device__ __forceinline__ float operator()(float x) const {
        float y = __builtin_amdgcn_fmed3f(x, lo, hi);
        if (leak != 0.f) y += leak * fminf(x, 0.f);
        return y;
    }
    __device__ __forceinline__ half4_t operator()(half4_t x) const {
        if (packed) return act_half4(x, hlo, hhi);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = (_Float16)(*this)((float)x[e]);
        return x;
    }
};

// SRC = 1: a batch-norm layer in front of the block, applied while staging (p.in_mul, p.in_add).  PROJ: the last layer adds
// a 1x1 layer on the block's input (the shortcut projection), computed from the staged window.  C0: chunks of 32 channels of
// the input; M: fragments of 16 channels of the two layers in between; NPR: pairs of fragments of output channels per wave.
template <bool HS, int SRC, bool PROJ, int C0, int M, int NPR>
__global__ __launch_bounds__(512, HS && M == 4 && SRC == 0 ? 4 : 2) void conv_b16_kernel(const ConvB16Params p) {
    constexpr int NPL = HS ? 1 : 2, NPASS = HS ? 1 : 3;
    constexpr int KS = WAVES / M, CM = M / 2;             // shares of the reduction of the first two layers; chunks of theirs
    constexpr int T0 = (C0 + KS - 1) / KS, S1 = 9 * CM, T1 = (S1 + KS - 1) / KS, T2 = 2 * CM, T3 = PROJ ? 2 * C0 : 0;   // fragments of a wave
    constexpr int TW = T0 + T1 + NPR * (T2 + T3);
    constexpr int RD = TW < (HS ? 32 : 18) ? TW : (HS ? 32 : 18);   // of them in registers
    static_assert(WAVES % M == 0 && M % 2 == 0, "every wave has a share");
    constexpr int GROUPS = C0 * 4, ITEMS = NWIN * GROUPS, NB = (ITEMS + 511) / 512;   // staging items: (pixel, 8 channels)
    constexpr int IN_PIT = C0 * 64 + 16, IN_PLANE = NWIN * IN_PIT, MID_PIT = CM * 64 + 16, MID_PLANE = NWIN * MID_PIT, M2_PLANE = 16 * MID_PIT;
    constexpr int MID = NPL * IN_PLANE, MID2 = MID + NPL * MID_PLANE, RED = MID2 + NPL * M2_PLANE, SB = RED + (KS > 1 ? WAVES * NPF * 1024 : 0);
    constexpr int OUT = 2 * NPR * WAVES * 16;             // channels of the output's fragments
    typedef typename std::conditional<HS, _Float16, float>::type store_t;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ unsigned box[4];   // largest magnitude of the two layers in between (bit patterns), and what range_publish_waves takes
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mq = lane & 15, kq = lane >> 4;
    if (tid < 4) box[tid] = 0u;
    // (neighbouring tiles, whose windows overlap, meet in one XCD's L2)
    int bid = blockIdx.x;
    {
        const int per = (int)gridDim.x >> 3;
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const int tyi = (int)(((float)bid + 0.5f) * p.rcp_tiles_x), txi = bid - tyi * p.tiles_x;
    const int y0 = tyi * TILE, x0 = txi * TILE;
    const unsigned range_bits = p.in_amax ? range_load(p.in_amax) : 0u;

    // ---- everything the workgroup reads is requested here, in the order in which it is used ----
    struct RawF { float4 a, b; };
    typedef typename std::conditional<HS, half8_t, RawF>::type raw_t;
    raw_t raw[NB];
    int l_off[NB], ch_of[NB];   // (-1: no item; reads as zero)
    const store_t* const in = reinterpret_cast<const store_t*>(p.in);
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int item = tid + i * 512, pix = item / GROUPS, g = item - pix * GROUPS;
        const int wy = pix / WIN, wx = pix - wy * WIN;
        const int y = y0 - 1 + wy, x = x0 - 1 + wx;
        const bool ok = item < ITEMS && (unsigned)y < (unsigned)p.h && (unsigned)x < (unsigned)p.w && g * 8 < p.in_cp;
        l_off[i] = item < ITEMS ? pix * IN_PIT + g * 16 : -1;
        ch_of[i] = ok ? g * 8 : -1;
        const store_t* src = in + (ok ? ((y + p.in_off) * p.in_wp + x + p.in_off) * p.in_cp + g * 8 : 0);
        if constexpr (HS) {
            raw[i] = *reinterpret_cast<const half8_t*>(src);
        } else {
            raw[i].a = *reinterpret_cast<const float4*>(src);
            raw[i].b = *reinterpret_cast<const float4*>(src + 4);
        }
    }
    // (a batch-norm layer in front: a thread's items have the same channels)
    static_assert(SRC == 0 || 512 % GROUPS == 0, "one group of channels per thread");
    [[maybe_unused]] float4 bn[4];
    if constexpr (SRC == 1) {
        const int c = tid % GROUPS * 8 < p.in_cp ? tid % GROUPS * 8 : 0;
        bn[0] = *reinterpret_cast<const float4*>(p.in_mul + c); bn[1] = *reinterpret_cast<const float4*>(p.in_mul + c + 4);
        bn[2] = *reinterpret_cast<const float4*>(p.in_add + c); bn[3] = *reinterpret_cast<const float4*>(p.in_add + c + 4);
    }
    const int mf = wave / KS, share = wave % KS;          // the first two layers: this wave's fragment of channels and share of the reduction
    const f32x4_t sc0 = *reinterpret_cast<const f32x4_t*>(p.scale[0] + mf * 16 + kq * 4), bi0 = *reinterpret_cast<const f32x4_t*>(p.bias[0] + mf * 16 + kq * 4);
    const unsigned char* const weights = reinterpret_cast<const unsigned char*>(p.wpack) + (size_t)wave * (TW * NPL * 1024) + lane * 16;
    half8_t ring[RD][NPL];
    auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int pl = 0; pl < NPL; pl++) ring[t % RD][pl] = *reinterpret_cast<const half8_t*>(weights + (t * NPL + pl) * 1024);
    };
#pragma unroll
    for (int t = 0; t < T0 && t < RD; t++) load(t);
    const f32x4_t sc1 = *reinterpret_cast<const f32x4_t*>(p.scale[1] + mf * 16 + kq * 4), bi1 = *reinterpret_cast<const f32x4_t*>(p.bias[1] + mf * 16 + kq * 4);
    const int oy = y0 + (mq >> 2), ox = x0 + (mq & 3);
    const bool pos_ok = oy < p.h && ox < p.w;
    typedef typename std::conditional<HS, half4_t, f32x4_t>::type res_t;
    [[maybe_unused]] res_t rv[2 * NPR];
    const bool add = !PROJ && p.res;
    if (add) {
        const store_t* res = reinterpret_cast<const store_t*>(p.res);
#pragma unroll
        for (int j = 0; j < 2 * NPR; j++) {
            const int ch = (wave + j * WAVES) * 16 + kq * 4;
            rv[j] = *reinterpret_cast<const res_t*>(res + (pos_ok && ch + 4 <= p.out_cp ? ((size_t)(p.res_off + oy) * p.res_wp + p.res_off + ox) * p.res_cp + ch : 0));
        }
    }
    constexpr int SBN = (PROJ ? 4 : 2) * OUT, SBT = (SBN + 511) / 512;   // scale and bias of the last layer (and the projection): through the LDS
    float sb_reg[SBT];
#pragma unroll
    for (int i = 0; i < SBT; i++) {
        const int at = tid + i * 512, c = at % OUT, which = at / OUT;
        const float* from = which == 0 ? p.scale[2] : which == 1 ? p.bias[2] : which == 2 ? p.scale[3] : p.bias[3];
        sb_reg[i] = at < SBN && c < p.out_cp ? from[c] : 0.f;
    }
#pragma unroll
    for (int t = T0; t < RD; t++) load(t);

    // ---- activation and operand conversion of the window ----
    float in_scale = 1.f, inv_in = 1.f;
    if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act[0]), &inv_in);
    auto convert = [&](auto kind_) __attribute__((always_inline)) {
        constexpr int KIND = decltype(kind_)::value;
        _Float16 hlo, hhi;
        const bool packed = act_half_exact(p.act[0], hlo, hhi);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const bool ok = ch_of[i] >= 0;
            float x[8];
            if constexpr (!HS) {
                x[0] = raw[i].a.x; x[1] = raw[i].a.y; x[2] = raw[i].a.z; x[3] = raw[i].a.w; x[4] = raw[i].b.x; x[5] = raw[i].b.y; x[6] = raw[i].b.z; x[7] = raw[i].b.w;
            } else if constexpr (SRC == 1) {
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = (float)raw[i][e];
            }
            if constexpr (SRC == 1) {
                const float m[8] = {bn[0].x, bn[0].y, bn[0].z, bn[0].w, bn[1].x, bn[1].y, bn[1].z, bn[1].w}, a[8] = {bn[2].x, bn[2].y, bn[2].z, bn[2].w, bn[3].x, bn[3].y, bn[3].z, bn[3].w};
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = x[e] * m[e] + a[e];
            }
            if constexpr (HS) {
                half8_t v = raw[i];
                if constexpr (SRC == 1) {
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = (_Float16)x[e];   // (what the batch-norm layer would have stored)
                }
                if (packed) {
                    v = ok ? act_half(v, hlo, hhi) : (half8_t)((_Float16)0.f);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = ok ? (_Float16)act_p16((float)v[e], p.act[0]) : (_Float16)0.f;
                }
                if (l_off[i] >= 0) *reinterpret_cast<half8_t*>(lds + l_off[i]) = v;
            } else {
                half8_t hi, lo;
                split8<KIND>(x, ok, p.act[0], in_scale, hi, lo);
                if (l_off[i] >= 0) {
                    *reinterpret_cast<half8_t*>(lds + l_off[i]) = hi;
                    *reinterpret_cast<half8_t*>(lds + IN_PLANE + l_off[i]) = lo;
                }
            }
        }
    };
    if (HS || p.act[0].kind == ACT_LEAKY || p.act[0].kind == ACT_CLIP) convert(std::integral_constant<int, ACT_LEAKY>());
    else if (p.act[0].kind == ACT_RELU) convert(std::integral_constant<int, ACT_RELU>());
    else convert(std::integral_constant<int, ACT_NONE>());
    if (blockIdx.x == 0) range_clear(p.reset[0], p.reset[1], p.reset[2], p.reset[3], p.nreset);
    lds_barrier();   // the window is staged

    // A pass of the operand split (hi*hi, lo*hi, hi*lo) of a step, 32 products per output of one fragment of channels (the
    // stream's t-th) and one of positions.  (Successive instructions on one accumulator wait for each other: where a wave
    // has few of them, the passes have accumulators of their own.)
    auto mac = [&](f32x4_t& acc, int t, const half8_t (&b)[NPL], int pass) __attribute__((always_inline)) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[t % RD][pass == 1 ? NPL - 1 : 0], b[pass == 2 ? NPL - 1 : 0], acc, 0, 0, 0);
    };
    auto refill = [&](int t) __attribute__((always_inline)) {
        if (t + RD < TW) load(t + RD);
    };
    auto fetch = [&](half8_t (&b)[NPL], const unsigned char* at, int plane) __attribute__((always_inline)) {
#pragma unroll
        for (int pl = 0; pl < NPL; pl++) b[pl] = *reinterpret_cast<const half8_t*>(at + pl * plane);
    };

    // ---- first layer: 1x1 on the window ----
    f32x4_t acc0[NPF];
    {
        const unsigned char* base[NPF];
        half8_t b[2][NPF][NPL];
#pragma unroll
        for (int nf = 0; nf < NPF; nf++) {
            acc0[nf] = (f32x4_t)(0.f);
            base[nf] = lds + min(nf * 16 + mq, NWIN - 1) * IN_PIT + kq * 16 + share * 64;
            fetch(b[0][nf], base[nf], IN_PLANE);
        }
#pragma unroll
        for (int t = 0; t < T0; t++) {
            if (t + 1 < T0)
#pragma unroll
                for (int nf = 0; nf < NPF; nf++)
                    if (C0 % KS == 0 || share + (t + 1) * KS < C0) fetch(b[(t + 1) & 1][nf], base[nf] + (t + 1) * KS * 64, IN_PLANE);
            if (C0 % KS == 0 || share + t * KS < C0)
#pragma unroll
                for (int i = 0; i < NPASS; i++)
#pragma unroll
                    for (int nf = 0; nf < NPF; nf++) mac(acc0[nf], t, b[t & 1][nf], i);
            refill(t);
        }
    }
#pragma unroll
    for (int i = 0; i < SBT; i++)
        if (tid + i * 512 < SBN) reinterpret_cast<float*>(lds + SB)[tid + i * 512] = sb_reg[i];
    // The shares of a fragment meet: each wave of a fragment finishes some of its positions.
    constexpr int OWN = (NPF + KS - 1) / KS;
    if constexpr (KS > 1) {
#pragma unroll
        for (int nf = 0; nf < NPF; nf++) *reinterpret_cast<f32x4_t*>(lds + RED + (wave * NPF + nf) * 1024 + lane * 16) = acc0[nf];
        lds_barrier();
#pragma unroll
        for (int j = 0; j < OWN; j++) {
            const int nf = min(share + j * KS, NPF - 1);
            acc0[j] = (f32x4_t)(0.f);
#pragma unroll
            for (int k = 0; k < KS; k++) acc0[j] += *reinterpret_cast<const f32x4_t*>(lds + RED + ((mf * KS + k) * NPF + nf) * 1024 + lane * 16);
        }
    }
    {
        const MidAct act(p.act[1]);
        const float mul = p.acc_mul[0] * inv_in;
        float top = 0.f;
        half4_t hv[OWN];
#pragma unroll
        for (int j = 0; j < OWN; j++) {
            const int idx = (share + j * KS) * 16 + mq, wy = idx / WIN, wx = idx - wy * WIN;
            // (window positions outside the layer's output are its zero padding)
            const bool inside = idx < NWIN && (unsigned)(y0 - 1 + wy) < (unsigned)p.h && (unsigned)(x0 - 1 + wx) < (unsigned)p.w;
            f32x4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc0[j][e] * (sc0[e] * mul) + bi0[e];
            if constexpr (HS) {
#pragma unroll
                for (int e = 0; e < 4; e++) hv[j][e] = (_Float16)v[e];   // (as the layer would have stored it)
                hv[j] = inside ? act(hv[j]) : (half4_t)((_Float16)0.f);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    acc0[j][e] = inside ? act(v[e]) : 0.f;
                    top = fmaxf(top, inside ? fabsf(v[e]) : 0.f);   // (in front of the activation, whose clamp makes a number of a NaN)
                }
            }
        }
        float s = 1.f;
        if constexpr (!HS) {   // the operand split needs the window's largest magnitude (range.h), as the layer's word would give the tensor's
            top = range_wave_max(top);
            if (lane == 0) atomicMax(&box[0], __float_as_uint(top));
            lds_barrier();
            float unused;
            s = range_scale(range_after_act(__uint_as_float(box[0]), p.act[1]), &unused);
        }
#pragma unroll
        for (int j = 0; j < OWN; j++) {
            const int idx = (share + j * KS) * 16 + mq;
            if (idx >= NWIN) continue;
            unsigned char* const to = lds + MID + idx * MID_PIT + (mf * 16 + kq * 4) * 2;
            if constexpr (HS) {
                *reinterpret_cast<half4_t*>(to) = hv[j];
            } else {
                uint2 hi, lo;
                split_pair(acc0[j][0], acc0[j][1], s, hi.x, lo.x);
                split_pair(acc0[j][2], acc0[j][3], s, hi.y, lo.y);
                *reinterpret_cast<uint2*>(to) = hi;
                *reinterpret_cast<uint2*>(to + MID_PLANE) = lo;
            }
        }
    }
    lds_barrier();   // the first layer's result is there

    // ---- second layer: 3x3 on the tile ----
    f32x4_t acc1 = (f32x4_t)(0.f);
    {
        constexpr int CH = NPASS == 1 ? 2 : NPASS;   // accumulators
        f32x4_t part[CH];
#pragma unroll
        for (int i = 0; i < CH; i++) part[i] = (f32x4_t)(0.f);
        const unsigned char* const base = lds + MID + ((mq >> 2) * WIN + (mq & 3)) * MID_PIT + kq * 16;
        auto at = [&](int t) __attribute__((always_inline)) {
            const int step = share + t * KS, tap = step / CM, c = step % CM, ky = (tap * 11) >> 5;   // (tap / 3)
            return base + (ky * WIN + tap - 3 * ky) * MID_PIT + c * 64;
        };
        constexpr int LA = 3;   // steps that their positions are requested ahead
        half8_t b[LA + 1][NPL];
#pragma unroll
        for (int t = 0; t < LA && t < T1; t++)
            if (S1 % KS == 0 || share + t * KS < S1) fetch(b[t], at(t), MID_PLANE);
#pragma unroll
        for (int t = 0; t < T1; t++) {
            if (t + LA < T1 && (S1 % KS == 0 || share + (t + LA) * KS < S1)) fetch(b[(t + LA) % (LA + 1)], at(t + LA), MID_PLANE);
            if (S1 % KS == 0 || share + t * KS < S1)
#pragma unroll
                for (int i = 0; i < NPASS; i++) mac(part[NPASS == 1 ? t % 2 : i], T0 + t, b[t % (LA + 1)], i);
            refill(T0 + t);
        }
#pragma unroll
        for (int i = 0; i < CH; i++) acc1 += part[i];
    }
    if constexpr (KS > 1) {
        *reinterpret_cast<f32x4_t*>(lds + RED + wave * 1024 + lane * 16) = acc1;
        lds_barrier();
        acc1 = (f32x4_t)(0.f);
#pragma unroll
        for (int k = 0; k < KS; k++) acc1 += *reinterpret_cast<const f32x4_t*>(lds + RED + (mf * KS + k) * 1024 + lane * 16);
    }
    float inv_mid = 1.f, inv_mid2 = 1.f;
    {
        const MidAct act(p.act[2]);
        if constexpr (!HS) (void)range_scale(range_after_act(__uint_as_float(box[0]), p.act[1]), &inv_mid);
        const float mul = p.acc_mul[1] * inv_mid;
        f32x4_t v;
        half4_t hv;
        float top = 0.f, s = 1.f;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = acc1[e] * (sc1[e] * mul) + bi1[e];
        if constexpr (HS) {
#pragma unroll
            for (int e = 0; e < 4; e++) hv[e] = (_Float16)v[e];
            hv = pos_ok ? act(hv) : (half4_t)((_Float16)0.f);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                top = fmaxf(top, pos_ok ? fabsf(v[e]) : 0.f);
                v[e] = pos_ok ? act(v[e]) : 0.f;
            }
            top = range_wave_max(top);
            if (lane == 0) atomicMax(&box[1], __float_as_uint(top));
            lds_barrier();
            s = range_scale(range_after_act(__uint_as_float(box[1]), p.act[2]), &inv_mid2);
        }
        if (share == 0) {   // (every wave of a fragment has the sum)
            unsigned char* const to = lds + MID2 + mq * MID_PIT + (mf * 16 + kq * 4) * 2;
            if constexpr (HS) {
                *reinterpret_cast<half4_t*>(to) = hv;
            } else {
                uint2 hi, lo;
                split_pair(v[0], v[1], s, hi.x, lo.x);
                split_pair(v[2], v[3], s, hi.y, lo.y);
                *reinterpret_cast<uint2*>(to) = hi;
                *reinterpret_cast<uint2*>(to + M2_PLANE) = lo;
            }
        }
    }
    lds_barrier();   // the second layer's result is there

    // ---- third layer: 1x1, and the projection of the input; two fragments of output channels at a time ----
    float vmax = 0.f;
    const unsigned char* const base2 = lds + MID2 + mq * MID_PIT + kq * 16;
    const unsigned char* const base3 = lds + (((mq >> 2) + 1) * WIN + (mq & 3) + 1) * IN_PIT + kq * 16;
    const float mul2 = p.acc_mul[2] * inv_mid2, mul3 = p.acc_mul[3] * inv_in;
    store_t* const out = reinterpret_cast<store_t*>(p.out);
    half8_t b2[CM][NPL];
#pragma unroll
    for (int c = 0; c < CM; c++) fetch(b2[c], base2 + c * 64, M2_PLANE);
#pragma unroll
    for (int pr = 0; pr < NPR; pr++) {
        constexpr int T01 = T0 + T1;
        f32x4_t part[2][NPASS];
        [[maybe_unused]] f32x4_t partp[2][NPASS];
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int i = 0; i < NPASS; i++) part[f][i] = partp[f][i] = (f32x4_t)(0.f);
        auto step = [&](f32x4_t (&to)[2][NPASS], int t, const half8_t (&b)[NPL]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NPASS; i++)
#pragma unroll
                for (int f = 0; f < 2; f++) mac(to[f][i], t + f, b, i);
            refill(t); refill(t + 1);
        };
#pragma unroll
        for (int c = 0; c < CM; c++) step(part, T01 + pr * (T2 + T3) + 2 * c, b2[c]);
        if constexpr (PROJ) {
#pragma unroll
            for (int c = 0; c < C0; c++) {
                half8_t b3[NPL];
                fetch(b3, base3 + c * 64, IN_PLANE);
                step(partp, T01 + pr * (T2 + T3) + T2 + 2 * c, b3);
            }
        }
        f32x4_t acc[2];
        [[maybe_unused]] f32x4_t accp[2];
#pragma unroll
        for (int f = 0; f < 2; f++) {
            acc[f] = part[f][0]; accp[f] = partp[f][0];
#pragma unroll
            for (int i = 1; i < NPASS; i++) { acc[f] += part[f][i]; accp[f] += partp[f][i]; }
        }
#pragma unroll
        for (int f = 0; f < 2; f++) {
            const int ch = (wave + (2 * pr + f) * WAVES) * 16 + kq * 4;
            const bool ok = pos_ok && ch + 4 <= p.out_cp;
            const float* const sb = reinterpret_cast<const float*>(lds + SB) + ch;
            const f32x4_t sc = *reinterpret_cast<const f32x4_t*>(sb), bi = *reinterpret_cast<const f32x4_t*>(sb + OUT);
            f32x4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc[f][e] * (sc[e] * mul2) + bi[e];
            if constexpr (PROJ) {
                const f32x4_t scp = *reinterpret_cast<const f32x4_t*>(sb + 2 * OUT), bip = *reinterpret_cast<const f32x4_t*>(sb + 3 * OUT);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float r = accp[f][e] * (scp[e] * mul3) + bip[e];
                    if (p.res_scale) r *= sc[e];
                    v[e] += r;
                }
            } else if (add) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float r = (float)rv[2 * pr + f][e];
                    if (p.res_relu) r = fmaxf(r, 0.f);
                    if (p.res_scale) r *= sc[e];
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
    if (p.out_amax) range_publish_waves(p.out_amax, vmax, &box[2], WAVES);
}

typedef void (*b16_fn)(const ConvB16Params);
struct B16Entry {
    int f16, src, proj, c0, m, npr;
    size_t frags, lds;
    b16_fn fn;
};
template <bool HS, int SRC, bool PROJ, int C0, int M, int NPR>
constexpr B16Entry b16_entry() {
    constexpr int npl = HS ? 1 : 2, ks = WAVES / M, cm = M / 2;
    return B16Entry{HS, SRC, PROJ, C0, M, NPR,
                    (size_t)WAVES * ((C0 + ks - 1) / ks + (9 * cm + ks - 1) / ks + NPR * 2 * (cm + (PROJ ? C0 : 0))),
                    (size_t)npl * (NWIN * (C0 * 64 + 16) + (NWIN + 16) * (cm * 64 + 16)) + (ks > 1 ? WAVES * NPF * 1024 : 0) + (PROJ ? 4 : 2) * 2 * NPR * WAVES * 16 * 4,
                    conv_b16_kernel<HS, SRC, PROJ, C0, M, NPR>};
}
#define B16_BOTH(SRC, PROJ, C0, M, NPR) b16_entry<false, SRC, PROJ, C0, M, NPR>(), b16_entry<true, SRC, PROJ, C0, M, NPR>()
const B16Entry kB16[] = {
    B16_BOTH(0, true, 2, 4, 1), B16_BOTH(0, false, 8, 4, 1), B16_BOTH(1, false, 8, 4, 1),
    b16_entry<true, 0, false, 16, 8, 2>(), b16_entry<true, 1, false, 16, 8, 2>(),   // (fp32 tensors: 1.1 MB of weights per workgroup, 18 us against 15 apart at 28x28)
};
const B16Entry* find_b16(const ConvB16Params& p) {
    for (const B16Entry& e : kB16)
        if (e.f16 == (p.f16 ? 1 : 0) && e.src == (p.in_mul ? 1 : 0) && e.proj == (p.proj ? 1 : 0) && e.c0 == p.chunks && e.m == p.mid && e.npr * 2 * WAVES * 16 >= p.out_cp && e.npr * 2 * WAVES * 16 < p.out_cp + 256) return &e;
    return nullptr;
}
}  // namespace

size_t conv_b16_weight_frags(const ConvB16Params& p) {
    const B16Entry* e = find_b16(p);
    return e ? e->frags : 0;
}
size_t conv_b16_lds_bytes(const ConvB16Params& p) {
    const B16Entry* e = find_b16(p);
    return e ? e->lds : 0;
}

int launch_conv_b16(const ConvB16Params& p, hipStream_t s) {
    const B16Entry* e = find_b16(p);
    if (!e) return -1;
    const long long tiles = (long long)p.tiles_x * p.tiles_y;
    if (!p.in || !p.out || !p.wpack || p.in_cp % 8 != 0 || p.in_cp < 8 || p.in_cp > p.chunks * KC || p.h < 1 || p.w < 1 || p.in_off < 0 || p.h + p.in_off > p.in_hp || p.w + p.in_off > p.in_wp ||
        (long long)p.in_hp * p.in_wp * p.in_cp > (1ll << 30) || p.out_cp % 4 != 0 || p.out_cp < 4 || (p.res && (p.proj || p.res_cp < p.out_cp || p.res_cp % 4 != 0)) ||
        p.tiles_x != (p.w + TILE - 1) / TILE || p.tiles_y != (p.h + TILE - 1) / TILE || tiles > (1 << 20) || p.nreset < 0 || p.nreset > 4 || (p.in_mul != nullptr) != (p.in_add != nullptr))
        return -5;
    if (ensure_lds(reinterpret_cast<const void*>(e->fn), e->lds) != 0) return -2;
    hipLaunchKernelGGL(e->fn, dim3((unsigned)tiles), dim3(512), e->lds, s, p);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace fynhip
