// 1x1 convolutions on many positions with few channels (up to 128 in, 64 out): the layers of decoders at image size
// (reference: gpu/deep/deepconvlayer1x1.cpp:67-117), and the arg-max over the channels of such a layer's result
// (gpu/deep/deepargmaxlayer.cpp:113-152).
//
// Such a layer is a copy with arithmetic on the way: what bounds it is the tensors' traffic, and what keeps a kernel from
// that bound is having too few bytes on their way.  conv_d16 (conv_d16.hip) ends a wave after 16 positions -- address,
// one load, one result, one memory latency each.  Here waves stay: the layer's weights lie in registers, a wave takes U
// times 16 positions per trip and requests the next trip's values before it multiplies this one's, and workgroups walk
// bands of positions per XCD.  Measured on fp16 tensors (against conv_d16, conv_mfma): 32 -> 21 channels at
// 644x484 14.7 -> 8.5 us (35 MB: 4.1 TB/s), with the arg-max behind it 23.6 -> 15.2; 96 -> 32 at 322x242 10.6 -> 6.7.
// The arg-max works on the values as they are stored: a lane compares its channels in rising order, the four lanes of a
// position then meet in two steps (larger value, lower index among equals).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kernels.h"
#include "p16_common.h"
#include "range.h"

namespace fynhip {

namespace {
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// NS = chunks of 32 input channels, FR = fragments of 16 output channels (a wave computes all of them).
template <bool HS, int NS, int FR, bool ARG>
__global__ __launch_bounds__(256, 2) void conv_s16_kernel(const ConvP16Params p, const ArgMaxTail tail) {
    constexpr int NPL = HS ? 1 : 2, NPASS = HS ? 1 : 3;
    constexpr int U = NS == 1 ? 4 : (HS || NS == 2) ? 2 : 1;
    typedef typename std::conditional<HS, _Float16, float>::type store_t;
    typedef float f32x8_t __attribute__((ext_vector_type(8)));
    typedef typename std::conditional<HS, half8_t, f32x8_t>::type raw_t;
    typedef typename std::conditional<HS, half4_t, f32x4_t>::type out_t;
    if (blockIdx.x == 0) range_clear(p.reset[0], p.reset[1], p.reset[2], p.reset[3], p.nreset);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mq = lane & 15, kq = lane >> 4;
    const unsigned range_bits = p.in_amax ? range_load(p.in_amax) : 0u;

    // this wave's trips of U * 16 positions: a band per XCD, the band's trips dealt to the XCD's waves
    const int npos = p.npos_y * p.npos_x, trips = (npos + 16 * U - 1) / (16 * U);
    const int bands = min(8, (int)gridDim.x), band = (int)blockIdx.x & 7;
    const int band_waves = (((int)gridDim.x - band + 7) >> 3) * 4;
    const int trip_end = (int)((long long)trips * (band + 1) / bands);
    int trip = (int)((long long)trips * band / bands) + ((int)blockIdx.x >> 3) * 4 + wave;

    auto place = [&](int pos, int& py, int& px) {
        // (the reciprocal of the row length comes with the launch, one step of correction makes the quotient exact)
        if (npos <= (1 << 22)) {
            py = (int)(((float)pos + 0.5f) * p.rcp_tiles_x);
            px = pos - py * p.npos_x;
            if (px < 0) { py--; px += p.npos_x; }
            else if (px >= p.npos_x) { py++; px -= p.npos_x; }
        } else {
            py = pos / p.npos_x;
            px = pos - py * p.npos_x;
        }
    };
    const store_t* in = reinterpret_cast<const store_t*>(p.in);
    raw_t raw[U][NS];
    int ys[U], xs[U];   // where the values in `raw` come from
    auto fetch = [&](int t) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            place(min((t * U + u) * 16 + mq, npos - 1), ys[u], xs[u]);
            const store_t* src = in + ((size_t)(ys[u] * p.stride + p.in_y0) * p.in_wp + xs[u] * p.stride + p.in_x0) * p.in_cp + kq * 8;
#pragma unroll
            for (int s = 0; s < NS; s++)   // (channels behind the pitch: the pixel's last ones, which meet zero weights)
                raw[u][s] = *reinterpret_cast<const raw_t*>(s < NS - 1 || s * 32 + kq * 8 < p.in_cp ? src + s * 32 : src + (p.in_cp - 8 - kq * 8));
        }
    };
    if (trip < trip_end) fetch(trip);

    half8_t a[FR][NS][NPL];
#pragma unroll
    for (int f = 0; f < FR; f++)
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int pl = 0; pl < NPL; pl++)
                a[f][s][pl] = *reinterpret_cast<const half8_t*>(reinterpret_cast<const unsigned char*>(p.wpack) + ((f * NS + s) * NPL + pl) * 1024 + lane * 16);
    f32x4_t sc[FR], bi[FR];
#pragma unroll
    for (int f = 0; f < FR; f++) {
        sc[f] = *reinterpret_cast<const f32x4_t*>(p.scale + f * 16 + kq * 4);
        bi[f] = *reinterpret_cast<const f32x4_t*>(p.bias + f * 16 + kq * 4);
    }
    float in_scale = 1.f, inv_in_scale = 1.f;
    if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act), &inv_in_scale);
    const float acc_mul = p.acc_mul * inv_in_scale;
    _Float16 hlo, hhi;
    const bool half_act = HS && act_half_exact(p.act, hlo, hhi);
    const bool pad_lane = (NS - 1) * 32 + kq * 8 >= p.in_cp;   // the last chunk's group lies behind the pitch

    float vmax = 0.f;
    while (trip < trip_end) {
        half8_t b[U][NS][NPL];
        int py[U], px[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            py[u] = ys[u];
            px[u] = xs[u];
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const bool ok = !(s == NS - 1 && pad_lane);
                if constexpr (HS) {
                    if (half_act) {
                        b[u][s][0] = ok ? act_half(raw[u][s], hlo, hhi) : (half8_t)((_Float16)0.f);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e++) b[u][s][0][e] = ok ? (_Float16)act_p16((float)raw[u][s][e], p.act) : (_Float16)0.f;
                    }
                } else {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) x[e] = __builtin_amdgcn_fmed3f(raw[u][s][e], ok ? p.act.lo : 0.f, ok ? p.act.hi : 0.f);
                    if (p.act.leak != 0.f) {
#pragma unroll
                        for (int e = 0; e < 8; e++) x[e] += ok ? p.act.leak * fminf(raw[u][s][e], 0.f) : 0.f;
                    }
                    typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
                    u32x4_t H, L;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        unsigned h, l;
                        split_pair(x[2 * e], x[2 * e + 1], in_scale, h, l);
                        H[e] = h;
                        L[e] = l;
                    }
                    b[u][s][0] = __builtin_bit_cast(half8_t, H);
                    b[u][s][NPL - 1] = __builtin_bit_cast(half8_t, L);
                }
            }
        }
        const int pos0 = trip * U * 16 + mq;
        trip += band_waves;
        if (trip < trip_end) fetch(trip);
#pragma unroll
        for (int u = 0; u < U; u++) {
            f32x4_t acc[FR];
#pragma unroll
            for (int f = 0; f < FR; f++) acc[f] = (f32x4_t)(0.f);
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int i = 0; i < NPASS; i++)
#pragma unroll
                    for (int f = 0; f < FR; f++)
                        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[f][s][i == 1 ? NPL - 1 : 0], b[u][s][i == 2 ? NPL - 1 : 0], acc[f], 0, 0, 0);
            const int pos = pos0 + u * 16;
            const bool okp = pos < npos;
            const size_t opos = ((size_t)(p.out_off_y + py[u]) * p.out_wp + p.out_off_x + px[u]) * p.out_cp + kq * 4;
            const size_t rpos = ((size_t)(p.res_off_y + py[u]) * p.res_wp + p.res_off_x + px[u]) * p.res_cp + kq * 4;
            [[maybe_unused]] float best = -INFINITY;
            [[maybe_unused]] int bidx = 0x7fffffff;
#pragma unroll
            for (int f = 0; f < FR; f++) {
                const bool okc = okp && f * 16 + kq * 4 + 4 <= p.out_cp;   // (the last fragment may reach beyond the channel pitch)
                f32x4_t v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = acc[f][e] * (sc[f][e] * acc_mul) + bi[f][e];
                if (p.res && okc) {
                    const out_t r4 = *reinterpret_cast<const out_t*>(reinterpret_cast<const store_t*>(p.res) + rpos + f * 16);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float r = (float)r4[e];
                        if (p.res_relu) r = fmaxf(r, 0.f);
                        if (p.res_scale) r *= sc[f][e];
                        v[e] += r;
                    }
                }
                out_t o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = (store_t)v[e];
                if (okc) *reinterpret_cast<out_t*>(reinterpret_cast<store_t*>(p.out) + opos + f * 16) = o;
                if constexpr (!HS) {
#pragma unroll
                    for (int e = 0; e < 4; e++) vmax = fmaxf(vmax, okc ? fabsf(v[e]) : 0.f);
                }
                if constexpr (ARG) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float x = (float)o[e];
                        if (tail.act.kind != ACT_NONE) x = fminf(tail.act.hi, fmaxf(tail.act.lo, x)) + tail.act.leak * fminf(x, 0.f);
                        const int c = f * 16 + kq * 4 + e;
                        const bool up = c < tail.channels && x > best;
                        best = up ? x : best;
                        bidx = up ? c : bidx;
                    }
                }
            }
            if constexpr (ARG) {
#pragma unroll
                for (int step = 16; step <= 32; step *= 2) {
                    const float ob = __shfl_xor(best, step, 64);
                    const int oi = __shfl_xor(bidx, step, 64);
                    if (ob > best || (ob == best && oi < bidx)) {
                        best = ob;
                        bidx = oi;
                    }
                }
                if (okp && kq == 0) {
                    const out_t o = {(store_t)(float)bidx, (store_t)best, (store_t)0.f, (store_t)0.f};
                    *reinterpret_cast<out_t*>(reinterpret_cast<store_t*>(tail.out.ptr) + ((size_t)(py[u] + tail.out.pad) * tail.out.wp() + px[u] + tail.out.pad) * tail.out.cp) = o;
                    tail.idx[pos] = bidx;
                }
            }
        }
    }
    if (!HS && p.out_amax) range_publish_block256(p.out_amax, vmax);
}

typedef void (*s16_fn)(const ConvP16Params, const ArgMaxTail);
// (fp32 tensors: as many fragments as leave the weights room in the registers)
template <bool HS, int NS, int FR, bool ARG>
constexpr s16_fn s16_entry() {
    if constexpr (HS || NS * FR <= 8) return conv_s16_kernel<HS, NS, FR, ARG>;
    else return nullptr;
}
template <bool HS, int NS, bool ARG>
s16_fn pick_s16_fr(int fr) {
    switch (fr) {
        case 1: return s16_entry<HS, NS, 1, ARG>();
        case 2: return s16_entry<HS, NS, 2, ARG>();
        case 3: return s16_entry<HS, NS, 3, ARG>();
        case 4: return s16_entry<HS, NS, 4, ARG>();
        default: return nullptr;
    }
}
template <bool HS, bool ARG>
s16_fn pick_s16(int chunks, int fr) {
    switch (chunks) {
        case 1: return pick_s16_fr<HS, 1, ARG>(fr);
        case 2: return pick_s16_fr<HS, 2, ARG>(fr);
        case 3: return pick_s16_fr<HS, 3, ARG>(fr);
        case 4: return pick_s16_fr<HS, 4, ARG>(fr);
        default: return nullptr;
    }
}
s16_fn pick(bool half, bool arg, int chunks, int fr) {
    if (half) return arg ? pick_s16<true, true>(chunks, fr) : pick_s16<true, false>(chunks, fr);
    return arg ? pick_s16<false, true>(chunks, fr) : pick_s16<false, false>(chunks, fr);
}
}  // namespace

bool conv_s16_supported(int k, int dil, int in_cp, int cout, int out_cp, bool f16) {
    return k == 1 && dil == 1 && in_cp % 8 == 0 && in_cp >= 8 && in_cp <= 128 && cout >= 4 && cout <= 64 && out_cp % 4 == 0 && out_cp >= cout &&
           pick(f16, false, (in_cp + 31) / 32, (cout + 15) / 16) != nullptr;
}

// p.cin_chunks = chunks of 32 input channels, p.mfrags = fragments of 16 output channels (scale and bias hold 16*mfrags
// values, wpack as for launch_conv_d16), in_y0 / in_x0 = input padding, p.stride = pixel step per position
int launch_conv_s16(const ConvP16Params& p, const ArgMaxTail& tail, hipStream_t s) {
    const s16_fn fn = pick(p.f16 != 0, tail.idx != nullptr, p.cin_chunks, p.mfrags);
    if (!fn) return -1;
    const long long npos = (long long)p.npos_y * p.npos_x;
    if (npos < 1 || npos > (1ll << 28) || p.in_cp % 8 != 0 || p.in_cp > 32 * p.cin_chunks || p.in_cp <= 32 * (p.cin_chunks - 1) || p.stride < 1 || p.in_clamp || p.in_y0 < 0 || p.in_x0 < 0 ||
        (long long)(p.npos_y - 1) * p.stride + p.in_y0 >= p.in_hp || (long long)(p.npos_x - 1) * p.stride + p.in_x0 >= p.in_wp || p.out_cp % 4 != 0 || p.out_cp < 4 ||
        (p.res && (p.res_cp < p.out_cp || p.res_cp % 4 != 0)) || p.nreset < 0 || p.nreset > 4 || p.dw_in || p.in_mul || p.in2)
        return -5;
    if (tail.idx && (!tail.out.ptr || tail.out.cp < 4 || tail.out.h != p.npos_y || tail.out.w != p.npos_x || tail.channels < 1 || tail.channels > 16 * p.mfrags)) return -5;
    ConvP16Params q = p;
    q.rcp_tiles_x = 1.0f / (float)p.npos_x;   // (this kernel's use of the field: the reciprocal of a row of positions)
    // (four workgroups per CU where the registers allow it; every wave the same number of trips)
    const int u = p.cin_chunks == 1 ? 4 : (p.f16 || p.cin_chunks == 2) ? 2 : 1;
    const long long trips = (npos + 16 * u - 1) / (16 * u), per = (trips + 4095) / 4096;
    unsigned wgs = (unsigned)((trips + 4 * per - 1) / (4 * per));
    if (wgs > 8) wgs = (wgs + 7) / 8 * 8;
    hipLaunchKernelGGL(fn, dim3(wgs), dim3(256), 0, s, q, tail);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace fynhip
