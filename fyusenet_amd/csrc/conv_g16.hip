// 3x3 convolutions between tensors of few channels (16 to 64 in, up to 64 out), any stride, edge rule and source step:
// layers at image size like those of small style nets and decoders (reference:
// gpu/vanilla/convlayerNxN_vanilla.cpp, gpu/vanilla/fractionalconvlayerNxN_vanilla.cpp, gpu/deep/deepconvlayerNxN.cpp:129-211).
//
// The forms that stage pixels in LDS (conv_p16.hip) work on chunks of 32 input channels and blocks of 64 output
// channels: 12 -> 20 channels fill a seventh of that, 40 -> 40 two fifths.  Here a step of the matrix instruction
// (v_mfma_f32_16x16x32_f16, 16 positions
// x 32 values of the reduction) is four groups of eight channels wherever they lie: the window's 9 * G groups (G = groups
// per pixel) are numbered tap by tap, lane group kq of step s takes group 4s + kq straight from the tensor, and only the
// last step is padded (40 channels: 12 steps instead of 18, 16 channels: 5 instead of 9).  The window's nine-fold
// overlap is left to the L1.  A wave owns 16 positions at a time and all its fragments of output channels; the weights
// lie in LDS, staged once per workgroup; the registers a step has emptied take the next tile's values at once, so a
// whole tile of loads is always in flight and no barrier stands in the loop.  Workgroups walk bands of positions per XCD.
// Bound: the L1's rate at the nine-fold window on large layers, memory latency on small ones.  24 -> 12 channels at step
// 1/4, 312x256 positions, fp32 tensors: 11.4 us where the general forms take 14.4 (7.4 MB: 0.6 TB/s, matrix pipes 7 %
// busy).  960x540 positions, fp16: 16 -> 16 channels 18.2 us against 22.2, 24 -> 24 25.3 against 27.8.  Behind from 40
// channels on (each output fragment's waves fetch the window again where registers do not hold all fragments): 64 -> 64 at
// 256x256, fp32, 79.8 us against 11.8.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "p16_common.h"
#include "range.h"

namespace fynhip {

namespace {
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// G = groups of 8 channels per pixel, FR = fragments of 16 output channels per wave.
template <bool HS, int G, int FR>
__global__ __launch_bounds__(256, 2) void conv_g16_kernel(const ConvP16Params p) {
    constexpr int NS = (9 * G + 3) / 4, NPL = HS ? 1 : 2, NPASS = HS ? 1 : 3, ESZ = HS ? 2 : 4;
    typedef typename std::conditional<HS, _Float16, float>::type store_t;
    typedef float f32x8_t __attribute__((ext_vector_type(8)));
    typedef typename std::conditional<HS, half8_t, f32x8_t>::type raw_t;
    extern __shared__ __align__(16) unsigned char lds[];
    if ((blockIdx.x | blockIdx.y) == 0) range_clear(p.reset[0], p.reset[1], p.reset[2], p.reset[3], p.nreset);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mq = lane & 15, kq = lane >> 4;
    const unsigned range_bits = p.in_amax ? range_load(p.in_amax) : 0u;

    // this wave's tiles: a band per XCD (its rows then come into one L2), the band's tiles dealt to the XCD's waves
    const int npos = p.npos_y * p.npos_x, tiles = (npos + 15) >> 4;
    const int bands = min(8, (int)gridDim.x), band = (int)blockIdx.x & 7;
    const int band_waves = (((int)gridDim.x - band + 7) >> 3) * 4;
    const int tile_end = (int)((long long)tiles * (band + 1) / bands);
    int tile = (int)((long long)tiles * band / bands) + ((int)blockIdx.x >> 3) * 4 + wave;

    // where a lane's group of step s lies in the window: row, column and first channel, and (for windows inside the
    // frame) the byte offset from the window's first pixel
    int info[NS];
    unsigned ioff[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int g = min(4 * s + kq, 9 * G - 1), t = g / G, ty = t / 3;
        info[s] = ty | ((t - 3 * ty) << 2) | ((g - t * G) << 7);   // (channel of the group << 4)
        ioff[s] = (unsigned)(((ty * p.in_wp + (t - 3 * ty)) * p.in_cp + (g - t * G) * 8) * ESZ);
    }
    const bool pad_lane = 4 * (NS - 1) + kq >= 9 * G;   // the last step's group is padding
    const int vh = p.in_hp << p.in_shift, vw = p.in_wp << p.in_shift;   // the frame in which positions and taps count

    struct At {
        int y0, x0, py;  // the lane's window, the row of its position
        unsigned base;   // byte offset of its first pixel
        bool inside;     // every lane's window lies inside the frame (and no pixel is repeated)
    };
    auto locate = [&](int t) {
        const int pos = min(t * 16 + mq, npos - 1);
        // (the reciprocal of the row length comes with the launch, one step of correction makes the quotient exact)
        int py, px;
        if (npos <= (1 << 22)) {
            py = (int)(((float)pos + 0.5f) * p.rcp_tiles_x);
            px = pos - py * p.npos_x;
            if (px < 0) { py--; px += p.npos_x; }
            else if (px >= p.npos_x) { py++; px -= p.npos_x; }
        } else {
            py = pos / p.npos_x;
            px = pos - py * p.npos_x;
        }
        At a;
        a.py = py;
        a.y0 = py * p.stride + p.in_y0;
        a.x0 = px * p.stride + p.in_x0;
        const bool in = p.in_shift == 0 && a.y0 >= 0 && a.x0 >= 0 && a.y0 + 2 < vh && a.x0 + 2 < vw;
        a.inside = __builtin_amdgcn_ballot_w64(in) == ~0ull;
        a.base = (unsigned)((a.y0 * p.in_wp + a.x0) * p.in_cp * ESZ);
        return a;
    };
    // byte offsets of the window's groups and, one bit a step, whether they lie in the frame
    unsigned off[NS];
    auto aim = [&](const At& a) {
        if (a.inside) {
#pragma unroll
            for (int s = 0; s < NS; s++) off[s] = a.base + ioff[s];
            return ~0u;
        }
        unsigned okm = 0u;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int y = a.y0 + (info[s] & 3), x = a.x0 + ((info[s] >> 2) & 3);
            const int yc = min(max(y, 0), vh - 1), xc = min(max(x, 0), vw - 1);
            const bool ok = (p.in_clamp != 0) | ((y == yc) & (x == xc));
            okm |= ok ? 1u << s : 0u;
            off[s] = (unsigned)((__mul24(yc >> p.in_shift, p.in_wp) + (xc >> p.in_shift)) * p.in_cp + (info[s] >> 4)) * ESZ;
        }
        return okm;
    };
    auto fetch = [&](int s) { return *reinterpret_cast<const raw_t*>(reinterpret_cast<const char*>(p.in) + off[s]); };

    raw_t raw[NS];
    At at = locate(min(tile, tiles - 1));
    unsigned okm = aim(at);
#pragma unroll
    for (int s = 0; s < NS; s++) raw[s] = fetch(s);

    // the block's weights: [fragment][step][plane][lane][8 halves]
    const int f0 = (int)blockIdx.y * FR;
    {
        constexpr int BYTES = FR * NS * NPL * 1024;
        const unsigned char* src = reinterpret_cast<const unsigned char*>(p.wpack) + (size_t)f0 * NS * NPL * 1024;
#pragma unroll 6
        for (int o = tid * 16; o < BYTES; o += 4096) *reinterpret_cast<half8_t*>(lds + o) = *reinterpret_cast<const half8_t*>(src + o);
    }
    f32x4_t sc[FR], bi[FR];
#pragma unroll
    for (int f = 0; f < FR; f++) {
        sc[f] = *reinterpret_cast<const f32x4_t*>(p.scale + (f0 + f) * 16 + kq * 4);
        bi[f] = *reinterpret_cast<const f32x4_t*>(p.bias + (f0 + f) * 16 + kq * 4);
    }
    float in_scale = 1.f, inv_in_scale = 1.f;
    if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act), &inv_in_scale);
    const float acc_mul = p.acc_mul * inv_in_scale;
#pragma unroll
    for (int f = 0; f < FR; f++)
#pragma unroll
        for (int e = 0; e < 4; e++) sc[f][e] *= acc_mul;
    const float inv_acc_mul = p.res_scale ? 1.f / acc_mul : 0.f;   // (a power of two)
    _Float16 hlo, hhi;
    const bool half_act = HS && act_half_exact(p.act, hlo, hhi);
    lds_barrier();   // the weights are there

    float vmax = 0.f;
        while (tile < tile_end) {
            // (the weights of few steps and fragments stay in registers from tile to tile; more of them do not fit)
            if constexpr (NS * FR * NPL > 10) asm volatile("" ::: "memory");
            const int next = tile + band_waves;
            const bool more = next < tile_end;
            const At an = locate(min(next, tiles - 1));
            const unsigned okn = aim(an);
            f32x4_t acc[FR];
            half8_t a[2][FR][NPL];
#pragma unroll
            for (int f = 0; f < FR; f++) {
                acc[f] = (f32x4_t)(0.f);
#pragma unroll
                for (int pl = 0; pl < NPL; pl++) a[0][f][pl] = *reinterpret_cast<const half8_t*>(lds + (f * NS * NPL + pl) * 1024 + lane * 16);
            }
#pragma unroll
            for (int s = 0; s < NS; s++) {
                if (s + 1 < NS) {
#pragma unroll
                    for (int f = 0; f < FR; f++)
#pragma unroll
                        for (int pl = 0; pl < NPL; pl++)
                            a[(s + 1) & 1][f][pl] = *reinterpret_cast<const half8_t*>(lds + ((f * NS + s + 1) * NPL + pl) * 1024 + lane * 16);
                }
                const bool ok = ((okm >> s) & 1u) && !(s == NS - 1 && pad_lane);
                half8_t b[NPL];
                if constexpr (HS) {
                    if (half_act) {
                        b[0] = ok ? act_half(raw[s], hlo, hhi) : (half8_t)((_Float16)0.f);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e++) b[0][e] = ok ? (_Float16)act_p16((float)raw[s][e], p.act) : (_Float16)0.f;
                    }
                } else {
                    // (a clamp whose bounds collapse outside the frame; a leak is rare and costs its two instructions only then)
                    const float bottom = ok ? p.act.lo : 0.f, top = ok ? p.act.hi : 0.f;
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) x[e] = __builtin_amdgcn_fmed3f(raw[s][e], bottom, top);
                    if (p.act.leak != 0.f) {
                        const float leak = ok ? p.act.leak : 0.f;
#pragma unroll
                        for (int e = 0; e < 8; e++) x[e] += leak * (ok ? fminf(raw[s][e], 0.f) : 0.f);
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
                    b[0] = __builtin_bit_cast(half8_t, H);
                    b[NPL - 1] = __builtin_bit_cast(half8_t, L);
                }
                if (more) raw[s] = fetch(s);
#pragma unroll
                for (int i = 0; i < NPASS; i++)
#pragma unroll
                    for (int f = 0; f < FR; f++)
                        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[s & 1][f][i == 1 ? NPL - 1 : 0], b[i == 2 ? NPL - 1 : 0], acc[f], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            const int pos = tile * 16 + mq;
            const bool okp = pos < npos;
            {
                const int pc = okp ? pos : npos - 1;
                const int py = at.py, px = pc - py * p.npos_x;
                const store_t* res = reinterpret_cast<const store_t*>(p.res);
                store_t* out = reinterpret_cast<store_t*>(p.out);
                const size_t rpos = ((size_t)(p.res_off_y + py) * p.res_wp + p.res_off_x + px) * p.res_cp + kq * 4;
                const size_t opos = ((size_t)(p.out_off_y + py) * p.out_wp + p.out_off_x + px) * p.out_cp + kq * 4;
#pragma unroll
                for (int f = 0; f < FR; f++) {
                    const int ch = (f0 + f) * 16;
                    const bool okc = okp && ch + kq * 4 + 4 <= p.out_cp;   // (the last fragment may reach beyond the channel pitch)
                    f32x4_t v;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = acc[f][e] * sc[f][e] + bi[f][e];
                    if (res && okc) {
                        float r[4];
                        if constexpr (HS) {
                            const half4_t rh = *reinterpret_cast<const half4_t*>(res + rpos + ch);
#pragma unroll
                            for (int e = 0; e < 4; e++) r[e] = (float)rh[e];
                        } else {
                            const f32x4_t rv = *reinterpret_cast<const f32x4_t*>(res + rpos + ch);
#pragma unroll
                            for (int e = 0; e < 4; e++) r[e] = rv[e];
                        }
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if (p.res_relu) r[e] = fmaxf(r[e], 0.f);
                            if (p.res_scale) r[e] *= sc[f][e] * inv_acc_mul;
                            v[e] += r[e];
                        }
                    }
                    if constexpr (HS) {
                        half4_t hv;
#pragma unroll
                        for (int e = 0; e < 4; e++) hv[e] = (_Float16)v[e];
                        if (okc) *reinterpret_cast<half4_t*>(out + opos + ch) = hv;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++) vmax = fmaxf(vmax, okc ? fabsf(v[e]) : 0.f);
                        if (okc) *reinterpret_cast<f32x4_t*>(out + opos + ch) = v;
                    }
                }
            }
            tile = next;
            at = an;
            okm = okn;
        }
    if (!HS && p.out_amax) range_publish_block256(p.out_amax, vmax);
}

typedef void (*g16_fn)(const ConvP16Params);
// (fp32 tensors: combinations whose window, weights and accumulators fit the registers)
template <bool HS, int G, int FR>
constexpr g16_fn g16_entry() {
    if constexpr (HS || G * FR <= (G <= 4 ? 16 : G == 5 ? 15 : G == 6 ? 12 : 8)) return conv_g16_kernel<HS, G, FR>;
    else return nullptr;
}
template <bool HS, int G>
g16_fn pick_g16_fr(int fr) {
    switch (fr) {
        case 1: return g16_entry<HS, G, 1>();
        case 2: return g16_entry<HS, G, 2>();
        case 3: return g16_entry<HS, G, 3>();
        case 4: return g16_entry<HS, G, 4>();
        default: return nullptr;
    }
}
template <bool HS>
g16_fn pick_g16(int groups, int fr) {
    switch (groups) {
        case 2: return pick_g16_fr<HS, 2>(fr);
        case 3: return pick_g16_fr<HS, 3>(fr);
        case 4: return pick_g16_fr<HS, 4>(fr);
        case 5: return pick_g16_fr<HS, 5>(fr);
        case 6: return pick_g16_fr<HS, 6>(fr);
        case 8: return pick_g16_fr<HS, 8>(fr);
        default: return nullptr;
    }
}
}  // namespace

int conv_g16_steps(int in_cp) { return (9 * (in_cp / 8) + 3) / 4; }
bool conv_g16_exists(const ConvP16Params& p) { return (p.f16 ? pick_g16<true>(p.in_cp / 8, p.wm) : pick_g16<false>(p.in_cp / 8, p.wm)) != nullptr; }
size_t conv_g16_lds_bytes(const ConvP16Params& p) { return (size_t)p.wm * conv_g16_steps(p.in_cp) * (p.f16 ? 1 : 2) * 1024; }
bool conv_g16_supported(int k, int dil, int in_cp, int cout, int out_cp) {
    return k == 3 && dil == 1 && in_cp % 8 == 0 && pick_g16<true>(in_cp / 8, 1) != nullptr && cout >= 4 && cout <= 64 && out_cp % 4 == 0 && out_cp >= cout;
}

// p.wm = fragments of 16 output channels per wave (1..4), p.cout_blocks = grid rows that share the p.mfrags fragments
// (scale, bias and wpack hold 16 * wm * cout_blocks rows; rows beyond out_cp are not stored), p.pos_groups = workgroups
// along the positions; in_y0 / in_x0 = stored coordinate of tap (0,0) of position (0,0) in the frame whose pixels are
// repeated 2^in_shift times, p.stride = step of a position in it; pixels outside repeat the edge (in_clamp) or are zeros.
int launch_conv_g16(const ConvP16Params& p, hipStream_t s) {
    if (p.in_cp < 16 || p.in_cp % 8 != 0) return -1;
    const g16_fn fn = p.f16 ? pick_g16<true>(p.in_cp / 8, p.wm) : pick_g16<false>(p.in_cp / 8, p.wm);
    if (!fn) return -1;
    const long long npos = (long long)p.npos_y * p.npos_x, in_bytes = (long long)p.in_hp * p.in_wp * p.in_cp * (p.f16 ? 2 : 4);
    if (npos < 1 || npos > (1ll << 28) || in_bytes > (1ll << 31) || p.mfrags != p.wm * p.cout_blocks || p.cout_blocks < 1 || p.cout_blocks > 4 || p.stride < 1 || p.pos_groups < 1 ||
        p.pos_groups > 65535 || p.out_cp % 4 != 0 || p.out_cp < 4 || (p.res && (p.res_cp < p.out_cp || p.res_cp % 4 != 0)) || p.nreset < 0 || p.nreset > 4 || p.dw_in || p.in_mul || p.in2 ||
        p.in_shift < 0 || p.in_shift > 8 || ((long long)p.in_hp << p.in_shift) > (1 << 30) || ((long long)p.in_wp << p.in_shift) > (1 << 30))
        return -5;
    const size_t lds = conv_g16_lds_bytes(p);
    if (lds > 160 * 1024 || ensure_lds(reinterpret_cast<const void*>(fn), lds) != 0) return -2;
    ConvP16Params q = p;
    q.rcp_tiles_x = 1.0f / (float)p.npos_x;   // (this kernel's use of the field: the reciprocal of a row of positions)
    hipLaunchKernelGGL(fn, dim3((unsigned)p.pos_groups, (unsigned)p.cout_blocks), dim3(256), lds, s, q);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace fynhip
