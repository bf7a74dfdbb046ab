// 3x3 convolutions between tensors of few channels (16 to 64 in, up to 128 out) with the window of a tile in LDS: the layers
// of small style nets and decoders (reference: gpu/vanilla/convlayerNxN_vanilla.cpp,
// gpu/vanilla/fractionalconvlayerNxN_vanilla.cpp, gpu/deep/deepconvlayerNxN.cpp:129-211).
//
// As in conv_g16.hip a step of the matrix instruction (v_mfma_f32_16x16x32_f16: 16 positions x 32 values of the reduction)
// is four groups of eight channels wherever they lie in the window -- its 9 * G groups numbered tap by tap, lane group kq of
// step s takes group 4s + kq --, so 40 -> 40 channels take 12 steps and 3 fragments where the forms on chunks of 32 channels
// and blocks of 64 (conv_p16.hip) take 18 and 4.  But the window is fetched and converted once, into LDS, instead of nine
// times from the L1; a lane's address there is its position plus an offset that its step fixes.
//
// Such a layer is a launch's start, one memory round trip and about a microsecond of work, so everything is requested at
// once and nothing runs twice: a workgroup of four waves takes tiles of TH rows of sixteen positions and all output
// channels (a block of them where there are too few tiles for the chip); its waves all stage, then each takes every fourth step (its weights stay in registers from tile to tile: no
// two waves read the same ones, which is what a split by positions would cost), and the partial sums meet in LDS, where the
// fragments are dealt to the waves for the epilogue.  The next tile's window is requested before this one's matrix
// instructions.
// Measured (fp32 tensors, one launch): 12 -> 20 channels, step 2, at 312x256 positions 13.2 -> 11.0 us (conv_g16), at 24x32
// 6.4 -> 4.0 (conv_p16); 20 -> 40, step 2, at 12x16 6.0 -> 4.7 (conv_mfma); 40 -> 20 at step 1/2, 156x128 9.1 -> 7.6, 12x16
// 7.4 -> 5.0; 20 -> 12 at step 1/4, 24x32 5.8 -> 3.8; 40 -> 40 at 156x128 with a residual 8.2 -> 8.0; 64 -> 64 at
// 56x56 5.7 -> 5.2 (conv_kr16, whose waves split whole chunks of 32 channels: two of four had none).  The samples' 3x3 style
// net on a 64x48 frame 77-78 -> 70-71 us.  Bound: a launch's start and its memory round trip (a microsecond of matrix
// instructions in 40 -> 40 at 156x128), on large images the conversion and the partial sums beside them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "p16_common.h"
#include "range.h"

namespace fynhip {

namespace {
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// HS: fp16 tensors, G: groups of 8 channels per input pixel, FR: fragments of 16 output channels, S: input step per
// position (in the frame whose pixels are repeated 2^in_shift times), TH: rows of a tile
template <bool HS_, int G_, int FR_, int S_, int TH_>
struct GeoN {
    static constexpr bool HS = HS_;
    static constexpr int G = G_, FR = FR_, S = S_, TH = TH_;
    static constexpr int NS = (9 * G + 3) / 4, SPW = (NS + 3) / 4;      // steps, steps per wave
    static constexpr int NPL = HS ? 1 : 2, NPASS = HS ? 1 : 3, ESZ = HS ? 2 : 4;
    static constexpr int HW = S * 15 + 3, HH = S * (TH - 1) + 3;        // the window of a tile
    // bytes of a staged pixel and plane: an odd number of 16-byte pieces, so that eight neighbouring positions' reads
    // start in eight different pieces of the 128 bytes of the banks; with a step of two, even and odd columns apart
    static constexpr int PXB = (G % 2 ? G : G + 1) * 16;
    static constexpr int HALF = (HW + 1) / 2, SLOTS = S == 1 ? HW : 2 * HALF;
    static constexpr int ROWP = SLOTS * PXB, PLANE = HH * ROWP;
    static constexpr int NITEMS = HH * HW * G, NB = (NITEMS + 255) / 256;   // staging items: (pixel, 8 channels)
    static constexpr int NQ = FR * TH, NO = (NQ + 3) / 4;               // fragments of a tile, of a wave in the epilogue
    static constexpr int SUMS = NPL * PLANE;                            // the partial sums' place in LDS
    static constexpr int SB = SUMS + NQ * 3 * 1024;                     // scale and bias
    static constexpr int LDS = SB + FR * 128;
    __host__ __device__ static constexpr int slot(int c) { return S == 1 ? c : (c & 1) * HALF + (c >> 1); }
    static_assert(NPL * PLANE < 65536, "offsets fit the LDS instructions' immediate field");
};

template <class N>
__global__ __launch_bounds__(256, 2) void conv_p16n_kernel(const ConvP16Params p) {
    constexpr int G = N::G, FR = N::FR, S = N::S, TH = N::TH, NS = N::NS, SPW = N::SPW, NPL = N::NPL;
    constexpr bool HS = N::HS;
    typedef typename std::conditional<HS, _Float16, float>::type store_t;
    typedef float f32x8_t __attribute__((ext_vector_type(8)));
    typedef typename std::conditional<HS, half8_t, f32x8_t>::type raw_t;
    extern __shared__ __align__(16) unsigned char lds[];
    if ((blockIdx.x | blockIdx.y) == 0) range_clear(p.reset[0], p.reset[1], p.reset[2], p.reset[3], p.nreset);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mq = lane & 15, kq = lane >> 4;
    const unsigned range_bits = p.in_amax ? range_load(p.in_amax) : 0u;
    // Workgroups are dealt round-robin to the 8 XCDs; remap so that neighbouring tiles (shared windows) meet in one L2.
    int group = blockIdx.x;
    {
        const int per = p.pos_groups >> 3;
        if (group < (per << 3)) group = (group & 7) * per + (group >> 3);
    }
    const int ntiles = p.tiles_x * p.tiles_y;
    const int ch0 = (int)blockIdx.y * FR * 16;   // this grid row's block of output channels

    // ---- staging
    int i_yx[N::NB], l_off[N::NB];   // an item's pixel inside the window (row << 16 | column << 3 | group), its place in LDS
#pragma unroll
    for (int i = 0; i < N::NB; i++) {
        const int idx = tid + i * 256, pix = idx / G, g = idx - pix * G, y = pix / N::HW, x = pix - y * N::HW;
        i_yx[i] = y << 16 | x << 3 | g;
        l_off[i] = idx < N::NITEMS ? y * N::ROWP + N::slot(x) * N::PXB + g * 16 : -1;
    }
    const int vh = p.in_hp << p.in_shift, vw = p.in_wp << p.in_shift;   // the frame in which positions and taps count
    raw_t raw[N::NB];
    unsigned inside = 0u;   // one bit an item
    // (unconditional loads: items outside the frame read the tensor's first element and are staged as zeros)
    auto fetch = [&](int tile) {
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        const int y0 = tyi * TH * S + p.in_y0, x0 = txi * 16 * S + p.in_x0;
        inside = 0u;
#pragma unroll
        for (int i = 0; i < N::NB; i++) {
            int y = y0 + (i_yx[i] >> 16), x = x0 + ((i_yx[i] >> 3) & 0x1fff);
            if (p.in_clamp) {
                y = min(max(y, 0), vh - 1);
                x = min(max(x, 0), vw - 1);
            }
            const bool ok = l_off[i] >= 0 && (unsigned)y < (unsigned)vh && (unsigned)x < (unsigned)vw;
            inside |= ok ? 1u << i : 0u;
            raw[i] = *reinterpret_cast<const raw_t*>(reinterpret_cast<const store_t*>(p.in) + (ok ? ((y >> p.in_shift) * p.in_wp + (x >> p.in_shift)) * p.in_cp + (i_yx[i] & 7) * 8 : 0));
        }
    };
    int tile = group;
    fetch(tile);

    // ---- this wave's steps: its weights, and where a lane's group lies in the window
    half8_t a[SPW][FR][NPL];
    int off[SPW];
#pragma unroll
    for (int s = 0; s < SPW; s++) {
        const int step = min(wave + 4 * s, NS - 1);
        const int g = min(4 * step + kq, 9 * G - 1), t = g / G, ty = t / 3, tx = t - 3 * ty;
        off[s] = ty * N::ROWP + (S == 1 ? mq + tx : (tx & 1) * N::HALF + mq + (tx >> 1)) * N::PXB + (g - t * G) * 16;
#pragma unroll
        for (int f = 0; f < FR; f++)
#pragma unroll
            for (int pl = 0; pl < NPL; pl++)
                a[s][f][pl] = *reinterpret_cast<const half8_t*>(reinterpret_cast<const unsigned char*>(p.wpack) + (((int)blockIdx.y * FR + f) * NS + step) * NPL * 1024 + pl * 1024 + lane * 16);
    }
    const bool last_step = wave + 4 * (SPW - 1) < NS;                  // whether the wave has one (the same for all lanes)
    const bool pad_lane = 4 * (wave + 4 * (SPW - 1)) + kq >= 9 * G;    // its group is padding: zeros, whatever lies there

    // ---- the fragments this wave finishes: number wave + 4 i, of FR x TH
    float in_scale = 1.f, inv_in_scale = 1.f;
    if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act), &inv_in_scale);
    const float acc_mul = p.acc_mul * inv_in_scale;
    if (tid < FR * 16) {
        reinterpret_cast<float*>(lds + N::SB)[tid] = p.scale[ch0 + tid];
        reinterpret_cast<float*>(lds + N::SB)[FR * 16 + tid] = p.bias[ch0 + tid];
    }
    const float res_floor = p.res_relu ? 0.f : -__builtin_inff();
    float vmax = 0.f;

    auto stage = [&](auto kind) {
        constexpr int KIND = decltype(kind)::value;
        (void)KIND;
        _Float16 hlo, hhi;
        const bool half_act = HS && act_half_exact(p.act, hlo, hhi);
#pragma unroll
        for (int i = 0; i < N::NB; i++) {
            if (l_off[i] < 0) continue;
            const bool ok = (inside >> i) & 1u;
            if constexpr (HS) {
                half8_t v;
                if (half_act) {
                    v = ok ? act_half(raw[i], hlo, hhi) : (half8_t)((_Float16)0.f);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = ok ? (_Float16)act_p16((float)raw[i][e], p.act) : (_Float16)0.f;
                }
                *reinterpret_cast<half8_t*>(lds + l_off[i]) = v;
            } else {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = raw[i][e];
                half8_t hi, lo;
                split8<KIND>(x, ok, p.act, in_scale, hi, lo);
                *reinterpret_cast<half8_t*>(lds + l_off[i]) = hi;
                *reinterpret_cast<half8_t*>(lds + N::PLANE + l_off[i]) = lo;
            }
        }
    };
    for (;;) {
        if (p.act.kind == ACT_NONE) stage(std::integral_constant<int, ACT_NONE>());
        else if (p.act.kind == ACT_RELU) stage(std::integral_constant<int, ACT_RELU>());
        else stage(std::integral_constant<int, ACT_LEAKY>());
        lds_barrier();   // the window is there
        const int next = tile + p.pos_groups;
        const bool more = next < ntiles;
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        if (more) fetch(next);
        // the residual values of this wave's fragments
        const int px = txi * 16 + mq;
        store_t rv[N::NO][4];
        auto mine = [&](int i, int& f, int& py) {   // fragment and row of the wave's number i; whether its values are stored
            const int q = wave + 4 * i;
            f = q / TH;
            py = tyi * TH + q - f * TH;
            return q < N::NQ && py < p.npos_y && px < p.npos_x && ch0 + f * 16 + kq * 4 + 4 <= p.out_cp;   // (the last fragment may reach beyond the channel pitch)
        };
        if (p.res) {
#pragma unroll
            for (int i = 0; i < N::NO; i++) {
                int f, py;
                const bool ok = mine(i, f, py);
                const store_t* r = reinterpret_cast<const store_t*>(p.res) + (ok ? ((size_t)(p.res_off_y + py) * p.res_wp + p.res_off_x + px) * p.res_cp + ch0 + f * 16 + kq * 4 : 0);
                if constexpr (HS) *reinterpret_cast<half4_t*>(rv[i]) = *reinterpret_cast<const half4_t*>(r);
                else *reinterpret_cast<f32x4_t*>(rv[i]) = *reinterpret_cast<const f32x4_t*>(r);
            }
        }
        f32x4_t acc[FR][TH];
#pragma unroll
        for (int f = 0; f < FR; f++)
#pragma unroll
            for (int r = 0; r < TH; r++) acc[f][r] = (f32x4_t)(0.f);
#pragma unroll
        for (int s = 0; s < SPW; s++) {
            if (s == SPW - 1 && !last_step) continue;
            // (three fragments keep the matrix pipe busy row by row; fewer need several rows in flight)
            constexpr int RB = FR == 3 ? 1 : TH;
#pragma unroll
            for (int r0 = 0; r0 < TH; r0 += RB) {
                half8_t b[RB][NPL];
#pragma unroll
                for (int r = 0; r < RB; r++)
#pragma unroll
                    for (int pl = 0; pl < NPL; pl++) {
                        b[r][pl] = *reinterpret_cast<const half8_t*>(lds + off[s] + (r0 + r) * S * N::ROWP + pl * N::PLANE);
                        if (s == SPW - 1 && (9 * G) % 4 != 0 && pad_lane) b[r][pl] = (half8_t)((_Float16)0.f);
                    }
#pragma unroll
                for (int i = 0; i < N::NPASS; i++)
#pragma unroll
                    for (int r = 0; r < RB; r++)
#pragma unroll
                        for (int f = 0; f < FR; f++)
                            acc[f][r0 + r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[s][f][i == 1 ? NPL - 1 : 0], b[r][i == 2 ? NPL - 1 : 0], acc[f][r0 + r], 0, 0, 0);
            }
        }
        // partial sums: a wave keeps the fragments it will finish and hands the others over
        f32x4_t own[N::NO];
#pragma unroll
        for (int q = 0; q < N::NQ; q++) {
            const f32x4_t v = acc[q / TH][q % TH];
            if ((q & 3) == wave) own[q >> 2] = v;
            else *reinterpret_cast<f32x4_t*>(lds + N::SUMS + (q * 3 + ((wave - q - 1) & 3)) * 1024 + lane * 16) = v;
        }
        lds_barrier();   // (also: nobody reads this tile's window any more)
#pragma unroll
        for (int i = 0; i < N::NO; i++) {
            int f, py;
            const bool ok = mine(i, f, py);
            const int q = min(wave + 4 * i, N::NQ - 1);
            const f32x4_t sc = *reinterpret_cast<const f32x4_t*>(lds + N::SB + (min(f, FR - 1) * 16 + kq * 4) * 4);
            const f32x4_t bi = *reinterpret_cast<const f32x4_t*>(lds + N::SB + (FR * 16 + min(f, FR - 1) * 16 + kq * 4) * 4);
            f32x4_t v = own[i];
#pragma unroll
            for (int k = 0; k < 3; k++) v += *reinterpret_cast<const f32x4_t*>(lds + N::SUMS + (q * 3 + k) * 1024 + lane * 16);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = v[e] * (sc[e] * acc_mul) + bi[e];
                if (p.res) v[e] = fmaf(fmaxf((float)rv[i][e], res_floor), p.res_scale ? sc[e] : 1.f, v[e]);
                if constexpr (!HS) vmax = fmaxf(vmax, ok ? fabsf(v[e]) : 0.f);
            }
            store_t* o = reinterpret_cast<store_t*>(p.out) + ((size_t)(p.out_off_y + py) * p.out_wp + p.out_off_x + px) * p.out_cp + ch0 + f * 16 + kq * 4;
            if constexpr (HS) {
                half4_t hv;
#pragma unroll
                for (int e = 0; e < 4; e++) hv[e] = (_Float16)v[e];
                if (ok) *reinterpret_cast<half4_t*>(o) = hv;
            } else {
                if (ok) *reinterpret_cast<f32x4_t*>(o) = v;
            }
        }
        if (!more) break;
        tile = next;
    }
    if (!HS && p.out_amax) range_publish_block256(p.out_amax, vmax);
}

struct P16NEntry {
    bool f16;
    int groups, frags, step, rows;
    void (*fn)(const ConvP16Params);
    size_t lds;
};
template <bool HS, int G, int FR, int S, int TH>
constexpr P16NEntry p16n_entry() {
    typedef GeoN<HS, G, FR, S, TH> N;
    return P16NEntry{HS, G, FR, S, TH, conv_p16n_kernel<N>, (size_t)N::LDS};
}
// (a step of two doubles the window: four rows of it where five fit with a step of one; two rows of 64 channels, whose
// window of four, 88 KB in two planes, is beyond the immediate field.  Not compiled are 32 channels, 56, and 48 with a step of
// two, although they would gain at some sizes.  This form against the others, us, fp32 and fp16 tensors: 32 -> 32 at 56x56
// 3.9 / 4.4 and 3.6 / 3.6, at 112x112 4.8 / 4.9 and 4.1 / 4.0, at 256x256 10.1 / 8.7 and 7.4 / 6.6; 48 -> 48, step 2, at 56x56 5.4 / 6.8
// and 4.5 / 4.6, at 256x256 19.6 / 23.5 and 11.6 / 13.0; 56 -> 56 at 56x56 4.6 / 5.2 and 4.0 / 4.0, at 128x128 7.7 / 6.5 and 5.8 / 4.7)
#define P16N_ROWS(HS, G, FR, S) p16n_entry<HS, G, FR, S, 2>(), p16n_entry<HS, G, FR, S, S == 1 ? 5 : 4>()
#define P16N_FRAGS(HS, G, S) P16N_ROWS(HS, G, 1, S), P16N_ROWS(HS, G, 2, S), P16N_ROWS(HS, G, 3, S)
#define P16N_STEPS(HS, G) P16N_FRAGS(HS, G, 1), P16N_FRAGS(HS, G, 2)
// (64 input channels: a wave's weights for two fragments fill the registers that three take elsewhere)
#define P16N_WIDE(HS) p16n_entry<HS, 8, 1, 1, 2>(), p16n_entry<HS, 8, 2, 1, 2>(), p16n_entry<HS, 8, 1, 1, 5>(), p16n_entry<HS, 8, 2, 1, 5>(), p16n_entry<HS, 8, 1, 2, 2>(), p16n_entry<HS, 8, 2, 2, 2>()
const P16NEntry P16N_TABLE[] = {
    P16N_STEPS(false, 2), P16N_STEPS(false, 3), P16N_STEPS(false, 5), P16N_FRAGS(false, 6, 1), P16N_WIDE(false),
    P16N_STEPS(true, 2), P16N_STEPS(true, 3), P16N_STEPS(true, 5), P16N_FRAGS(true, 6, 1), P16N_WIDE(true),
};
const P16NEntry* p16n_find(const ConvP16Params& p) {
    for (const P16NEntry& e : P16N_TABLE)
        if (e.f16 == (p.f16 != 0) && e.groups * 8 == p.in_cp && e.frags == p.wm && e.step == p.stride && e.rows == p.tile_h) return &e;
    return nullptr;
}
}  // namespace

size_t conv_p16n_lds_bytes(const ConvP16Params& p) {
    const P16NEntry* e = p16n_find(p);
    return e ? e->lds : 0;
}

// p.tile_h = rows of a tile (2, or 5 with a step of one and 4 with a step of two), p.wm = fragments of 16 output channels per grid row, p.cout_blocks = grid rows, p.mfrags =
// wm * cout_blocks (scale, bias and wpack hold 16 * mfrags rows; rows beyond out_cp are not stored), tiles of tile_h x 16 positions, p.pos_groups = workgroups; weights, in_y0, in_x0,
// in_shift, in_clamp and stride as for launch_conv_g16.
int launch_conv_p16n(const ConvP16Params& p, hipStream_t s) {
    const P16NEntry* e = p16n_find(p);
    if (!e) return -1;
    const long long in_elems = (long long)p.in_hp * p.in_wp * p.in_cp;
    if (in_elems > (1ll << 30) || p.mfrags != p.wm * p.cout_blocks || p.cout_blocks < 1 || p.cout_blocks > 16 || p.tiles_x < 1 || p.tiles_y < 1 || p.tiles_x * 16 < p.npos_x || p.tiles_y * p.tile_h < p.npos_y || p.pos_groups < 1 ||
        p.pos_groups > p.tiles_x * p.tiles_y || p.tiles_x * p.tiles_y > 4000000 || p.rcp_tiles_x != 1.0f / (float)p.tiles_x || p.out_cp % 4 != 0 || p.out_cp < 4 ||
        (p.res && (p.res_cp < p.out_cp || p.res_cp % 4 != 0)) || p.nreset < 0 || p.nreset > 4 || p.dw_in || p.in_mul || p.in2 || !p.in || !p.out || !p.wpack || !p.scale || !p.bias ||
        p.in_shift < 0 || p.in_shift > 8 || ((long long)p.in_hp << p.in_shift) > (1 << 28) || ((long long)p.in_wp << p.in_shift) > (1 << 28))
        return -5;
    if (e->lds > 160 * 1024 || ensure_lds(reinterpret_cast<const void*>(e->fn), e->lds) != 0) return -2;
    hipLaunchKernelGGL(e->fn, dim3((unsigned)p.pos_groups, (unsigned)p.cout_blocks), dim3(256), e->lds, s, p);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace fynhip
