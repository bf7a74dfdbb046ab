// The first two layers of a style-transfer net as one launch: a 9x9 convolution of an image (at most four channels, up to 32
// out) and the 3x3 convolution with a step of two behind it (up to 64 out), on gfx950 matrix cores.
//
// Replaces, for such a pair, two render passes of DeepConvLayerNxN::forward (fyusenet/gpu/deep/deepconvlayerNxN.cpp:129-211).
//
// Bound: the matrix pipes.  Apart, the layers meet in the largest tensor of the net -- 265 MB at 1920x1080 on fp32 tensors,
// written and read again in half of their time --, and in the first one every workgroup multiplies and then stores.  Here it
// stays in LDS: a workgroup walks tiles of 4 rows x 31 positions of the second layer's output and computes the 9 rows x 63
// positions of the first layer under them (1.16 times its arithmetic; a tile's columns and rows overlap its neighbours' by
// one), as hi and lo planes with even and odd columns apart, so that the sixteen positions of a fragment of the second layer
// are neighbours there whatever the tap and a fragment is one contiguous kilobyte.  Four waves compute the first layer, sixteen
// columns each, with the schedule of the layer's own kernel (c4_rows, its weights in LDS).  Four others compute the second one
// of the tile before at the same time, 32 channels x 16 columns x 4 rows each, column of taps by column of taps, where the
// fragment of row j serves every tap that meets it, and make the operands of the tile behind in registers.  Behind a barrier the
// first ones split their result into the tensor in between while the others put the window in place and store theirs: the
// vector work of either half of the waves lies beside the matrix work of the other, or beside its vector work.  With one
// group of waves for all matrix work and one that staged a tile of fp32 tensors took 18.7k clocks, now 15.6k (fp16 9.1k and
// 7.8k); 10.4k of them are matrix instructions, of either group in one pipe.  0.6k are the tile's own scale for the tensor in
// between, which has to be known in front of the split: with one from a bound on the weights the launch at 1920x1080 took
// 118 us, and values far below that bound lost bits (1.2e-5 of error where 2.6e-7 are left now).  1920x1080, both layers
// timed back to back: 209 us apart, 123 here; fp16 tensors 88 and 60.
//
// At most 16 channels in between and 32 behind (SMALL): one fragment of channels in the first layer, two taps of 16 channels a
// step in the second, whose weights lie in LDS; bound by the fragment reads of the first layer (134 KB a wave and tile at 128
// bytes a clock: 4.2k of a tile's 9.1k clocks).  3 -> 12 -> 20 channels at 512x624: 35.7 us apart, 19 here (fp16 24 and 11).
#include "c4_common.h"

namespace fynhip {
namespace {
// The halves of values that carry their scale already, as split_pair gives them: packed conversions and subtractions, 26
// clocks a pair where the four mixed-precision FMAs of split_pair take 33 (each of them issues for eight).
template <int N, class V>
__device__ __forceinline__ void split_packed(const float (&x)[N], V& hi, V& lo) {
#pragma unroll
    for (int e = 0; e < N; e++) {
        hi[e] = (_Float16)x[e];
        lo[e] = (_Float16)(x[e] - (float)hi[e]);
    }
}

// The first layer's tile, as GeoC4 describes it for conv_p16c4_kernel (rows without the pad behind them: the LDS is full).
// SMALL: at most 16 channels in between and 32 behind.
template <bool SMALL>
struct GeoA {
    static constexpr int K = 9, TH = 9, TWG = 64, FN = TH, FM = SMALL ? 1 : 2, NS = 12, PIX = 8;
    static constexpr int HW = TWG + 9, HH = TH + K - 1;
    static constexpr int ROW_PITCH = (HW + 1) * PIX;
    static constexpr int COPY = HH * ROW_PITCH, COPY2 = (COPY + 127) / 128 * 128 + 48, PLANE = COPY2 + COPY + 16, BUF = NPL * PLANE;
    static constexpr int NITEMS = HH * HW, NB = (NITEMS + 255) / 256;
    // the second layer's: rows and columns of its tile, the tensor in between [row][even columns, odd columns][32 or 16 channels]
    static constexpr int TH2 = 4, TW2 = 31, SLOT = SMALL ? 32 : 64, MROW = 63 * SLOT, MPLANE = TH * MROW;
    static constexpr int STEPS2 = 5;                                // SMALL: the second layer's, two taps of 16 channels each; its weights lie in LDS too
    static constexpr int NW = HSTORE ? 4 : 8;                       // weight fragments of a pair of steps (c4_rows)
    static constexpr int WEIGHTS = BUF, MID = WEIGHTS + NS / 2 * NW * 1024, SB = MID + NPL * MPLANE, W2 = SB + (32 + 64) * 2 * 4, LDS = W2 + (SMALL ? STEPS2 * 2 * NPL * 1024 : 0);
    static_assert(LDS + 48 <= 160 * 1024 && BUF < 65536 && ROW_PITCH % 16 == 0, "fits a CU; 16-byte reads are aligned");
};

// (KEEP: the tensor in between is written to memory as well, for a net whose tensors all stay readable)
template <bool HS, bool KEEP, bool SMALL>
__global__ __launch_bounds__(512) void conv_a16_kernel(const ConvA16Params p) {
    using G = GeoA<SMALL>;
    constexpr bool C8 = !HS;
    constexpr int FN = G::FN, FM = G::FM, NW = G::NW;
    // a lane's first channel of a fragment, and from one fragment to the next (c4_common.h; one fragment alone is in order)
    constexpr int CK1 = SMALL ? 4 : CHK;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ unsigned range_box[2];
    __shared__ __align__(16) float mid_top[2][4];   // fp32 tensors: what the first layer's waves found, in this tile and the one before
    if (blockIdx.x == 0) range_clear(p.reset[0], p.reset[1], p.reset[2], p.reset[3], p.nreset);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (neighbouring tiles, whose windows overlap, meet in one XCD's L2)
    int group = blockIdx.x;
    {
        const int per = (int)gridDim.x >> 3;
        if (group < (per << 3)) group = (group & 7) * per + (group >> 3);
    }
    const int ntiles = p.tiles_x * p.tiles_y, step = (int)gridDim.x;
    if (tid < 2) range_box[tid] = 0u;
    const unsigned range_bits = p.in_amax ? range_load(p.in_amax) : 0u;
    float in_scale = 1.f, inv_in = 1.f;
    auto scales = [&]() __attribute__((always_inline)) {
        if (p.in_amax) in_scale = range_scale(range_after_act(range_reduce(range_bits), p.act[0]), &inv_in);
    };
    // The tensor in between takes its scale from the tile: no value is larger than its channel's largest sum of products there
    // allows, with the bias.  (Where a bias cancels such a sum, the sum's own 22 bits are what is left; a bound from the
    // weights alone can lie any number of bits above what a frame reaches, and values then lose theirs.)
    auto mid_scale = [&](int turn, float* inv) __attribute__((always_inline)) {
        const f32x4_t t = *reinterpret_cast<const f32x4_t*>(mid_top[turn]);
        return range_scale(range_after_act(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3])), p.act[1]), inv);
    };
    const int mq = lane & 15, kq = lane >> 4, w = wave & 3;
    const unsigned wlane = lane * 16;
    const float* const sb = reinterpret_cast<const float*>(lds + G::SB);
    if (wave < 4) {   // ------------------------------------------- the waves that stage and compute the second layer
        const store_t* in = reinterpret_cast<const store_t*>(p.in);
        typedef typename std::conditional<HS, half4_t, float4>::type raw_t;   // a pixel as it comes from memory
        raw_t raw[G::NB];
        int yx[G::NB], l_off[G::NB];
        unsigned inside = 0u;   // one bit an item
#pragma unroll
        for (int i = 0; i < G::NB; i++) {
            const int idx = tid + i * 256, py = idx / G::HW, px = idx - py * G::HW;
            yx[i] = py << 16 | px;
            l_off[i] = idx < G::NITEMS ? py * G::ROW_PITCH + px * G::PIX : -1;
        }
        auto fetch = [&](int tile) {
            const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
            // (row 2 y - 1, column 2 x - 1 of the first layer, four pixels further out)
            const int y0 = tyi * 2 * G::TH2 - 5, x0 = txi * 2 * G::TW2 - 5;
            inside = 0u;
#pragma unroll
            for (int i = 0; i < G::NB; i++) {
                int y = y0 + (yx[i] >> 16), x = x0 + (yx[i] & 0xffff);
                if (p.clamp) {
                    y = min(max(y, 0), p.h - 1);
                    x = min(max(x, 0), p.w - 1);
                }
                const bool ok = l_off[i] >= 0 && (unsigned)y < (unsigned)p.h && (unsigned)x < (unsigned)p.w;
                inside |= ok ? 1u << i : 0u;
                raw[i] = *reinterpret_cast<const raw_t*>(in + (ok ? ((y + p.in_off) * p.in_wp + x + p.in_off) * 4 : 0));
            }
        };
        const bool plain_act = p.act[0].kind == ACT_NONE;   // (a first layer reads its input as it is)
        // (the operands of an item take the registers that its pixel came in: they are made while the matrix pipes are busy and
        // wait there for the window's place)
        typedef typename std::conditional<HS, half4_t, int4>::type staged_t;
        auto convert = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < G::NB; i++) {
                const bool ok = (inside >> i) & 1u;
                if constexpr (HS) {
                    half4_t v;
                    _Float16 hlo, hhi;
                    if (act_half_exact(p.act[0], hlo, hhi)) {
                        v = ok ? act_half4(raw[i], hlo, hhi) : (half4_t)((_Float16)0.f);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = ok ? (_Float16)act_p16((float)raw[i][e], p.act[0]) : (_Float16)0.f;
                    }
                    raw[i] = v;
                } else {
                    const float r[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
                    float x[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] = ok ? (plain_act ? r[e] : act_p16(r[e], p.act[0])) : 0.f;
                    unsigned h0, l0, h1, l1;
                    split_pair(x[0], x[1], in_scale, h0, l0);
                    split_pair(x[2], x[3], in_scale, h1, l1);
                    const half4_t hi = __builtin_bit_cast(half4_t, uint2{h0, h1}), lo = __builtin_bit_cast(half4_t, uint2{l0, l1});
                    raw[i] = __builtin_bit_cast(float4, int4{(int)h0, (int)h1, (int)c8_quad(lo[0], lo[1], lo[2], lo[3], 0.03125f), (int)c8_quad(hi[0], hi[1], hi[2], hi[3], 64.f)});
                }
            }
        };
        auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < G::NB; i++) {
                if (l_off[i] < 0) continue;
                unsigned char* const at = lds + l_off[i];
                const staged_t v = __builtin_bit_cast(staged_t, raw[i]);
                if constexpr (HS) {
                    *reinterpret_cast<half4_t*>(at) = v;
                    *reinterpret_cast<half4_t*>(at + G::COPY2 + 8) = v;
                } else {
                    *reinterpret_cast<int2*>(at) = int2{v.x, v.y};
                    *reinterpret_cast<int2*>(at + G::COPY2 + 8) = int2{v.x, v.y};
                    *reinterpret_cast<int2*>(at + G::PLANE) = int2{v.z, v.w};
                    *reinterpret_cast<int2*>(at + G::PLANE + G::COPY2 + 8) = int2{v.z, v.w};
                }
            }
        };
        fetch(group);
        scales();
        {
            float* const to = reinterpret_cast<float*>(lds + G::SB);
            if (tid < 32) {
                to[tid] = tid < p.mid_cp ? p.scale[0][tid] : 0.f;
                to[32 + tid] = tid < p.mid_cp ? p.bias[0][tid] : 0.f;
            } else if (tid >= 64 && tid < 128) {
                to[tid] = tid - 64 < p.out_cp ? p.scale[1][tid - 64] : 0.f;
                to[64 + tid] = tid - 64 < p.out_cp ? p.bias[1][tid - 64] : 0.f;
            }
        }
        convert();
        put();
        const int cpair = SMALL ? 0 : w & 1, cfrag = w >> 1;   // of the second layer: 32 channels, 16 columns
        constexpr int ROWS2 = SMALL ? G::TH2 / 2 : G::TH2;
        const int row2 = SMALL ? (w & 1) * ROWS2 : 0;          // rows
        const unsigned char* const mid_at = lds + G::MID + (cfrag * 16 + mq) * G::SLOT + (SMALL ? (kq & 1) * 16 + row2 * 2 * G::MROW : kq * 16);
        // (buffer loads: the fragment's place is a scalar operand, where 64-bit addresses of all of them would fill the registers)
        const __amdgpu_buffer_rsrc_t weights2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.wpack[1]), 0, 36 * NPL * 1024, 0x00020000);   // [kx][32 channels][ky][fragment][plane]
        // SMALL: two taps a step, the lanes of either half of the wave one
        int tap_at[SMALL ? G::STEPS2 : 1];
        if constexpr (SMALL) {
#pragma unroll
            for (int s = 0; s < G::STEPS2; s++) {
                const int tap = min(2 * s + (kq >> 1), 8), ky = tap / 3, kx = tap - 3 * ky;
                tap_at[s] = ky * G::MROW + (kx == 1 ? 32 * G::SLOT : kx * (G::SLOT / 2));
            }
            for (int i = w; i < G::STEPS2 * 2 * NPL; i += 4)
                *reinterpret_cast<i32x4_t*>(lds + G::W2 + i * 1024 + wlane) = *reinterpret_cast<const i32x4_t*>(reinterpret_cast<const unsigned char*>(p.wpack[1]) + i * 1024 + wlane);
        }
        store_t* const out = reinterpret_cast<store_t*>(p.out);
        const bool through = store_through_pays(p.out, p.h2, p.w2, p.out_cp * ESZ, !p.plain_stores, hw_block_count());
        bool drop = through && wave == 0 && hw_block_id() < 8;
        float vmax = 0.f;
        f32x4_t acc[2][ROWS2];
        auto multiply = [&]() __attribute__((always_inline)) {   // rows 2 r + ky, columns 2 c + kx of the tensor in between
#pragma unroll
            for (int fm = 0; fm < 2; fm++)
#pragma unroll
                for (int r = 0; r < ROWS2; r++) acc[fm][r] = (f32x4_t)(0.f);
            constexpr int AHEAD = 3, Q = SMALL ? G::STEPS2 * ROWS2 : 3 * FN;
            half8_t wq[SMALL ? 1 : 2][3][2][NPL], b[AHEAD + 1][NPL], w2[SMALL ? G::STEPS2 : 1][2][NPL];
            typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
            auto load_w = [&](int set, int kx) __attribute__((always_inline)) {
#pragma unroll
                for (int ky = 0; ky < 3; ky++)
#pragma unroll
                    for (int fm = 0; fm < 2; fm++)
#pragma unroll
                        for (int pl = 0; pl < NPL; pl++)
                            wq[set][ky][fm][pl] = __builtin_bit_cast(half8_t, (u32x4_t)__builtin_amdgcn_raw_buffer_load_b128(weights2, wlane, (unsigned)(((kx * 2 + cpair) * 6 + ky * 2 + fm) * NPL + pl) * 1024u, 0));
            };
            if constexpr (!SMALL) load_w(0, 0);   // (a column of taps, two columns in flight)
            auto request = [&](int q) __attribute__((always_inline)) {
                const int kx = q / FN, j = q % FN;
                const unsigned char* const at = mid_at + (SMALL ? tap_at[SMALL ? q / ROWS2 : 0] + q % ROWS2 * 2 * G::MROW : (kx == 1 ? 32 * G::SLOT : kx * (G::SLOT / 2)) + j * G::MROW);
#pragma unroll
                for (int pl = 0; pl < NPL; pl++) b[q % (AHEAD + 1)][pl] = *reinterpret_cast<const half8_t*>(at + pl * G::MPLANE);
            };
#pragma unroll
            for (int q = 0; q < AHEAD; q++) request(q);
            auto weights2_of = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 2 * NPL; i++) w2[SMALL ? s : 0][i / NPL][i % NPL] = *reinterpret_cast<const half8_t*>(lds + G::W2 + (s * 2 * NPL + i) * 1024 + wlane);
            };
            if constexpr (SMALL) weights2_of(0);
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if (q + AHEAD < Q) request(q + AHEAD);
                if constexpr (SMALL) {
                    if (q % ROWS2 == 0 && q / ROWS2 + 1 < G::STEPS2) weights2_of(q / ROWS2 + 1);
#pragma unroll
                    for (int i = 0; i < NPASS; i++)
#pragma unroll
                        for (int fm = 0; fm < 2; fm++)
                            acc[fm][q % ROWS2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w2[q / ROWS2][fm][i == 1 ? NPL - 1 : 0], b[q % (AHEAD + 1)][i == 2 ? NPL - 1 : 0], acc[fm][q % ROWS2], 0, 0, 0);
                } else {
                    const int kx = q / FN, j = q % FN;
                    if (j == 0 && kx + 1 < 3) load_w((kx + 1) & 1, kx + 1);
#pragma unroll
                    for (int i = 0; i < NPASS; i++)
#pragma unroll
                        for (int ky = 0; ky < 3; ky++) {
                            if (((j - ky) & 1) || j < ky || (j - ky) / 2 >= G::TH2) continue;
#pragma unroll
                            for (int fm = 0; fm < 2; fm++)
                                acc[fm][(j - ky) / 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wq[kx & 1][ky][fm][i == 1 ? NPL - 1 : 0], b[q % (AHEAD + 1)][i == 2 ? NPL - 1 : 0], acc[fm][(j - ky) / 2], 0, 0, 0);
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto finish = [&](int tile, float mul2) __attribute__((always_inline)) {
            const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
            if (drop) {   // (ahead of this workgroup's first store: what it has read so far may go as well)
                drop_clean_l2_lines();
                drop = false;
            }
            f32x4_t sc[2], bi[2];
#pragma unroll
            for (int fm = 0; fm < 2; fm++) {
                sc[fm] = *reinterpret_cast<const f32x4_t*>(sb + 64 + cpair * 32 + kq * CHK + fm * CHF) * mul2;
                bi[fm] = *reinterpret_cast<const f32x4_t*>(sb + 128 + cpair * 32 + kq * CHK + fm * CHF);
            }
            const int c2 = cfrag * 16 + mq, ox = txi * G::TW2 + c2, ch0 = cpair * 32 + kq * CHK;
#pragma unroll
            for (int r = 0; r < ROWS2; r++) {
                const int oy = tyi * G::TH2 + row2 + r;
                const bool inside = c2 < G::TW2 && ox < p.w2 && oy < p.h2;
                const size_t at = ((size_t)(p.out_off + oy) * p.out_wp + p.out_off + ox) * p.out_cp + ch0;
                half8_t hv;
#pragma unroll
                for (int fm = 0; fm < 2; fm++) {
                    const bool ok = inside && ch0 + (HS ? 0 : fm * CHF) < p.out_cp;
                    f32x4_t v;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        v[e] = acc[fm][r][e] * sc[fm][e] + bi[fm][e];
                        if constexpr (!HS) vmax = fmaxf(vmax, ok ? fabsf(v[e]) : 0.f);
                        else hv[fm * 4 + e] = (_Float16)v[e];
                    }
                    if constexpr (HS) {
                        if (fm == 1 && ok) store_out(through, reinterpret_cast<half8_t*>(out + at), hv);
                    } else {
                        if (ok) store_out(through, reinterpret_cast<f32x4_t*>(out + at + fm * CHF), v);
                    }
                }
            }
        };
        lds_barrier();   // the first window is staged
        for (int tile = group, before = -1, turn = 0;; before = tile, tile += step, turn ^= 1) {   // (the tile that the other waves are on, the one before it)
            const bool more = tile < ntiles, next = tile + step < ntiles;
            if (next) fetch(tile + step);
            float inv_mid = 1.f;
            if constexpr (C8) {
                if (before >= 0) (void)mid_scale(turn ^ 1, &inv_mid);
            }
            if (before >= 0) multiply();
            if (next) convert();
            if (more) lds_barrier();   // the first layer is through: the window's place is free
            if (next) put();
            if (before >= 0) finish(before, p.acc_mul[1] * inv_mid);
            if (!more) break;
            lds_barrier();   // the window is staged, the tensor in between is there
        }
        if (p.out_amax) range_publish_waves(p.out_amax, vmax, range_box, 4);
        return;
    }
    // ------------------------------------------------------------- the waves that compute the first layer
    {   // the first layer's weights into LDS, as c4_rows takes them: [pair of steps][fragment][lane]
        constexpr int SHARE = G::NS / 2 * NW / 4;
        i32x4_t v[SHARE];
#pragma unroll
        for (int i = 0; i < SHARE; i += SMALL ? 2 : 1) {   // (SMALL: the first fragment's alone)
            const int c = w * SHARE + i, k = c % NW, st = c / NW * 2 + (k / 2) % 2, fm = k % 2, plane = k < 4 ? 0 : 2;
            v[i] = *reinterpret_cast<const i32x4_t*>(reinterpret_cast<const unsigned char*>(p.wpack[0]) + (size_t)((st * p.mfrags0 + fm) * NPLW + plane) * 1024 + wlane);
        }
#pragma unroll
        for (int i = 0; i < SHARE; i += SMALL ? 2 : 1) *reinterpret_cast<i32x4_t*>(lds + G::WEIGHTS + (w * SHARE + i) * 1024 + wlane) = v[i];
    }
    // this lane's places: in the window, in the tensor in between (as it writes and as it reads)
    const int x1 = w * 16 + mq;   // column of the first layer's tile
    const unsigned char* const col = lds + x1 * G::PIX + ((x1 & 1) ? G::COPY2 + 8 : 0);
    const unsigned char* const rows_at = col + 2 * kq * G::PIX;
    const unsigned char* const ninth_at = col + kq * G::ROW_PITCH + 8 * G::PIX;
    const unsigned char* const last_at = col + 8 * G::ROW_PITCH + 8 * G::PIX;
    unsigned char* const mid_to = lds + G::MID + ((x1 & 1) ? 32 + (x1 >> 1) : x1 >> 1) * G::SLOT + kq * (G::SLOT / 4);   // (its eight channels side by side; the second layer's weights are laid out for that)
    scales();
    const float mul1 = p.acc_mul[0] * inv_in;
    const float lo1 = p.act[1].kind == ACT_NONE ? -3.0e38f : p.act[1].kind == ACT_RELU ? 0.f : p.act[1].lo;
    const float hi1 = p.act[1].kind == ACT_NONE || p.act[1].kind == ACT_RELU ? 3.0e38f : p.act[1].hi;
    const float leak1 = p.act[1].kind == ACT_NONE || p.act[1].kind == ACT_RELU ? 0.f : p.act[1].leak;
    _Float16 hlo1, hhi1;
    const bool packed1 = act_half_exact(p.act[1], hlo1, hhi1);
    C4Ring<G> ring;
    constexpr int LA = C4Ring<G>::LA;
    lds_barrier();   // the first window is staged, the weights are there
#pragma unroll
    for (int d = 0; d < C4Ring<G>::LW; d++)
#pragma unroll
        for (int k = 0; k < NW; k += SMALL ? 2 : 1) rows_put_w(ring.a0[d], ring.a2[d], k, *reinterpret_cast<const i32x4_t*>(lds + G::WEIGHTS + (d * NW + k) * 1024 + wlane));
    for (int tile = group, turn = 0;; turn ^= 1) {
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        {   // ---- first layer ----
            f32x4_t acc[FM][FN];
#pragma unroll
            for (int fm = 0; fm < FM; fm++)
#pragma unroll
                for (int fn = 0; fn < FN; fn++) acc[fm][fn] = (f32x4_t)(0.f);
#pragma unroll
            for (int r = 0; r <= LA; r++) ring.b0[r] = *reinterpret_cast<const half8_t*>(rows_at + r * G::ROW_PITCH);
            if constexpr (C8) {
#pragma unroll
                for (int r = 0; r < LA; r++)
#pragma unroll
                    for (int h = 0; h < 2; h++) rows_load_b8<G>(ring.b8[r], h, rows_at + (r + h) * G::ROW_PITCH + G::PLANE);
            }
            c4_rows<G, false>(acc, ring, rows_at, ninth_at, last_at, rows_at, lds + G::WEIGHTS + wlane);
            __builtin_amdgcn_sched_barrier(0);
            const int px = txi * 2 * G::TW2 - 1 + x1, py = tyi * 2 * G::TH2 - 1;
            const bool x_ok = (unsigned)px < (unsigned)p.w;
            f32x4_t scm[FM], bi[FM];
            auto scale_and_bias = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int fm = 0; fm < FM; fm++) {
                    scm[fm] = *reinterpret_cast<const f32x4_t*>(sb + kq * CK1 + fm * CHF) * mul1;
                    bi[fm] = *reinterpret_cast<const f32x4_t*>(sb + 32 + kq * CK1 + fm * CHF);
                }
            };
            float mid = 1.f, inv_mid = 1.f;
            if constexpr (C8) {
                scale_and_bias();
                f32x4_t m[FM];
                auto larger = [](f32x4_t& m, const f32x4_t v) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 4; e++) m[e] = fmaxf(m[e], fabsf(v[e]));
                };
#pragma unroll
                for (int fm = 0; fm < FM; fm++) m[fm] = (f32x4_t)(0.f);
                if (py >= 0 && py + FN <= p.h) {
#pragma unroll
                    for (int r = 0; r < FN; r++)
#pragma unroll
                        for (int fm = 0; fm < FM; fm++) larger(m[fm], acc[fm][r]);
                } else {   // (positions outside the layer's output don't count)
#pragma unroll
                    for (int r = 0; r < FN; r++)
                        if ((unsigned)(py + r) < (unsigned)p.h)
#pragma unroll
                            for (int fm = 0; fm < FM; fm++) larger(m[fm], acc[fm][r]);
                }
                float top = 0.f;
#pragma unroll
                for (int i = 0; i < 4 * FM; i++) top = fmaxf(top, m[i / 4][i % 4] * fabsf(scm[i / 4][i % 4]) + fabsf(bi[i / 4][i % 4]));
                top = range_wave_max(x_ok && x1 < 63 ? top : 0.f);
                if (lane == 0) mid_top[turn][w] = top;
            }
            lds_barrier();   // the window's place is free, and nobody reads the tensor in between any more
            if constexpr (C8) {
                mid = mid_scale(turn, &inv_mid);
#pragma unroll
                for (int fm = 0; fm < FM; fm++) { scm[fm] *= mid; bi[fm] *= mid; }
            } else {
                scale_and_bias();
            }
            const float lo_mid = lo1 * mid, hi_mid = hi1 * mid;   // (its values carry the scale)
            typedef typename std::conditional<SMALL, half4_t, half8_t>::type piece_t;
            auto leave = [&](auto general_) __attribute__((always_inline)) {   // (general: an activation other than none, a clamp exact on halves, or a clamp)
                constexpr bool GENERAL = decltype(general_)::value;
#pragma unroll
                for (int r = 0; r < FN; r++) {
                    // (positions outside the layer's output are its zero padding)
                    const bool ok = x_ok && (unsigned)(py + r) < (unsigned)p.h;
                    unsigned char* const to = mid_to + r * G::MROW;
                    // (a tile's first row and column are its neighbours' to write)
                    const bool own = KEEP && ok && r > 0 && x1 > 0;
                    store_t* const kept = reinterpret_cast<store_t*>(p.mid) + ((size_t)(p.mid_off + py + r) * p.mid_wp + p.mid_off + px) * p.mid_cp + kq * CK1;
                    if constexpr (HS) {
                        piece_t v;
#pragma unroll
                        for (int fm = 0; fm < FM; fm++)
#pragma unroll
                            for (int e = 0; e < 4; e++) v[fm * 4 + e] = (_Float16)(acc[fm][r][e] * scm[fm][e] + bi[fm][e]);   // (as the layer would have stored it)
                        if constexpr (KEEP) {
                            if (own && kq * CK1 < p.mid_cp) *reinterpret_cast<piece_t*>(kept) = v;
                        }
                        if constexpr (GENERAL) {
#pragma unroll
                            for (int e = 0; e < 4 * FM; e++) v[e] = (_Float16)act_p16((float)v[e], p.act[1]);
                        } else if constexpr (SMALL) {
                            v = act_half4(v, hlo1, hhi1);
                        } else {
                            v = act_half(v, hlo1, hhi1);
                        }
                        *reinterpret_cast<piece_t*>(to) = ok ? v : (piece_t)((_Float16)0.f);
                    } else {
                        const float lo = ok ? lo_mid : 0.f, hi = ok ? hi_mid : 0.f, leak = ok ? leak1 : 0.f;
                        if constexpr (KEEP) {
#pragma unroll
                            for (int fm = 0; fm < FM; fm++)
                                if (own && kq * CK1 + fm * CHF < p.mid_cp) *reinterpret_cast<f32x4_t*>(kept + fm * CHF) = (acc[fm][r] * scm[fm] + bi[fm]) * inv_mid;
                        }
                        float x[4 * FM];
#pragma unroll
                        for (int i = 0; i < 4 * FM; i++) {
                            const float v = acc[i / 4][r][i % 4] * scm[i / 4][i % 4] + bi[i / 4][i % 4];
                            x[i] = __builtin_amdgcn_fmed3f(v, lo, hi);
                            if constexpr (GENERAL) x[i] += leak * fminf(v, 0.f);
                        }
                        piece_t H, L;
                        split_packed<4 * FM>(x, H, L);
                        *reinterpret_cast<piece_t*>(to) = H;
                        *reinterpret_cast<piece_t*>(to + G::MPLANE) = L;
                    }
                    if (!SMALL || r % 3 == 2) __builtin_amdgcn_sched_barrier(0);   // (four values are too few chains of dependent instructions)
                }
            };
            if (x1 < 63) {   // (the 64th column belongs to nobody)
                if (HS ? !packed1 : leak1 != 0.f) leave(std::integral_constant<bool, true>());
                else leave(std::integral_constant<bool, false>());
            }
            if (p.clamp && (txi == 0 || tyi == 0)) {   // what lies above or to the left of the layer's output repeats its first row and column
                asm volatile("" ::: "memory");   // (the first column reads what another lane of its wave stored: in this order)
                if (txi == 0 && x1 == 0)
                    for (int i = 0; i < FN * NPL; i++) {
                        unsigned char* const to = mid_to + (i % FN) * G::MROW + (i / FN) * G::MPLANE;
                        *reinterpret_cast<piece_t*>(to) = *reinterpret_cast<const piece_t*>(to + 32 * G::SLOT);
                    }
                if (tyi == 0 && x1 < 63)
                    for (int pl = 0; pl < NPL; pl++) *reinterpret_cast<piece_t*>(mid_to + pl * G::MPLANE) = *reinterpret_cast<const piece_t*>(mid_to + pl * G::MPLANE + G::MROW);
            }
        }
        lds_barrier();   // the tensor in between is there, and the next window
        tile += step;
        if (tile >= ntiles) return;
    }
}
}  // namespace

#if FYN_P16_HALF
#define A16_NAME(n) n##_half
size_t conv_a16_lds_half(bool small) { return small ? (size_t)GeoA<true>::LDS : (size_t)GeoA<false>::LDS; }
#else
#define A16_NAME(n) n
int launch_conv_a16_half(const ConvA16Params& p, hipStream_t s);
size_t conv_a16_lds_half(bool small);
size_t conv_a16_lds_bytes(bool f16, bool small) { return f16 ? conv_a16_lds_half(small) : small ? (size_t)GeoA<true>::LDS : (size_t)GeoA<false>::LDS; }
void conv_a16_tile(int* rows, int* cols) { *rows = GeoA<false>::TH2; *cols = GeoA<false>::TW2; }
#endif
int A16_NAME(launch_conv_a16)(const ConvA16Params& p, hipStream_t s) {
#if !FYN_P16_HALF
    if (p.f16) return launch_conv_a16_half(p, s);
#endif
    const long long tiles = (long long)p.tiles_x * p.tiles_y;
    const int rows = p.mid ? (p.h + 2 * GeoA<false>::TH2 - 1) / (2 * GeoA<false>::TH2) : (p.h2 + GeoA<false>::TH2 - 1) / GeoA<false>::TH2;
    const int cols = p.mid ? (p.w + 2 * GeoA<false>::TW2 - 1) / (2 * GeoA<false>::TW2) : (p.w2 + GeoA<false>::TW2 - 1) / GeoA<false>::TW2;
    if ((p.f16 != 0) != HSTORE || !p.in || !p.out || !p.wpack[0] || !p.wpack[1] || (!HSTORE && !p.in_amax) || p.h < 2 || p.w < 2 || p.h2 != p.h / 2 || p.w2 != p.w / 2 || p.in_off < 0 ||
        p.h + p.in_off > p.in_hp || p.w + p.in_off > p.in_wp || (long long)p.in_hp * p.in_wp * 4 > (1ll << 30) || p.mid_cp < 1 || p.mid_cp > 32 || p.mfrags0 < (p.small && HSTORE ? 1 : 2) || p.out_cp < 8 || p.out_cp > 64 ||
        p.out_cp % 8 != 0 || p.tiles_x != cols || p.tiles_y != rows || tiles > 4000000 || p.rcp_tiles_x != 1.0f / (float)p.tiles_x || p.groups < 1 || p.groups > tiles || p.nreset < 0 || p.nreset > 4 || (p.small && (p.mid_cp > 16 || p.out_cp > 32)) ||
        (p.mid && (p.mid_cp % (HSTORE && !p.small ? 8 : 4) != 0 || p.mid_off < 0 || p.mid_wp < p.w + p.mid_off)))
        return -5;
    const auto kernel = p.small ? (p.mid ? conv_a16_kernel<HSTORE, true, true> : conv_a16_kernel<HSTORE, false, true>)
                                : (p.mid ? conv_a16_kernel<HSTORE, true, false> : conv_a16_kernel<HSTORE, false, false>);
    const size_t lds = p.small ? GeoA<true>::LDS : GeoA<false>::LDS;
    if (ensure_lds(reinterpret_cast<const void*>(kernel), lds) != 0) return -2;
    hipLaunchKernelGGL(kernel, dim3((unsigned)p.groups), dim3(512), lds, s, p);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace fynhip
