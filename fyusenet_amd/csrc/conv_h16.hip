// K x K convolution (K = 3 or 9, stride 1) between wide layers with fp16 storage -- the residual blocks of a
// style-transfer net at full resolution -- as an implicit GEMM on gfx950 matrix cores with 16-position fragments
// (v_mfma_f32_16x16x32_f16, fp32 accumulate), one MFMA per fragment pair.
//
// Replaces, for such layers, the render passes of DeepConvLayerNxN::forward (fyusenet/gpu/deep/deepconvlayerNxN.cpp:
// 129-211); epilogue order of shaders/deep/deepconv3x3_tiled.frag:36-45 (acc*scale + bias, then the residual).
//
// Why another MFMA kernel: these layers run for hundreds of microseconds, and what bounds them is how the operands reach
// the matrix cores.  A fragment here is one row of sixteen positions, so the fragment that output row r needs at tap row
// ky is the one row r + 1 needed at ky - 1: the taps are walked column by column (kx outside, ky inside), a wave keeps
// the TH fragments of its tile's rows in registers and every step replaces one of them.  A kernel column of K steps
// reads TH + K - 1 fragments from LDS instead of TH * K (20 instead of 108 for K = 9, TH = 12).  That makes the position
// side so cheap that the four MFMA waves can each take 32 output channels of the workgroup's 128 and ALL of its
// positions: no two waves load the same weights, 21 bytes per MFMA cycle and CU through the L1 (which delivers 64) and 23
// from LDS (128), where two groups of 64 channels x two tiles of positions took 43 and 64.
// Measured, fp16: 9x9 128 -> 128 at 464x381 positions (469 GFLOP) 290-297 us a layer in a frame = 1.58-1.62 PFLOP/s, what the
// library reaches on a 16384^3 product here (1.63).  Twenty launches of a layer in a row on one card, before and now: 313-326 and
// 272-286 us; 352x225 167 and 139; 3x3 128 -> 128 at 156x128 (5.9 GFLOP) 11.4 and 8.4.
// Bound: the matrix pipes at the clock the part holds under them (79 % busy at 1.95-2.0 GHz in the launch of 12-row
// tiles; without any operand traffic the same loop is 90 % busy at 2.2).  Weights requested 2, 3, 4 or 8 steps ahead,
// results stored by the staging waves, and the weights brought into the L2 ahead of use: no difference.
//
// GEMM view: M = output channels (A = weights, packed per lane, streamed through L2/L1 into a register ring), N = positions (B = activations, a halo tile of one 32-channel chunk in LDS), K = taps x channels, one tap of one
// chunk per step.  The code of nine steps is unrolled: one kernel column of the 9x9 kernel (the columns are a loop that
// moves one base register by a pixel), the whole chunk of a 3x3 kernel.
//
// Workgroup = 4 staging waves + 4 MFMA waves (32 output channels each x TH rows of 16 positions).  The weights are packed
// so that a lane's eight accumulators of a row are eight consecutive output channels of one position: no transposition in
// the epilogue, one 16-byte store per lane and row; residual (staged to LDS by the staging waves during a tile's last
// chunk) and scale/bias from LDS.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <type_traits>

#include "kernels.h"
#include "p16_common.h"

namespace fynhip {

namespace {
constexpr int HNS = 9;    // unrolled steps, and slots of the weight-fragment ring
constexpr int HFM = 2;    // fragments of 16 output channels per wave

// (TW_: the workgroup's tile is two times TW_ = 8 columns wide, the sixteen positions of a fragment)
template <int K_, int TH_, int TW_>
struct GeoH {
    static constexpr int K = K_, TH = TH_, TW = TW_;
    static constexpr int WM = 4, TWG = 2 * TW;
    static constexpr int HW = TWG + K - 1, HH = TH + K - 1;
    static constexpr int ROW_PITCH = HW * PITCH + p16_row_pad(TH, TWG, 1, 1, HW);
    static constexpr int BUF = HH * ROW_PITCH;            // one staging buffer (fp16 storage: one plane)
    static constexpr int FN = TH;                         // position fragments: rows of the tile
    // steps from the request of a weight fragment to its use (so many slots of the ring are registers; eight are no faster)
    static constexpr int LEAD = (K == 3 && TH > 10) ? 2 : 3;
    static constexpr int NITEMS = HH * HW * (KC / 8);     // staging items: (pixel, 8 channels)
    static constexpr int NB = (NITEMS + 255) / 256;
    static constexpr int CPB = 16 * HFM * WM;             // output channels per workgroup
    static constexpr int RES_PITCH = CPB * 2 + 16;        // bytes per position of the residual tile
    static constexpr int RPIECES = TH * TWG * (CPB / 8);  // residual 16-byte pieces
    static constexpr int RNB = RPIECES / 256;
    static_assert(RPIECES % 256 == 0, "whole turns of the staging threads");
    static_assert(TWG == 16, "a fragment is a row of the tile");
    static_assert(HNS % K == 0 && (K * K) % HNS == 0, "the unrolled steps are whole kernel columns");
    static_assert(HH * ROW_PITCH + K * PITCH < 65536, "offsets inside a staging buffer fit the LDS instructions' immediate field");
};

// Nine steps of a stage: HNS / K kernel columns of K taps each.  `col`: per-lane LDS offset of (row 0, first of these
// columns); `next_col`: the same for the column behind the last one (LAST: the first column of the next stage, in the
// other staging buffer -- the stage's barrier sits in front of the first such read; the staging waves have filled that
// buffer by then, and all reads of this stage's buffer were issued a step earlier).  The fragment of input row r lives in
// slot r % TH: at tap row ky the live rows are ky .. ky + TH - 1, the slots are used in their order, and the one that held
// row ky takes row ky + TH behind its last MFMA; a column's last step refills every slot with the next column's rows 0 ..
// TH - 1.  A refilled slot is used a whole step later.  One slot of the schedule per MFMA: the MFMA, then a share of the
// step's memory instructions, fenced so that the compiler keeps the order.  A step also
// requests the weights of the step LEAD further on.
template <class G, bool LAST>
__device__ __forceinline__ void h16_steps(f32x4_t (&acc)[HFM][G::FN], half8_t (&a_q)[HNS][HFM], half8_t (&b)[G::FN], int col, int next_col,
                                          const unsigned char* lds, const __amdgpu_buffer_rsrc_t weights, unsigned& wnext, unsigned wend, unsigned wstep,
                                          unsigned wlane) {
    constexpr int FN = G::FN, K = G::K;
    typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int d = 0; d < HNS; d++) {
        const int kx = d / K, ky = d % K;
        const unsigned w_ = wnext;
        wnext += wstep;
        if (wnext == wend) wnext = 0;
#pragma unroll
        for (int i = 0; i < HFM * FN; i++) {
            const int slot = i / HFM, fm = i % HFM;
            const int row = ((slot - ky) % FN + FN) % FN;   // the output row whose fragment this slot holds
            acc[fm][row] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_q[d][fm], b[slot], acc[fm][row], 0, 0, 0);
            if (LAST && d == HNS - 1 && i == 0) lds_barrier();
            if (fm == HFM - 1) {
                if (ky + 1 < K) {
                    if (row == 0) b[slot] = *reinterpret_cast<const half8_t*>(lds + col + kx * PITCH + (ky + FN) * G::ROW_PITCH);
                } else if (d + 1 < HNS) {
                    b[slot] = *reinterpret_cast<const half8_t*>(lds + col + (kx + 1) * PITCH + slot * G::ROW_PITCH);
                } else {
                    b[slot] = *reinterpret_cast<const half8_t*>(lds + next_col + slot * G::ROW_PITCH);
                }
            }
#pragma unroll
            for (int j = 0; j < HFM; j++)   // the weight fragments, spread over the step's slots
                if (i == j * FN + 1) a_q[(d + G::LEAD) % HNS][j] = __builtin_bit_cast(half8_t, (u32x4_t)__builtin_amdgcn_raw_buffer_load_b128(weights, wlane + j * 1024, w_, 0));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The staging waves (threads 0..255): stage after stage -- a 32-channel chunk of a tile's halo: global loads, activation,
// LDS writes -- one stage ahead of the MFMA waves, across tile boundaries; scale and bias at the start and, during a
// tile's last chunk, its residual tile.  One barrier per stage, after the one that hands over the first.  (A stage of
// the MFMA waves lasts thousands of cycles; the staging waves spend most of it waiting at the barrier.)
template <class G>
__device__ __forceinline__ void h16_stager(const ConvP16Params& p, unsigned char* lds, int stid, int cb, int group, int ntiles, int nchunks) {
    constexpr int CPB = G::CPB;
    constexpr int sb_off = 2 * G::BUF;
    constexpr int res_off = sb_off + 2 * CPB * 4;
    const _Float16* in = reinterpret_cast<const _Float16*>(p.in);
    int i_y[G::NB], i_x[G::NB], l_off[G::NB];
#pragma unroll
    for (int i = 0; i < G::NB; i++) {
        const int idx = stid + i * 256;
        l_off[i] = -1; i_y[i] = 1 << 20; i_x[i] = 0;
        if (idx < G::NITEMS) {
            const int pix = idx >> 2, g = idx & 3;
            const int py = pix / G::HW, px = pix - py * G::HW;
            i_y[i] = py; i_x[i] = px;
            l_off[i] = py * G::ROW_PITCH + px * PITCH + g * 16;
        }
    }
    const int g8 = (stid & 3) * 8;
    int g_off[G::NB];          // element offsets of the items, -1: outside the frame (reads as 0)
    half8_t raw[G::NB];
    // (unconditional loads: items outside the tensor read its first element and are zeroed when stored)
    auto fetch = [&](int tile, int chunk) {
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        const int y0 = tyi * G::TH + p.in_y0, x0 = txi * G::TWG + p.in_x0;
#pragma unroll
        for (int i = 0; i < G::NB; i++) {
            int gy = y0 + i_y[i], gx = x0 + i_x[i];
            if (p.in_clamp && l_off[i] >= 0) {
                gy = min(max(gy, 0), p.in_hp - 1);
                gx = min(max(gx, 0), p.in_wp - 1);
            }
            g_off[i] = ((unsigned)gy < (unsigned)p.in_hp && (unsigned)gx < (unsigned)p.in_wp) ? (gy * p.in_wp + gx) * p.in_cp + g8 + chunk * KC : -1;
            raw[i] = *reinterpret_cast<const half8_t*>(in + (g_off[i] >= 0 ? g_off[i] : 0));
        }
    };
    auto store = [&](unsigned char* buf) {
#pragma unroll
        for (int i = 0; i < G::NB; i++) {
            if (l_off[i] < 0) continue;
            const bool ok = g_off[i] >= 0;
            half8_t v;
            _Float16 hlo, hhi;
            if (act_half_exact(p.act, hlo, hhi)) {
                // (on the packed halves: two instructions per item instead of seven per value; the staging waves share their
                // SIMDs' issue slots with the MFMA waves)
                v = ok ? act_half(raw[i], hlo, hhi) : (half8_t)((_Float16)0.f);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = ok ? (_Float16)act_p16((float)raw[i][e], p.act) : (_Float16)0.f;
            }
            *reinterpret_cast<half8_t*>(buf + l_off[i]) = v;
        }
    };
    auto residual_in = [&](int tile) {   // the residual tile of a tile: [position][CPB channels] fp16
        const _Float16* res = reinterpret_cast<const _Float16*>(p.res);
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        half8_t rv[G::RNB];
#pragma unroll
        for (int i = 0; i < G::RNB; i++) {
            const int idx = stid + i * 256;
            const int m = idx / (CPB / 8), c8 = idx % (CPB / 8);
            const int ty = m / G::TWG, tx = m - ty * G::TWG;
            const int py = tyi * G::TH + ty, px = txi * G::TWG + tx;
            const bool ok = py < p.npos_y && px < p.npos_x;
            rv[i] = *reinterpret_cast<const half8_t*>(res + (ok ? ((size_t)(p.res_off_y + py) * p.res_wp + p.res_off_x + px) * p.res_cp + cb * CPB + c8 * 8 : 0));
        }
#pragma unroll
        for (int i = 0; i < G::RNB; i++) {
            const int idx = stid + i * 256;
            *reinterpret_cast<half8_t*>(lds + res_off + (idx / (CPB / 8)) * G::RES_PITCH + (idx % (CPB / 8)) * 16) = rv[i];
        }
    };
    auto advance = [&](int& tile, int& c) {
        if (++c == nchunks) { c = 0; tile += p.pos_groups; }
        return tile < ntiles;
    };
    int tile = group, c = 0;          // the stage the MFMA waves are on (stage n)
    int t1 = group, c1 = 0;           // stage n+1
    fetch(tile, 0);
    bool have1 = advance(t1, c1);
    if (stid < CPB) {
        reinterpret_cast<float*>(lds + sb_off)[stid] = p.scale[cb * CPB + stid];
        reinterpret_cast<float*>(lds + sb_off)[CPB + stid] = p.bias[cb * CPB + stid];
    }
    store(lds);
    lds_barrier();
    int buf = 0;                      // the buffer of stage n
    for (;;) {
        if (have1) fetch(t1, c1);
        if (c + 1 == nchunks && p.res) residual_in(tile);
        if (have1) store(lds + (1 - buf) * G::BUF);
        lds_barrier();
        if (!have1) break;
        tile = t1; c = c1; buf = 1 - buf;
        have1 = advance(t1, c1);
    }
}

// Grid: cout_blocks x pos_groups workgroups; a workgroup keeps its block of 128 output channels and walks the tiles
// group, group + pos_groups, ...
template <int K, int TH, int TW>
__global__ __launch_bounds__(512) void conv_h16_kernel(const ConvP16Params p) {
    using G = GeoH<K, TH, TW>;
    constexpr int FN = G::FN, CPB = G::CPB;
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroups are dealt round-robin to the 8 XCDs; remap so that neighbouring tiles (shared halos) meet in one L2.
    int bid = blockIdx.x;
    {
        const int nblk = p.pos_groups * p.cout_blocks;
        const int per = nblk >> 3;
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const int cb = bid % p.cout_blocks;
    const int group = bid / p.cout_blocks;
    const int ntiles = p.tiles_x * p.tiles_y;
    const int nchunks = p.cin_chunks;
    constexpr int sb_off = 2 * G::BUF;
    constexpr int res_off = sb_off + 2 * CPB * 4;

    if (wave < 4) {   // the first four waves stage: they start first
        h16_stager<G>(p, lds, tid & 255, cb, group, ntiles, nchunks);
        return;
    }

    // ---------------------------------------------------------------------- MFMA waves
    const int mq = lane & 15, kq = lane >> 4;
    const int mw = wave - 4;   // this wave's 32 output channels of the workgroup's 128
    const int base = mq * PITCH + kq * 16;   // per-lane LDS offset of the fragments at row 0, tap column 0 in staging buffer 0
    // A fragments: [(chunk*K + kx)*K + ky][cout fragment of 16][lane] x 8 halves
    const unsigned wstep = (unsigned)p.mfrags * 1024;
    const unsigned char* wbase = reinterpret_cast<const unsigned char*>(p.wpack) + (size_t)(cb * (CPB / 16) + mw * HFM) * 1024;   // (uniform)
    const unsigned wlane = lane * 16;
    const unsigned wend = (unsigned)(nchunks * K * K) * wstep;
    // (as a buffer: the step's offset is a scalar operand of the load, no address arithmetic per lane)
    const __amdgpu_buffer_rsrc_t weights = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(wbase), 0, (int)wend, 0x00020000);
    half8_t a_q[HNS][HFM];
#pragma unroll
    for (int d = 0; d < G::LEAD; d++)
#pragma unroll
        for (int fm = 0; fm < HFM; fm++) a_q[d][fm] = *reinterpret_cast<const half8_t*>(wbase + (size_t)d * wstep + fm * 1024 + wlane);
    f32x4_t acc[HFM][FN];
    auto zero_acc = [&]() {
#pragma unroll
        for (int fm = 0; fm < HFM; fm++)
#pragma unroll
            for (int fn = 0; fn < FN; fn++) acc[fm][fn] = (f32x4_t)(0.f);
    };
    zero_acc();
    const bool res_scale = p.res_scale != 0;
    const float res_floor = p.res_relu ? 0.f : -__builtin_inff();

    auto finish_tile = [&](int tile) {
        const float* sb = reinterpret_cast<const float*>(lds + sb_off);
        f32x4_t rs[HFM], bi[HFM], scm[HFM];
#pragma unroll
        for (int fm = 0; fm < HFM; fm++) {
            const f32x4_t sc = *reinterpret_cast<const f32x4_t*>(sb + mw * 32 + kq * 8 + fm * 4);
            bi[fm] = *reinterpret_cast<const f32x4_t*>(sb + CPB + mw * 32 + kq * 8 + fm * 4);
            scm[fm] = sc * p.acc_mul;
            rs[fm] = res_scale ? sc : (f32x4_t)(1.f);
        }
        // a lane's eight channels of each row
        const int tyi = (int)(((float)tile + 0.5f) * p.rcp_tiles_x), txi = tile - tyi * p.tiles_x;
        const int px = txi * G::TWG + mq;
        _Float16* out = reinterpret_cast<_Float16*>(p.out) + ((size_t)(p.out_off_y + tyi * TH) * p.out_wp + p.out_off_x + px) * p.out_cp + cb * CPB + mw * 32 + kq * 8;
        const int row_pitch = p.out_wp * p.out_cp;
        const int nrows = px < p.npos_x ? p.npos_y - tyi * TH : 0;
        auto rows = [&](auto residual) {
#pragma unroll
            for (int ty = 0; ty < FN; ty++) {
                half8_t rv, hv;
                if constexpr (decltype(residual)::value)
                    rv = *reinterpret_cast<const half8_t*>(lds + res_off + (ty * G::TWG + mq) * G::RES_PITCH + (mw * 32 + kq * 8) * 2);
#pragma unroll
                for (int fm = 0; fm < HFM; fm++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float v = acc[fm][ty][e] * scm[fm][e] + bi[fm][e];
                        if constexpr (decltype(residual)::value) v = fmaf(fmaxf((float)rv[fm * 4 + e], res_floor), rs[fm][e], v);
                        hv[fm * 4 + e] = (_Float16)v;
                    }
                if (ty < nrows) *reinterpret_cast<half8_t*>(out + (size_t)ty * row_pitch) = hv;
                if (ty % 3 == 2) __builtin_amdgcn_sched_barrier(0);   // (no more than three rows' residuals at a time in registers)
            }
        };
        if (p.res) rows(std::true_type());
        else rows(std::false_type());
    };

    lds_barrier();   // the first stage is staged
    half8_t b[FN];
#pragma unroll
    for (int r = 0; r < FN; r++) b[r] = *reinterpret_cast<const half8_t*>(lds + base + r * G::ROW_PITCH);
    unsigned wnext = G::LEAD * wstep;
    int tile = group, c = 0, buf = 0;
    for (;;) {
        int col = base + buf * G::BUF;
        for (int kx = HNS / K; kx < K; kx += HNS / K) {
            h16_steps<G, false>(acc, a_q, b, col, col + HNS / K * PITCH, lds, weights, wnext, wend, wstep, wlane);
            col += HNS / K * PITCH;
        }
        buf = 1 - buf;
        h16_steps<G, true>(acc, a_q, b, col, base + buf * G::BUF, lds, weights, wnext, wend, wstep, wlane);
        if (++c == nchunks) {
            finish_tile(tile);
            c = 0; tile += p.pos_groups;
            if (tile >= ntiles) break;
            zero_acc();
        }
    }
}

struct H16Entry {
    int k, th, tw;
    void (*fn)(const ConvP16Params);
    size_t buf_bytes, res_bytes;
};
template <int K, int TH, int TW>
constexpr H16Entry h16_entry() {
    using G = GeoH<K, TH, TW>;
    return H16Entry{K, TH, TW, conv_h16_kernel<K, TH, TW>, (size_t)(2 * G::BUF + 2 * G::CPB * 4), (size_t)(TH * G::TWG * G::RES_PITCH)};
}
const H16Entry H16_TABLE[] = {
    h16_entry<9, 12, 8>(), h16_entry<9, 10, 8>(), h16_entry<9, 8, 8>(), h16_entry<9, 6, 8>(), h16_entry<9, 5, 8>(), h16_entry<9, 4, 8>(),
    h16_entry<3, 12, 8>(), h16_entry<3, 10, 8>(), h16_entry<3, 8, 8>(), h16_entry<3, 6, 8>(), h16_entry<3, 5, 8>(), h16_entry<3, 4, 8>(),
};
constexpr int H16_COUNT = sizeof(H16_TABLE) / sizeof(H16_TABLE[0]);
const H16Entry* h16_find(const ConvP16Params& p, int k) {
    for (int i = 0; i < H16_COUNT; i++)
        if (H16_TABLE[i].k == k && H16_TABLE[i].th == p.tile_h && H16_TABLE[i].tw == p.tile_w)
            return (size_t)p.cin_chunks * k * k * p.mfrags * 1024 < (size_t)1 << 31 ? &H16_TABLE[i] : nullptr;   // (offsets into the weights are 32 bits wide)
    return nullptr;
}
}  // namespace

bool conv_h16_supported(int k, int stride, int dil, int in_cp, int cout, int out_cp, bool f16_storage) {
    bool have_k = false;
    for (int i = 0; i < H16_COUNT; i++) have_k = have_k || H16_TABLE[i].k == k;
    return f16_storage && have_k && stride == 1 && dil == 1 && in_cp % KC == 0 && cout % 128 == 0 && out_cp >= cout;
}
int conv_h16_tile_count() { return H16_COUNT; }
void conv_h16_tile(int i, int* k, int* th, int* tw) {
    *k = H16_TABLE[i].k; *th = H16_TABLE[i].th; *tw = H16_TABLE[i].tw;
}
size_t conv_h16_lds_bytes(const ConvP16Params& p, int k) {
    const H16Entry* e = h16_find(p, k);
    if (!e) return 0;
    return e->buf_bytes + (p.res ? e->res_bytes : 0);
}
int launch_conv_h16(const ConvP16Params& p, int k, hipStream_t s) {
    const H16Entry* e = h16_find(p, k);
    if (!e) return -1;
    // what the kernel and its grid assume
    if (p.cin_chunks < 1 || p.in_cp < p.cin_chunks * KC || p.mfrags % 8 != 0 || p.cout_blocks * 8 != p.mfrags || p.out_cp < p.cout_blocks * 128 ||
        (p.res && p.res_cp < p.cout_blocks * 128) || (p.res && p.cin_chunks < 2 && p.pos_groups != p.tiles_x * p.tiles_y) ||
        p.pos_groups < 1 || p.pos_groups > p.tiles_x * p.tiles_y || p.tiles_x < 1 || p.tiles_y < 1 || !p.f16 ||
        p.rcp_tiles_x != 1.0f / (float)p.tiles_x || p.tiles_x * p.tiles_y > 4000000 || p.in_cp % 8 != 0 || p.out_cp % 8 != 0 || (p.res && p.res_cp % 8 != 0) ||
        p.tiles_x * 2 * e->tw < p.npos_x || p.tiles_y * e->th < p.npos_y || !p.in || !p.out || !p.wpack || !p.scale || !p.bias)
        return -1;
    const size_t lds = conv_h16_lds_bytes(p, k);
    if (ensure_lds(reinterpret_cast<const void*>(e->fn), lds) != 0) return -2;
    hipLaunchKernelGGL(e->fn, dim3((unsigned)(p.pos_groups * p.cout_blocks)), dim3(512), lds, s, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fynhip
