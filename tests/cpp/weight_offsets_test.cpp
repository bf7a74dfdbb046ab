// Convolution forms whose kernels reach their packed weights through 32-bit offsets, asked on the host for layers around that
// limit: "no such combination" is what takes a layer to another form.  One check per call, named by the argument; exit status
// 0: it holds.  Nothing is launched: calls within the limit ask for the LDS size only.
#include <cstdio>
#include <cstring>

#include "../../fyusenet_amd/csrc/kernels.h"

using namespace fynhip;

#define CHECK(x)                                              \
    do {                                                      \
        if (!(x)) {                                           \
            fprintf(stderr, "line %d: %s\n", __LINE__, #x);   \
            return 1;                                         \
        }                                                     \
    } while (0)

// a 3x3 layer of cin -> cout channels (multiples of 256) on 64x64 positions
static ConvP16Params layer(int cin, int cout, int th, int tw, int wm, bool f16) {
    ConvP16Params p{};
    const int twg = (4 / wm) * tw;
    p.in_hp = p.in_wp = 66; p.in_cp = cin; p.stride = 1;
    p.npos_y = p.npos_x = 64; p.out_wp = 64; p.out_cp = cout;
    p.tile_h = th; p.tile_w = tw; p.wm = wm;
    p.tiles_x = (64 + twg - 1) / twg; p.tiles_y = (64 + th - 1) / th;
    p.rcp_tiles_x = 1.0f / (float)p.tiles_x;
    p.pos_groups = 1;
    p.cin_chunks = cin / 32; p.mfrags = cout / 16; p.cout_blocks = cout / (32 * wm);
    p.f16 = f16 ? 1 : 0;
    return p;
}

// conv_p16, tiles whose fragments are rows of sixteen positions
static int p16_rows() {
    static unsigned amax;   // (a value-range word: the fp8 form; its address is all that is looked at)
    const int rows[][2] = {{8, 4}, {6, 4}, {5, 4}, {4, 4}, {6, 2}, {4, 2}};
    for (auto& t : rows) {
        // 6144 -> 6144 channels: 192 chunks x 9 taps x 384 fragments x 3 KB = 2.04e9 bytes; 9216 -> 9216: 4.6e9; 6400 -> 6400: 2.2e9
        for (int channels : {6144, 6400, 9216}) {
            ConvP16Params p = layer(channels, channels, t[0], 16, t[1], false);
            p.in_amax = &amax;
            if (channels == 6144) {
                CHECK(conv_p16_lds_bytes(p) != 0);
            } else {
                CHECK(conv_p16_lds_bytes(p) == 0);
                CHECK(launch_conv_p16(p, nullptr) == -1);
            }
        }
    }
    // the other tiles walk their weights by pointer
    CHECK(conv_p16_lds_bytes(layer(9216, 9216, 8, 10, 4, false)) != 0);
    CHECK(conv_p16_lds_bytes(layer(9216, 9216, 4, 8, 2, false)) != 0);
    CHECK(conv_p16_lds_bytes(layer(16384, 16384, 8, 8, 4, true)) != 0);
    return 0;
}

// conv_h16 (wide fp16 tensors): a layer that it cannot take has no candidates and keeps the forms behind it
static int h16() {
    for (int k : {3, 9})
        for (int rows : {12, 10, 8, 6, 5, 4}) {
            // 9x9: 3584 -> 3584 channels 2.08e9 bytes, 3712 -> 3712 2.23e9; 3x3: 10752 -> 10752 2.08e9, 11008 -> 11008 2.18e9
            ConvP16Params p = layer(k == 9 ? 3584 : 10752, k == 9 ? 3584 : 10752, rows, 8, 4, true);
            CHECK(conv_h16_lds_bytes(p, k) != 0);
            p = layer(k == 9 ? 3712 : 11008, k == 9 ? 3712 : 11008, rows, 8, 4, true);
            CHECK(conv_h16_lds_bytes(p, k) == 0);
            CHECK(launch_conv_h16(p, k, nullptr) == -1);
        }
    return 0;
}

int main(int argc, char** argv) {
    if (argc == 2 && !strcmp(argv[1], "h16")) return h16();
    if (argc == 2 && !strcmp(argv[1], "p16_rows")) return p16_rows();
    return 2;
}
