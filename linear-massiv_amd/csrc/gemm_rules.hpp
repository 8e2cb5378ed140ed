// The rules that choose a product's kernel by its shape, on the host alone:
// estimated times (us) of the two kernels, fitted to measured products.
#pragma once

#include <cstdint>

namespace lmx {

// Tile shapes of the plain (non-batched, non-SYRK) GEMM dispatch.
enum GemmTile { TILE_DEFAULT = 0, TILE_64x64 = 1, TILE_128x64 = 2, TILE_128x128 = 3 };
inline int64_t rule_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
// Tiles of a grid, or of its lower trapezoid (rows >= columns).
inline int64_t rule_tiles(int64_t rows, int64_t cols, bool lower) {
    return lower ? cols * (cols + 1) / 2 + (rows - cols) * cols : rows * cols;
}

// The tile of gemm_ksplit_kernel (16 mt x 16 nt): the largest that still gives
// KS_FILL workgroups (one a CU), else the smallest; and the workgroups it has.
constexpr int64_t KS_FILL = 256;
constexpr int KS_MIN_K = 48;
struct KsTile {
    int mt, nt;
    int64_t count;
};
inline KsTile ksplit_tile(int64_t m, int64_t n, bool lower, int64_t batch) {
    const int64_t t16 = rule_cdiv(m, 16), u16 = rule_cdiv(n, 16), t32 = rule_cdiv(m, 32), u32 = rule_cdiv(n, 32);
    if ((lower ? t32 * u32 / 2 : t32 * u32) * batch >= KS_FILL)
        return {2, 2, rule_tiles(t32, u32, lower) * batch};
    if (!lower && t16 * u32 * batch >= KS_FILL) return {1, 2, t16 * u32 * batch};
    return {1, 1, rule_tiles(t16, u16, lower) * batch};
}

// gemm_ksplit_kernel or the 64 x 64 tiles, for fewer of those than CUs (`nn`:
// gemm_nn_kernel would take them): whichever the two's times say (us).  The
// tiles take one round, bound by its k loop; the split takes a round of the CUs
// for every 256 of its smaller tiles, and each has its start and its sum
// through LDS.  So with nearly a tile a CU and a short k there is nothing to
// gain (FP64 960 x 960 x 64 7.7 against 14.2 us, 16000 x 64 x 48 6.8 against
// 12.6), with a long k or few tiles much (500 x 500 x 500 32 -> 10 us).
//   The times are fitted to 1168 products (FP64 and FP32, every transpose, k
// from 48 to 8192), where they choose the slower kernel by more than 3% in 5 of
// the cases that the tiles win (11% at most); the split for all of them was
// slower in 75, up to 1.85 times.
inline bool ksplit_is_faster(int bytes, const KsTile &t, bool nn, bool tb, int64_t k) {
    const bool D = bytes == 8;
    const double kk = (double)k, r = (double)rule_cdiv(t.count, 256);
    const double tiles = 3.8 + kk * (D ? (nn ? 0.057 : 0.066) : (nn ? 0.0295 : 0.0425));
    double split;
    if (t.mt == 2 && nn)  // several rounds of operands that the NN kernel reads from LDS
        split = D ? 1.9 + r * (2.1 + (tb ? 0.0128 : 0.0115) * kk) : 2.35 + r * (1.2 + 0.0064 * kk);
    else if (t.mt == 2)
        split = D ? 1.9 + r * (1.9 + 0.0106 * kk) : 2.35 + r * (0.7 + 0.0064 * kk);
    else if (t.nt == 2)
        split = D ? 0.7 + r * (1.34 + 0.0075 * kk) : 0.6 + r * (1.2 + 0.0041 * kk);
    else
        split = D ? 3.0 + r * (0.14 + 0.0038 * kk) : 3.1 + r * (0.03 + 0.002 * kk);
    return split < tiles;
}

// gemm_direct_kernel or the tiles through LDS, for an FP64 product on an idle
// device: whichever the two's times say (us), one tile a CU a round.  Both are
// bound by the matrix cores within a round, so what decides is how the output
// divides: a direct tile has 64 x 128, of which n <= 64 wastes half, and 129
// columns or a grid just past a round of the CUs a third, where 64 x 64 tiles
// waste little.
//   The times are fitted to 1043 products (m, n from 1 to 100000, k from 64 to
// 4096, every transpose, rows aligned and not), where they choose the slower
// kernel by more than 3% in 8 of the cases that the tiles win (6% at most);
// taking the direct kernel from 140 tiles on had 361 slower ones, up to 1.8
// times (32668 x 4 x 78: 9.7 against 17.4 us, 40000 x 64 x 256 36 against 57,
// 9000 x 192 x 1024 92 against 134), and 7% more time over all.
//   Aligned A B^T is not in it: 51.7 TF through LDS, 49.9 TF direct at 4096^3
// (both operands cost 16 lines a load).  Nor is FP32, whose MFMA takes half the
// time for half the bytes: it lost everywhere.
constexpr int DIRECT_MIN_K = 64;
inline bool direct_is_faster(bool ta, bool tb, bool nn, int tile, int64_t m, int64_t n, int64_t k) {
    auto rounds = [&](int64_t bm, int64_t bn) { return (double)rule_cdiv(rule_cdiv(m, bm) * rule_cdiv(n, bn), 256); };
    const double kk = (double)k;
    // one transpose of the two: the operands cost fewer lines
    const double direct = 3.2 + rounds(64, 128) * (3.9 + (ta != tb ? 0.0600 : 0.0645) * kk);
    double tiles;
    if (tile == TILE_64x64) {
        // a round or less is gemm_ksplit_kernel's (16 x 16 x 8192: 30 us, one
        // direct tile 490)
        const double r = rounds(64, 64);
        if (r < 2) return false;
        // the first tiles of a CU hide each other's latency
        const double first[2] = {nn ? 0.088 : 0.097, nn ? 0.119 : 0.131};
        tiles = 1.5 + 2.0 * r + kk * (r <= 3 ? first[(int)r - 2] : r * (nn ? 0.0405 : 0.045));
    } else if (tile == TILE_128x64) {
        tiles = 1.5 + rounds(128, 64) * (3.0 + (nn ? 0.082 : 0.1) * kk);
    } else {
        tiles = 1.5 + rounds(128, 128) * (6.0 + 0.188 * kk);
    }
    return direct < tiles;
}

// The tile (256 or 128) that gemm_bf16_large_kernel takes a product with, 0
// where the 128 x 128 x 32 and 64 x 64 x 32 tiles of gemm_bf16_kernel are the
// faster ones: whichever the times say (us, `w` million elements of C).
//   Rounds over the chip: one 256 x 256 tile a CU or two 128 x 128; a round of
// the former takes 40 / 23 of the latter's time (2048 x 4096 x 8192 NT: 206
// against 160 us, one round each).  Below BX_MIN_TILES the 64 x 64 tiles spread
// better (1024^3 NT: 15.0 against 19.3 us).  A large tile's start and its C
// cost 5 to 12 us a round, which its k steps have to pay for: 2048 x 2048 x 8
// took 8.4 us in place of 6.5, 13216 x 40 x 8 6.9 in place of 3.8.
//   The times are fitted to 637 products (m, n from 8 to 65536, k from 8 to
// 8192, every transpose), where they choose the slower kernel by more than 3%
// in 10 of the cases that the smaller steps win (14% at most); the large tiles
// for all of them were slower in 328, up to 1.83 times, and gained nothing over
// all, against 11% now.
constexpr int64_t BX_MIN_TILES = 100;
inline int bf16_large_tile(bool ta, bool tb, int64_t m, int64_t n, int64_t k) {
    const int64_t t256 = rule_cdiv(m, 256) * rule_cdiv(n, 256), t128 = rule_cdiv(m, 128) * rule_cdiv(n, 128);
    if (t128 < BX_MIN_TILES) return 0;
    const int tile = 40 * rule_cdiv(t256, 256) <= 23 * rule_cdiv(t128, 512) ? 256 : 128;
    // us of one round per k: NN, NT, TN, TT
    static const double first256[4] = {0.0307, 0.0291, 0.0342, 0.0312}, more256[4] = {0.0343, 0.0330, 0.0355, 0.0345},
                        one128[4] = {0.0147, 0.0129, 0.0177, 0.0151}, two128[4] = {0.0184, 0.0166, 0.0214, 0.0194},
                        small128[4] = {0.0145, 0.0122, 0.0190, 0.0150},
                        small64[3][4] = {{0.0170, 0.0136, 0.0207, 0.0172},
                                         {0.0084, 0.0078, 0.0105, 0.0091},
                                         {0.0074, 0.0053, 0.0097, 0.0074}};
    const int f = 2 * ta + tb;
    const double kk = (double)k, w = (double)m * (double)n * 1e-6;
    double large, small;
    if (tile == 256) {
        const double r = (double)rule_cdiv(t256, 256);
        large = r == 1 ? 12.2 + 0.11 * w + first256[f] * kk : 0.9 * w + r * more256[f] * kk;
    } else if (t128 <= 256) {  // one tile a CU
        large = 4.5 + 1.05 * w + one128[f] * kk;
    } else {
        large = 5.0 + 0.77 * w + (double)rule_cdiv(t128, 512) * two128[f] * kk;
    }
    if (t128 >= 512) {
        small = 4.3 + 0.68 * w + (double)rule_cdiv(t128, 256) * small128[f] * kk;
    } else {
        const int64_t r = rule_cdiv(rule_cdiv(m, 64) * rule_cdiv(n, 64), 256);
        small = 2.7 + (r < 5 ? 0.9 : 0.68) * w + (double)r * small64[r < 3 ? r - 1 : 2][f] * kk;
    }
    return large < small ? tile : 0;
}

}  // namespace lmx
