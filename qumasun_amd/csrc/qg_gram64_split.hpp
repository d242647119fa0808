// qg_gram64_split.hpp — how the FP64 Gram kernel (qg_dense64.hip) cuts a product, and where it is faster
// than the library's product: host arithmetic without HIP, also compiled by the tests.
#pragma once
#include <algorithm>
#include <cstdint>

namespace qg {

struct GramSplit {
    int mb, nb, bm, bn;     // blocks, and the tiles (16 x 16) of the largest
    int64_t nch, per;       // ranges of points, points of one
};

// The tiles in the fewest blocks of at most 10 x 12, as even as they go; one workgroup per CU in all (its
// accumulators take the registers), or up to four rounds of them where the blocks alone come near that; no
// range shorter than 512 points
inline GramSplit gram64_split(int64_t K, int M, int N) {
    GramSplit g;
    const int mt = (M + 15) / 16, nt = (N + 15) / 16;
    g.mb = (mt + 9) / 10;
    g.nb = (nt + 11) / 12;
    g.bm = (mt + g.mb - 1) / g.mb;
    g.bn = (nt + g.nb - 1) / g.nb;
    const int64_t blocks = (int64_t)g.mb * g.nb;
    const int64_t want = std::min<int64_t>((K + 511) / 512, std::max<int64_t>(1, (blocks <= 32 ? 256 : 1024) / blocks));
    g.per = ((K + want - 1) / want + 15) / 16 * 16;
    g.nch = (K + g.per - 1) / g.per;
    return g;
}

// Tiles of the fullest SIMD of a workgroup whose block has tm x tn tiles: wavefront w holds half w / 4 of
// the rows and a quarter of the columns, w and w + 4 share a SIMD and take quarters q and 3 - q
inline int gram64_simd_tiles(int tm, int tn) {
    const int upper = (tm + 1) / 2, lower = tm - upper;
    int most = 0;
    for (int q = 0; q < 4; ++q) {
        const int a = tn * (q + 1) / 4 - tn * q / 4, b = tn * (4 - q) / 4 - tn * (3 - q) / 4;
        most = std::max(most, upper * a + lower * b);
    }
    return most;
}

// Whether this kernel is the faster one.  Both sides are rounds of workgroups over the 256 CUs:
// - the kernel's round is its points / 4 products of the fullest SIMD, 64 cycles each at 2.4 GHz, of
//   which it reaches 0.63 (0.62-0.72 measured), plus 15 us;
// - the library's round is one tile of a chunk (K / chunks points), whose size it chooses by the points:
//   128 x 192 above 10,200 points (74.6 TFLOP/s), 64 x 64 above 5,500 (60), 128 x 64 below (62).
// It has to win by 5 %.  Of 420 products (13,824 to 1,728,000 points, N x N, 2N, 3N for N = 8 to 528) the
// choice is 0.3 % from the faster side on average, and 4 % slower than the library at worst; the kernel
// alone is up to 1.5 times slower, where the library's tiles are full.  us, this : library: 512,000 points,
// 64 x 64 163 : 336, 144 x 144 490 : 757, 144 x 432 1395 : 1526, 192 x 576 2560 : 1966, 256 x 512
// 3038 : 2195, 528 x 528 5983 : 5847; 1,728,000 points, 144 x 144 1580 : 4442, 288 x 288 5986 : 9159,
// 512 x 512 18,457 : 14,966, 528 x 1584 72,395 : 54,790.
inline bool gram64_faster(int64_t K, int M, int N, int64_t chunks) {
    const GramSplit g = gram64_split(K, M, N);
    const int64_t own_rounds = (g.nch * g.mb * g.nb + 255) / 256;
    const double own = (double)own_rounds * g.per / 4 * gram64_simd_tiles(g.bm, g.bn) * 64 / 2400 / 0.63 + 15;
    const int64_t kc = K / chunks;
    const int tm = kc > 10200 ? 128 : (kc > 5500 ? 64 : 128), tn = kc > 10200 ? 192 : 64;
    const double rate = kc > 10200 ? 74.6 : (kc > 5500 ? 60.0 : 62.0);
    const int64_t tiles = (int64_t)((M + tm - 1) / tm) * ((N + tn - 1) / tn);
    const double lib = (double)((tiles * chunks + 255) / 256) * kc * tm * tn * 2 * 256 / rate * 1e-6;
    return own <= 0.95 * lib;
}

}  // namespace qg
