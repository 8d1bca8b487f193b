// The machine that the emitters and kernels of this back-end are shaped for: one MI355X (gfx950).
// Plain constants and the tile model, usable from host C++ (the recognisers, the runtime's dispatch)
// and from device code alike; nothing else in the tree spells these numbers.
#ifndef TIRAMISU_AMD_TARGET_GFX950_H
#define TIRAMISU_AMD_TARGET_GFX950_H

namespace ttarget {

constexpr int COMPUTE_UNITS = 256;        // 8 XCDs x 32
constexpr int XCDS = 8;                   // each with its own L2; workgroup ids are dealt to them round-robin
constexpr int WAVEFRONT = 64;
constexpr int LDS_BYTES_PER_CU = 160 * 1024;
constexpr int MAX_THREADS_PER_WORKGROUP = 1024;

// Square C tiles of the fp32 MFMA kernel and the share of the matrix-core rate that a tile of each size
// sustains (larger tiles re-read less through LDS); 256 and 192 are used for whole tiles only.
struct square_tile { int edge; double rate; bool whole_only; };
constexpr square_tile SQUARE_TILES[] = {{256, 1.0, true}, {192, 0.9, true}, {128, 0.8, false}, {64, 0.68, false}};

// The square tile whose launch is modelled fastest for an M x N result: a compute unit works through
// ceil(tiles / COMPUTE_UNITS) tiles, each costing its area over its rate.
inline int square_tile_for(long M, long N) {
    double best = 0;
    int edge = 64;
    for (const square_tile &c : SQUARE_TILES) {
        if (c.whole_only && (M % c.edge != 0 || N % c.edge != 0)) continue;
        if (c.edge == 128 && M < 128) continue;
        const long tiles = ((M + c.edge - 1) / c.edge) * ((N + c.edge - 1) / c.edge);
        const double cost = (double)((tiles + COMPUTE_UNITS - 1) / COMPUTE_UNITS) * c.edge * c.edge / c.rate;
        if (best == 0 || cost < best) { best = cost; edge = c.edge; }
    }
    return edge;
}

// Where 64 x 64 is the square tile chosen and its tiles are few, smaller ones whose four groups of wavefronts share a slice's k: the
// launch is bound by the chain of a tile's slices, not by the matrix cores.  Modelled like the fp64 tiles: `fixed` microseconds and,
// per k, `first` for a round of tiles over the compute units, `further` for each of several, whichever is more; 64 x 64 is faster
// per k where no tile hangs over the operands.  Fits to whole launches at sizes that no tile divides (measured / modelled, us):
// 700 x 900 x 1000 26.3 / 26.5 with 64 x 64, 26.4 / 25.8 with 64 x 32, 23.2 / 22.5 with 32 x 32; 1100 x 1300 x 2000 82 / 80, 69 / 71,
// 76 / 81; 2001 x 1501 x 1001 60 / 61, 67 / 71, 72 / 81; 400 x 400 x 500 14.5 / 14.8, 9.7 / 9.3, 8.1 / 7.5.
enum small_tile { TILE_64, TILE_64x32, TILE_32 };
inline small_tile small_tile_for(long M, long N, long K, long problems, bool whole) {
    if (M < 32 || N < 32) return TILE_32;
    static const struct { int m, n; double fixed, first, further; } model[3] = {
        {64, 64, 3.0, 0.0235, 0.0193}, {64, 32, 3.2, 0.0122, 0.0113}, {32, 32, 3.0, 0.009, 0.0065}};
    int best = 0;
    double best_cost = 0;
    for (int i = 0; i < 3; i++) {
        const long tiles = ((M + model[i].m - 1) / model[i].m) * ((N + model[i].n - 1) / model[i].n) * problems;
        const double rounds = (double)((tiles + ttarget::COMPUTE_UNITS - 1) / ttarget::COMPUTE_UNITS);
        const bool whole_64 = i == 0 && whole;
        const double first = whole_64 ? 0.0165 : model[i].first, further = rounds * (whole_64 ? 0.0155 : model[i].further);
        const double cost = model[i].fixed + K * (first > further ? first : further);
        if (i == 0 || cost < best_cost) { best = i; best_cost = cost; }
    }
    return (small_tile)best;
}

// The k of a slice of those smaller tiles: 64, dealt to four groups of wavefronts by sixteen k each; 32 and two groups where K
// holds no more, so that no half of a slice is padding.  The partial sums are the same ones.  us of a call before (with 64 x 64
// tiles), with slices of 64 and of 32: 384 x 3104 x 32 6.1, 8.5, 6.0; 480 x 5216 x 32 8.3, 12.1, 8.3; 1696 x 3168 x 20 13.7, 24.6,
// 14.4; with one row 1 x 142339 x 20 17.8 (one thread per element), 18.2, 10.2.
inline int small_tile_slice(long K) { return K <= 32 ? 32 : 64; }

// C tiles of the bf16-input kernels.  What the loops over K of a launch take is modelled as `fixed` microseconds (start, first
// slices) plus, for every 32 k of whole slices, `first` for the first round of tiles over the compute units and `further` for
// each round after it.  Reading and writing C is left out: it takes every tile the same (64 MiB in and out at 4096 x 4096 20 us),
// so the model only orders the tiles.  It is fitted to whole launches of 32 ... 4096 k with a tenth of the chip's tiles up to
// sixteen rounds: 300 x 260 x 3000 takes 13.0 us with 64 x 64 (14.1 modelled) and 21.6 with 128 x 128 (19.9), 1000 x 750 x 500
// 5.6 and 8.0 (4.7, 6.6), 2000 x 1500 x 1000 15.6 with 128 x 128 and 18.0 with 64 x 64 (9.3, 14.3), 3000 x 2700 x 4000 82 with
// 256 x 256 and 109 with 128 x 128 (78, 95), 4096 x 3072 x 32, half of a slice of the 64 x 64 tiles, 17.3 with 128 x 128 and
// 20.5 with 64 x 64 (4.6, 5.7).
// Direct tiles load their slices straight into LDS; the others serve rows of an odd number of elements and other operands that
// those loads cannot address.
struct bf16_tile {
    int edge, k, waves_m, waves_n, stages;
    bool direct;
    double fixed, first, further;
};
constexpr bf16_tile BF16_TILES[] = {{256, 32, 4, 2, 4, true, 9.0, 0.55, 0.85}, {128, 32, 2, 4, 4, true, 3.9, 0.17, 0.28},
                                    {64, 64, 2, 2, 3, true, 2.8, 0.12, 0.12},
                                    {128, 64, 2, 2, 2, false, 8.0, 0.42, 0.4}, {64, 64, 2, 2, 2, false, 3.5, 0.19, 0.195}};
constexpr bf16_tile BF16_TILE_ANY_SIZE = BF16_TILES[4];    // sizes known at run time only

inline bf16_tile bf16_tile_for(long M, long N, long K, bool direct) {
    const bf16_tile *best = nullptr;
    double best_cost = 0;
    for (const bf16_tile &c : BF16_TILES) {
        if (c.direct != direct) continue;
        const long tiles = ((M + c.edge - 1) / c.edge) * ((N + c.edge - 1) / c.edge), rounds = (tiles + COMPUTE_UNITS - 1) / COMPUTE_UNITS;
        const double cost = c.fixed + ((K + c.k - 1) / c.k * c.k / 32) * (c.first + (rounds - 1) * c.further);
        if (!best || cost < best_cost) { best = &c; best_cost = cost; }
    }
    return *best;
}

}  // namespace ttarget
#endif
