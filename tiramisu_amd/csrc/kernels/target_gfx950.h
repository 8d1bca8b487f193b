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

// C tiles of the bf16-input kernels.  A launch is modelled to take `fixed` microseconds (start, first slices, epilogue) plus,
// for every 32 k, `first` for the first round of tiles over the compute units and `further` for each round after it.  The
// figures are fits to whole launches of 100 ... 4096 k with a tenth of the chip's tiles up to sixteen rounds (measured /
// modelled: 300 x 260 x 3000 12.8 / 14.2 us with 64 x 64, 1000 x 750 x 500 5.3 / 4.7, 2000 x 1500 x 1000 15.4 / 9.3 with
// 128 x 128 against 17.8 / 14.3 with 64 x 64, 3000 x 2700 x 4000 82 / 78 with 256 x 256 against 109 / 165 with 128 x 128).
// Direct tiles load their slices straight into LDS; the others serve rows of an odd number of elements.
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
        const double cost = c.fixed + ((K + 31) / 32) * (c.first + (rounds - 1) * c.further);
        if (!best || cost < best_cost) { best = &c; best_cost = cost; }
    }
    return *best;
}

}  // namespace ttarget
#endif
