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

// The fp32 tiles of a library product; `aligned`: rows and operands begin at multiples of 16 bytes.  (A slice of 32 k is guarded like
// any other.  256 x 256 and 192 x 192 come whole only: where K or the alignment asks for guards, 64 x 64 take their place.)
struct fp32_tiles { int m, n; bool guarded; };
inline fp32_tiles library_tiles_for(long M, long N, long K, long problems, bool aligned) {
    const int edge = square_tile_for(M, N);
    const bool guarded = !(aligned && M % edge == 0 && N % edge == 0 && K % (edge == 64 ? 32 : 16) == 0);
    if (edge == 64 || M < 32 || N < 32) {
        const small_tile t = small_tile_for(M, N, K, problems, !guarded);
        const int m = t == TILE_64x32 ? 64 : 32;
        if (t != TILE_64) return {m, 32, !(aligned && M % m == 0 && N % 32 == 0 && K % small_tile_slice(K) == 0)};
    }
    if (guarded && edge > 128) return {64, 64, true};
    return {edge, edge, guarded};
}

// C tiles of the kernels that split fp32 operands into bf16 parts (gemm_mfma_split.hip.h), and when they replace the fp32 instruction.
// Whole launches of both kinds are modelled like the tiles above: `fixed` microseconds and `first` per k for a round of tiles over the
// compute units, `round` and `further` per k for each round after it; fitted at 64 ... 4096 k, up to sixteen rounds, uniform
// random operands (rms error 3 to 8 %).  us measured with the fp32 instruction / split: 4096^3 946 / 607 (256 x 256),
// 2048^3 136 / 97 (128 x 128), 4096 x 4096 x 128 43 / 33, 2048 x 2048 x 256 23.1 / 20.3, 1024^3 21.5 / 19.0 (64 x 64), guarded 3623 x 2943 x 920
// 193 / 130, 1218 x 2748 x 611 50 / 37; and where the fp32 instruction stays: 1024 x 1024 x 256 8.2 / 8.8, 2048 x 2048 x 128
// 14.8 / 14.9, 1520 x 3116 x 503 51 / 54.
// Tiles of 256 and 192 that are guarded, which divide M and N but not K (programs, which also read C; fp32 / split): 4096 x 4096 x 1000
// 257 / 179, x 250 90 / 73, 3072 x 6144 x 1000 294 / 264; left: 3072 x 3072 x 250 51 / 55, x 2030 283 / 291, 3072 x 6144 x 250 97 / 114.
// Library calls, whose fp32 tiles are then 64 x 64: 4096 x 4096 x 1000 316 / 180, x 4095 1115 / 620, 3072 x 3072 x 3000 469 / 386, x 100 31 / 28.
struct launch_model { int m, n; bool guarded; double fixed, round, first, further; };
constexpr launch_model FP32_LAUNCHES[] = {
    {256, 256, false, 11.0, 2.0, 0.2242, 0.23}, {192, 192, false, 9.2, 2.6, 0.1322, 0.132}, {128, 128, false, 4.9, 3.2, 0.0617, 0.0587},
    {64, 64, false, 3.1, 0.7, 0.0175, 0.0157}, {64, 32, false, 3.3, 0.8, 0.0093, 0.0080}, {32, 32, false, 3.0, 0.5, 0.0061, 0.0043},
    {128, 128, true, 6.7, 4.8, 0.0669, 0.0601}, {64, 64, true, 4.1, 1.1, 0.0206, 0.0165}, {64, 32, true, 4.4, 1.5, 0.0104, 0.0091},
    {32, 32, true, 4.2, 0.8, 0.0073, 0.0048},
    {256, 256, true, 17.0, 17.0, 0.2275, 0.231}, {192, 192, true, 7.8, 2.0, 0.130, 0.1323}};       // (generated code only: library_tiles_for)
constexpr launch_model SPLIT_LAUNCHES[] = {
    {256, 256, false, 10.1, 2.3, 0.135, 0.145}, {128, 128, false, 7.9, 5.8, 0.0380, 0.0404}, {64, 64, false, 5.3, 3.5, 0.0132, 0.0121},
    {256, 256, true, 12.1, 2.3, 0.130, 0.145}, {128, 128, true, 9.2, 8.7, 0.0360, 0.0405}};
inline double modelled(const launch_model &l, long M, long N, long K, long problems) {
    const long tiles = ((M + l.m - 1) / l.m) * ((N + l.n - 1) / l.n) * problems;
    const double more = (double)((tiles + COMPUTE_UNITS - 1) / COMPUTE_UNITS - 1);
    return l.fixed + more * l.round + K * (l.first + more * l.further);
}
// k of a slice; LDS of a workgroup (two stages of three planes, or of eight wavefronts' own slices)
constexpr int split_slice(int edge) { return edge == 128 ? 32 : 16; }
constexpr int split_operand_words(int edge, bool kmajor) {
    return edge == 64 ? 64 * 16 + (kmajor ? 0 : 64) : 3 * (split_slice(edge) / 8) * 4 * (kmajor ? edge + 128 / split_slice(edge) : edge + 16);
}
constexpr int split_lds_bytes(int edge, bool a_kmajor, bool b_kmajor) {
    return 2 * 4 * (edge == 64 ? 8 : 1) * (split_operand_words(edge, a_kmajor) + split_operand_words(edge, b_kmajor));
}
// leading dimensions: four elements of a row at least, offsets within a tile in 32 bits
constexpr long SPLIT_LD_LIMIT = 1L << 22;
constexpr bool split_whole(int edge, long M, long N, long K) { return M % edge == 0 && N % edge == 0 && K % split_slice(edge) == 0; }
// ... of a workgroup of the windowed convolution on split operands (gemm_mfma_window_split.hip.h): three planes of 16-byte granules
constexpr long window_split_lds_bytes(long rows, long taps, long window) { return 3 * 16 * (rows * (taps | 1) + 1 + window); }
// The edge of the split tile that takes an M x N x K product from fp32 tiles of m x n (guarded or not), 0: none.  Where the fp32
// tiles are 32 wide, four groups of wavefronts add four partial sums: only the eight of the 64 x 64 tile are at least as close
// to 64 bits.  Below 96 k the two are equally close, and little is gained.  Tiles without a row above (64 x 256: a result of at most
// 64 rows, very wide) keep the fp32 instruction.
inline int split_tile_for(long M, long N, long K, long problems, int m, int n, bool guarded) {
    if (M < 64 || N < 64 || K < 96) return 0;
    double best = 0;
    for (const launch_model &l : FP32_LAUNCHES)
        if (l.m == m && l.n == n && l.guarded == guarded) best = 0.95 * modelled(l, M, N, K, problems);
    int edge = 0;
    for (const launch_model &l : SPLIT_LAUNCHES) {
        if (l.guarded == split_whole(l.m, M, N, K) || (n == 32 && l.m != 64)) continue;
        const double cost = modelled(l, M, N, K, problems);
        if (cost < best) { best = cost; edge = l.m; }
    }
    return edge;
}

// C tiles of a product with a gathered operand and at most 64 rows (an implicit GEMM: a convolution whose window is not staged in LDS; fp32
// instruction).  With few columns a launch is bound by the chain of a tile's slices, so four groups of wavefronts share slices of 64 k; with
// 32 rows or fewer a tile of 64 is half padding.  Modelled as whole launches: `fixed` microseconds, `round` for every round of tiles over the
// compute units, and per k `first` or rounds times `further`, whichever is more; fitted to 44 convolutions of 3 ... 64 channels, 5 ... 64 filters
// and 64 ... 300000 positions (rms error 9 to 14 %).  us of a launch with the tile of before (64 x 256 from 65536 columns on, else 64 x 64)
// and with the one chosen: 2 images of 40 x 40, 64 to 48 channels 14.0, 6.5 (32 x 32); 3 of 24 x 24, 41 to 6 9.0, 4.7; 1 of 96 x 96, 44 to 15 10.7, 6.9 (32 x 64);
// 32 of 100 x 100, 16 to 16 59, 35 (32 x 128); 7 of 96 x 96, 24 to 16 20.5, 12.2; 8 of 92 x 92, 40 to 50 53, 38 (64 x 64); 29 of 56 x 56, 46 to
// 35 59, 46 (64 x 128); 8 of 112 x 112, 3 to 64 13.3, 13.0; of the 44 none slower, 0.71 of the time in the geometric mean.
struct gathered_tile { int m, n, k, waves_m, waves_n, groups; double fixed, round, first, further; };
constexpr gathered_tile GATHERED_TILES[] = {
    {32, 32, 64, 1, 1, 4, 2.5, 0.66, 0.0056, 0.0047}, {32, 64, 64, 1, 2, 4, 1.8, 1.7, 0.0092, 0.0085}, {32, 128, 16, 1, 4, 1, 1.0, 1.7, 0.027, 0.0174},
    {64, 64, 32, 2, 2, 1, 2.15, 0.96, 0.0178, 0.0177}, {64, 128, 16, 2, 2, 1, 1.9, 1.4, 0.0395, 0.0313}};
// (whole 64 x 64 tiles whose slices of 64 k two groups share, a round of them)
constexpr double GATHERED_TWO_GROUPS_FIXED = 1.6, GATHERED_TWO_GROUPS_PER_K = 0.0185;
inline double modelled(const gathered_tile &c, long M, long N, long K) {
    const long tiles = ((M + c.m - 1) / c.m) * ((N + c.n - 1) / c.n);
    const double rounds = (double)((tiles + COMPUTE_UNITS - 1) / COMPUTE_UNITS), slope = rounds * c.further > c.first ? rounds * c.further : c.first;
    return c.fixed + rounds * c.round + (double)K * slope;
}
inline gathered_tile gathered_tile_for(long M, long N, long K) {
    const gathered_tile *best = nullptr;
    double best_cost = 0;
    for (const gathered_tile &c : GATHERED_TILES) {
        const double cost = modelled(c, M, N, K);
        if (!best || cost < best_cost) { best = &c; best_cost = cost; }
    }
    return *best;
}

// C tiles of the bf16-input kernels.  What the loops over K of a launch take is modelled as `fixed` microseconds (start, first
// slices) plus, for every 32 k of whole stages, `first` for the first round of tiles over the compute units and `further` for
// each round after it.  Reading and writing C is left out: it takes every tile about the same (1.07 us per million elements),
// so the model only orders the tiles.  It is fitted to whole launches of 100 sizes of 32 ... 4096 rows, columns and k (rms error
// 8 to 12 %).  A stage of the LDS ring holds `slices` slices of `k`: with 64 k a row of A is read 128 bytes at a time, a whole line
// of the L1, and there is one barrier for twice the work (4096^3 122.5 -> 119.0 us, 2000 x 1500 x 1000 16.2 -> 15.0 a call); slices of 32 in
// more stages start earlier and pad less.
// The tiles between the squares of 256, 128 and 64 are for results that those cover badly: 1500 x 1000 x 3000 are 96 tiles of 128 x 128
// (34 us) or 384 of 64 x 64, two rounds (28), but 192 of 64 x 128 (22); 1798 x 3830 x 3428 88 us with 128 x 128, 56 with 128 x 256;
// 1908 x 2550 x 858 27 and 20 with 192 x 128; 682 x 3212 x 1114 19 and 14.4 with 96 x 128; 417 x 396 x 3318 20 with 64 x 64 and 15 with 32 x 64.
// A tile is taken from `from` to `to` k.  Up to 512 k the squares keep the figures they were fitted with there: the tiles between them
// would give less than a microsecond, and the model errs by as much (805 x 1240 x 306 6.5 us with 64 x 64, 6.7 with 64 x 128).
// Where the rows of both operands lie at multiples of 16 bytes, two workgroups with 128 x 128 tiles to a compute unit cover each other better
// (`further_aligned`: 2328 x 3776 x 644 36.6 us, 3224 x 2688 x 592, as much work, 26.8); there they are ahead of several rounds of 192 x 128:
// 4096 x 2560 x 640 26.1 and 28.5, 4035 x 2816 x 688 31.6 and 32.8, 3456 x 3264 x 600 30.9 and 31.1; not where their last round is a quarter of the
// chip or less, which nothing covers: 2946 x 2752 x 584 27.0 and 26.1, 3000 x 3000 x 800 32.1 and 31.6.
// Tiles of 256 x 256 load their slices in pairs where the launch asks most of the L1: one tile for every compute unit, or 180 of them and rows of A
// that lie at whole lines (4096^3 122.5 -> 119.0 us, 4000 x 4000 x 1300 56.3 -> 55.3, 3840 x 3072 x 4096 99.1 -> 97.1).  With fewer two stages cover the way to
// memory worse than four: 3000 x 2700 x 4000 82.8 us one by one and 88.6 in pairs, 2560 x 3520 x 1368 40.1 and 42.7, 3383 x 3956 x 2808 87.4 and 88.5, in several rounds
// 7000 x 6000 x 3000 261 and 266.
// Direct tiles load their slices straight into LDS; the others serve rows of an odd number of elements and other operands that
// those loads cannot address.
struct bf16_tile {
    int m, n, k, slices, waves_m, waves_n, stages;
    bool direct;
    int from, to;
    double fixed, first, further, further_aligned;
};
constexpr int ANY_K = 0x7fffffff;
constexpr bf16_tile BF16_TILES[] = {
    {256, 256, 32, 1, 4, 2, 4, true, 0, ANY_K, 9.0, 0.55, 0.85, 0.85}, {128, 128, 32, 1, 2, 4, 4, true, 0, 512, 3.9, 0.17, 0.28, 0.28},
    {64, 64, 64, 1, 2, 2, 3, true, 0, 512, 2.8, 0.12, 0.12, 0.12}, {32, 64, 64, 1, 1, 2, 3, true, 192, 512, 2.7, 0.104, 0.092, 0.092},
    {128, 256, 64, 1, 2, 4, 3, true, 513, ANY_K, 6.2, 0.326, 0.51, 0.51}, {192, 128, 64, 1, 2, 4, 3, true, 513, ANY_K, 5.6, 0.283, 0.386, 0.386},
    {128, 128, 32, 1, 2, 4, 4, true, 513, ANY_K, 3.9, 0.251, 0.295, 0.24}, {128, 128, 32, 2, 2, 4, 3, true, 513, ANY_K, 4.4, 0.227, 0.349, 0.349},
    {96, 128, 64, 1, 1, 4, 3, true, 513, ANY_K, 5.8, 0.188, 0.285, 0.285}, {64, 128, 64, 1, 2, 2, 3, true, 513, ANY_K, 4.1, 0.167, 0.179, 0.179},
    {64, 64, 64, 1, 2, 2, 3, true, 513, ANY_K, 3.35, 0.132, 0.117, 0.117}, {32, 64, 64, 1, 1, 2, 3, true, 513, ANY_K, 3.2, 0.114, 0.090, 0.090},
    {128, 128, 64, 1, 2, 2, 2, false, 0, ANY_K, 8.0, 0.42, 0.4, 0.4}, {64, 64, 64, 1, 2, 2, 2, false, 0, ANY_K, 3.5, 0.19, 0.195, 0.195}};
constexpr bf16_tile BF16_TILE_ANY_SIZE = BF16_TILES[sizeof(BF16_TILES) / sizeof(BF16_TILES[0]) - 1];    // sizes known at run time only

// `lda`, `ldb`: elements from one row of A, of B to the next, or what they are multiples of
inline bf16_tile bf16_tile_for(long M, long N, long K, bool direct, long lda, long ldb) {
    const bf16_tile *best = nullptr;
    double best_cost = 0;
    const bool aligned = lda % 8 == 0 && ldb % 8 == 0;
    for (const bf16_tile &c : BF16_TILES) {
        if (c.direct != direct || K < c.from || K > c.to) continue;
        const long tiles = ((M + c.m - 1) / c.m) * ((N + c.n - 1) / c.n), rounds = (tiles + COMPUTE_UNITS - 1) / COMPUTE_UNITS, stage = c.k * c.slices;
        const bool covered = aligned && tiles - (rounds - 1) * COMPUTE_UNITS > COMPUTE_UNITS / 4;
        const double cost = c.fixed + ((K + stage - 1) / stage * stage / 32) * (c.first + (rounds - 1) * (covered ? c.further_aligned : c.further));
        if (!best || cost < best_cost) { best = &c; best_cost = cost; }
    }
    bf16_tile tile = *best;
    const long tiles = ((M + tile.m - 1) / tile.m) * ((N + tile.n - 1) / tile.n);
    if (tile.m == 256 && K > 512 && (tiles == COMPUTE_UNITS || (tiles >= 180 && lda % 64 == 0))) { tile.slices = 2; tile.stages = 2; }
    return tile;
}

}  // namespace ttarget
#endif
