// fp64 GEMM on the matrix cores of gfx950 (v_mfma_f64_16x16x4_f64): C = alpha * op(A) * op(B) + beta * C with
// every operand addressed through two strides, so that one kernel serves all four transposition cases of the
// library call, leading dimensions and offsets included.
//
// A workgroup of WGM x WGN wavefronts computes a tile of (16 TM WGM) x (16 TN WGN) elements, TM x TN instruction
// tiles of 16 x 16 per wavefront.  K is walked in slices of BK: the slice's A and B parts go from
// global memory to registers (8-byte loads, the thread-to-element mapping chosen so that consecutive lanes follow
// the operand's unit stride), from there to one of two LDS stages as [k][m] and [k][n], and each k-step (4) of a slice reads
// TM + TN operand fragments for TM * TN matrix instructions.  In all but the tiles of 128, of 96 with slices of their own and of 16 (AHEAD) a slice is
// stored to its stage while the one before it is multiplied, one slice after its loads were issued, and a step's fragments are read during the step
// before: one barrier per slice, ahead of its last step.
//
// What bounds it: with tiles enough, the fp64 matrix instruction (64 cycles each, so LDS is never short); with few, the chain of
// one tile's slices, each a trip to memory, two LDS accesses and a barrier.  Hence tiles from 128 x 128 down to 16 x 16, and groups
// of wavefronts that share a slice's k (WGK).  us of a library call among others (nothing transposed, C not read) with loads one slice ahead, fragments
// read by the step that multiplies them and fewer such groups -> now: 1500 x 1430 x 250 31.1 -> 28.5, 2000 x 1100 x 700 75 -> 65, 1500 x 1430 x 1000
// 106 -> 91, 1000^3 47.3 -> 44.2, 500^3 10.7 -> 10.0, 2048^3 314 -> 312 (55 TFLOP/s), 200 x 300 x 1000 8.9 either way.
//
// Instruction layout (one wavefront): lane l supplies A[row l % 16][k l / 16] and B[k l / 16][column l % 16];
// its four results are rows l / 16 + 0, 4, 8, 12 of column l % 16.
#ifndef TIRAMISU_AMD_GEMM_MFMA_F64_HIP_H
#define TIRAMISU_AMD_GEMM_MFMA_F64_HIP_H
#include <hip/hip_runtime.h>

#include "gemm_mfma.hip.h"

namespace tgemm64 {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// BK: the k of a slice.  PAD of 2 doubles: rows lie 4 words apart modulo the 64 banks, so the 16 k that the consecutive lanes of
// a k-contiguous operand store fall on different banks.
// WGK groups of wavefronts each multiply 1 / WGK of a slice's k for the same tile; their sums are added through LDS.
// AHEAD: the pipeline below; without it a slice is loaded and stored around the one that is multiplied, in the registers that two workgroups
// of the largest tiles have to a compute unit (2048^3 with 128 x 128 tiles 314 us; with the pipeline, which spills there, 349 to 513 by layout).
template <int TM_, int TN_, int WGM_, int WGN_, int BK_, int WGK_ = 1, bool AHEAD_ = true, int PAD = 2>
struct shape {
    static constexpr bool AHEAD = AHEAD_;
    static constexpr int TM = TM_, TN = TN_, WGM = WGM_, WGN = WGN_, BK = BK_, WGK = WGK_;
    static constexpr int NT = 64 * WGM * WGN * WGK;
    static constexpr int RESIDENT = WGK == 1 ? 2 : 1;                        // workgroups that share a compute unit
    static constexpr int WAVES_PER_SIMD = NT * RESIDENT >= 256 ? NT * RESIDENT / 256 : 1;
    static constexpr int BM = 16 * TM * WGM, BN = 16 * TN * WGN;
    static constexpr int A_ROW = BM + PAD, B_ROW = BN + PAD;                 // doubles per k row of a stage
    static constexpr int STAGE = BK * (A_ROW + B_ROW);
    static constexpr int LDS_BYTES = 2 * STAGE * (int)sizeof(double);
    static constexpr int A_PER_THREAD = BM * BK / NT, B_PER_THREAD = BN * BK / NT;   // elements per thread and slice
    static_assert((BM * BK) % NT == 0 && (BN * BK) % NT == 0, "slice parts divide over the threads");
    static_assert(RESIDENT * LDS_BYTES <= ttarget::LDS_BYTES_PER_CU, "LDS of the workgroups that share a compute unit");
    static_assert((BK / 4) % WGK == 0, "the k steps of a slice divide over the groups");
    static_assert((WGK - 1) * WGM * WGN * TM * TN * 4 * 64 <= 2 * STAGE, "LDS too small for the groups' sums");
};

// The tiles, and the one whose launch is modelled fastest: `fixed` microseconds (start, the last store), `round` for every round of
// tiles over the compute units (first slice, epilogue), and per k `first` for a round that a compute unit has to itself or
// `further` for each of several, whichever is more.  Fits to whole launches of 16 ... 2048 in each size of the tiles without the pipeline (measured / modelled:
// 1500 x 1430 x 250 32.5 / 34.1 with 32 x 32, 34.3 / 34.7 with 96 x 96, 46 / 47 with 128 x 128; x 1000 114 / 120, 107 / 108,
// 155 / 155; 2080 x 4832 x 32 25 / 29, 30 / 29, 27 / 29; 1000^3 48 / 46 with 64 x 64, 55 / 55 with 32 x 32; 700 x 900 x 1000 45.5 / 42.1 without and 42.4 / 41.9 with
// shared slices; 200 x 300 x 1000 9.7 / 8.6 with 16 x 16, 18.6 / 18 with 32 x 32); the order stays as the pipeline found it, so that no size gets fewer
// partial sums: 64 x 64 without shared slices, faster where its tiles are several rounds (1960 x 1449 x 466 57 and 75), has twice their error.
// Tiles of 96 x 96 that fit the chip in a round leave each SIMD one wavefront: with slices of 32 k shared by two groups it has two. They take the place of
// tiles whose sums are of one part, not of those of four or eight, which are closer, where they are modelled faster than these are now (`present`, fitted to
// 140 sizes on both sides of the line, rms error 3 to 6 %).  us of a call with the tile they replace / with them: 1504 x 1485 x 1664 171 / 143,
// 2000 x 1100 x 700 75 / 65, 1600 x 1293 x 1216 125 / 106 (96 x 96), 1440 x 1431 x 736 74 / 67, 1500 x 1430 x 250 31.1 / 28.5 (32 x 32), error against 64 bits and
// more 0.75 of it; left: 1664 x 1337 x 140 19.4 / 20.8, 1943 x 1135 x 170 22.5 / 23.4 (32 x 32).
enum tile { TILE_128, TILE_96, TILE_64, TILE_32, TILE_32_SHARED, TILE_16, TILES, TILE_96_SHARED };
typedef shape<4, 2, 2, 4, 16, 1, false> shape_128;   // 2 x 4 wavefronts: two per SIMD cover each other's waits
typedef shape<3, 3, 2, 2, 16, 1, false> shape_96;
typedef shape<3, 3, 2, 2, 32, 2> shape_96_shared;
typedef shape<2, 2, 2, 2, 64, 4> shape_64;
typedef shape<1, 1, 2, 2, 16> shape_32;              // eight workgroups to a compute unit: short reductions, many tiles
typedef shape<1, 1, 2, 2, 64, 4> shape_32_shared;
typedef shape<1, 1, 1, 1, 128, 8, false> shape_16;      // (241 x 288 x 1344 16.5 us; with the pipeline 16.8)
// For at most 32 k, which two groups hold sixteen each of, as in the slices above (the sums are the same ones): the other groups'
// wavefronts only cost their start.  us of a call with 32 x 32 tiles without shared slices, with all groups, with two:
// 384 x 512 x 32 3.9, 4.2, 3.9; 345 x 533 x 11 3.8, 4.3, 4.0; 1184 x 160 x 32 3.8, 4.3, 3.9.
typedef shape<1, 1, 2, 2, 32, 2> shape_32_short;
typedef shape<1, 1, 1, 1, 32, 2, false> shape_16_short;

inline tile tile_for(long M, long N, long K) {
    static const struct { int edge; double fixed, round, first, further; } model[TILES] = {
        {128, 8.0, 2.5, 0.1445, 0.14}, {96, 9.0, 1.3, 0.0975, 0.084}, {64, 1.3, 5.0, 0.0395, 0.0395},
        {32, 3.3, 0.25, 0.0235, 0.0127}, {32, 2.6, 0.9, 0.0145, 0.0122}, {16, 2.2, 0.9, 0.0055, 0.0052}};
    int best = TILE_128;
    double best_cost = 0;
    for (int i = 0; i < TILES; i++) {
        const long e = model[i].edge, tiles = ((M + e - 1) / e) * ((N + e - 1) / e);
        const double rounds = (double)((tiles + ttarget::COMPUTE_UNITS - 1) / ttarget::COMPUTE_UNITS);
        const double slope = rounds * model[i].further > model[i].first ? rounds * model[i].further : model[i].first;
        const double cost = model[i].fixed + rounds * model[i].round + (double)K * slope;
        if (i == 0 || cost < best_cost) { best = i; best_cost = cost; }
    }
    if (((M + 95) / 96) * ((N + 95) / 96) > ttarget::COMPUTE_UNITS) return (tile)best;
    static const struct { tile which; double fixed, round, first, further; } present[] = {
        {TILE_128, 6.5, 2.7, 0.1467, 0.1467}, {TILE_96, 5.8, 2.0, 0.1002, 0.1002}, {TILE_32, 3.0, 0.1, 0.0235, 0.0118}};
    for (const auto &p : present) {
        const long e = model[best].edge, tiles = ((M + e - 1) / e) * ((N + e - 1) / e);
        const double rounds = (double)((tiles + ttarget::COMPUTE_UNITS - 1) / ttarget::COMPUTE_UNITS);
        if (p.which == best && 8.2 + 0.083 * (double)K < p.fixed + rounds * p.round + (double)K * (rounds * p.further > p.first ? rounds * p.further : p.first)) return TILE_96_SHARED;
    }
    return (tile)best;
}

// The second launch bound (wavefronts per SIMD) holds the kernel to the registers that let two workgroups share a
// compute unit: at 136 registers instead of 128 a single workgroup is resident and the kernel is a quarter slower.
// A_KFAST: consecutive k of A are adjacent in memory (stride_ak == 1), else consecutive m are; likewise B_NFAST.
template <class S, bool A_KFAST, bool B_NFAST>
__global__ void __launch_bounds__(S::NT, S::WAVES_PER_SIMD) dgemm_kernel(const double *__restrict__ A, const double *__restrict__ B, double *__restrict__ C, int M, int N,
                                                   int K, long stride_am, long stride_ak, long stride_bk, long stride_bn, long ldc, double alpha,
                                                   double beta) {
    constexpr int TM = S::TM, TN = S::TN, NT = S::NT, BK = S::BK;
    extern __shared__ __attribute__((aligned(16))) double lds64[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wk = wave / (S::WGM * S::WGN), wmn = wave % (S::WGM * S::WGN), wm = wmn / S::WGN, wn = wmn % S::WGN;
    const int l16 = lane & 15, kq = lane >> 4;
    // the workgroups of one XCD (ids congruent modulo 8) cover a compact group of C tiles: the panels of A and B
    // that they share are fetched once into that XCD's L2
    int tile_m, tile_n;
    tgemm::tile_of_block((M + S::BM - 1) / S::BM, (N + S::BN - 1) / S::BN, tile_m, tile_n);
    const int m0 = tile_m * S::BM, n0 = tile_n * S::BN;

    // Element (x, k) of the slice that load v of this thread brings: a tile that hangs over C reads its last row again (that only
    // reaches elements of C that nobody stores), so a slice that K holds whole is loaded without a guard or a select; in the
    // last one an element behind K is read at the last k and taken as zero.
    auto a_m = [&](int v) { const int u = t + NT * v; return A_KFAST ? u / BK : u % S::BM; };
    auto a_k = [&](int v) { const int u = t + NT * v; return A_KFAST ? u % BK : u / S::BM; };
    auto b_n = [&](int v) { const int u = t + NT * v; return B_NFAST ? u % S::BN : u / BK; };
    auto b_k = [&](int v) { const int u = t + NT * v; return B_NFAST ? u / S::BN : u % BK; };
    double ra[S::A_PER_THREAD], rb[S::B_PER_THREAD];
    const double *pa[S::A_PER_THREAD], *pb[S::B_PER_THREAD];
#pragma unroll
    for (int v = 0; v < S::A_PER_THREAD; v++) {
        const int m = m0 + a_m(v);
        pa[v] = A + (long)(m < M ? m : M - 1) * stride_am + (long)a_k(v) * stride_ak;
    }
#pragma unroll
    for (int v = 0; v < S::B_PER_THREAD; v++) {
        const int n = n0 + b_n(v);
        pb[v] = B + (long)(n < N ? n : N - 1) * stride_bn + (long)b_k(v) * stride_bk;
    }
    auto load_slice = [&](int k0) {
        if (k0 + BK <= K) {
#pragma unroll
            for (int v = 0; v < S::A_PER_THREAD; v++) { ra[v] = *pa[v]; pa[v] += BK * stride_ak; }
#pragma unroll
            for (int v = 0; v < S::B_PER_THREAD; v++) { rb[v] = *pb[v]; pb[v] += BK * stride_bk; }
        } else {
#pragma unroll
            for (int v = 0; v < S::A_PER_THREAD; v++) {
                const int behind = k0 + a_k(v) - (K - 1);
                const double a = *(pa[v] - (behind > 0 ? behind : 0) * stride_ak);
                ra[v] = behind > 0 ? 0.0 : a;
            }
#pragma unroll
            for (int v = 0; v < S::B_PER_THREAD; v++) {
                const int behind = k0 + b_k(v) - (K - 1);
                const double b = *(pb[v] - (behind > 0 ? behind : 0) * stride_bk);
                rb[v] = behind > 0 ? 0.0 : b;
            }
        }
    };
    auto store_slice = [&](int stage) {
        double *la = lds64 + stage * S::STAGE, *lb = la + BK * S::A_ROW;
#pragma unroll
        for (int v = 0; v < S::A_PER_THREAD; v++) la[a_k(v) * S::A_ROW + a_m(v)] = ra[v];
#pragma unroll
        for (int v = 0; v < S::B_PER_THREAD; v++) lb[b_k(v) * S::B_ROW + b_n(v)] = rb[v];
    };

    f64x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

    // One slice is multiplied while the next travels: the other stage is filled from registers during the first k-step and its
    // successor asked for; a k-step's operands are read from LDS during the step before it, the first of a slice behind the one barrier,
    // which lies before the last step, so that its matrix instructions cover the reads.
    constexpr int KS = BK / 4 / S::WGK;
    static_assert(KS % 2 == 0, "k-steps of a wavefront in pairs: the registers of a slice's first step are free in its last");
    double fa[2][TM], fb[2][TN];
    auto read = [&](int stage, int ks, int buf) {
        const double *la = lds64 + stage * S::STAGE + wm * (16 * TM) + l16;
        const double *lb = lds64 + stage * S::STAGE + BK * S::A_ROW + wn * (16 * TN) + l16;
        const int k = 4 * (wk * KS + ks) + kq;
#pragma unroll
        for (int i = 0; i < TM; i++) fa[buf][i] = la[k * S::A_ROW + 16 * i];
#pragma unroll
        for (int j = 0; j < TN; j++) fb[buf][j] = lb[k * S::B_ROW + 16 * j];
    };
    const int slices = (K + BK - 1) / BK;
    if (slices > 0) {
        load_slice(0);
        store_slice(0);
        if (S::AHEAD && slices > 1) load_slice(BK);
    }
    __syncthreads();
    if (S::AHEAD && slices > 0) read(0, 0, 0);
    for (int s = 0; s < slices; s++) {
        const int stage = s & 1;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int buf = ks & 1;
            if (!S::AHEAD) {
                if (ks == 0 && s + 1 < slices) load_slice((s + 1) * BK);
                read(stage, ks, buf);
            } else if (ks == 0 && s + 1 < slices) {
                store_slice(stage ^ 1);
                if (s + 2 < slices) load_slice((s + 2) * BK);
            }
            if (!S::AHEAD) {
            } else if (ks + 1 < KS) {
                read(stage, ks + 1, buf ^ 1);
            } else {
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
                if (s + 1 < slices) read(stage ^ 1, 0, buf ^ 1);
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[buf][i], fb[buf][j], acc[i][j], 0, 0, 0);
            // (one matrix instruction to a step: the step's reads stay ahead of it; 500^3 10.7 us without, 10.4 so)
            if constexpr (TM * TN == 1 && S::WGM * S::WGN > 1) __builtin_amdgcn_sched_barrier(0);
        }
        if (!S::AHEAD) {
            if (s + 1 < slices) store_slice(stage ^ 1);
            __syncthreads();
        }
    }

    if (S::WGK > 1) {
        // (the barrier behind the last slice, or before the first if there is none, lies behind every other use of LDS)
        auto slot = [&](int g, int i, int j, int r) -> double & {
            return lds64[((((g - 1) * S::WGM * S::WGN + wmn) * TM + i) * TN + j) * 256 + r * 64 + lane];
        };
#pragma unroll
        for (int g = 1; g < S::WGK; g++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (wk == g) slot(g, i, j, r) = acc[i][j][r];
        __syncthreads();
        if (wk > 0) return;
#pragma unroll
        for (int g = 1; g < S::WGK; g++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] += slot(g, i, j, r);
    }

    // epilogue: the values of rows of instruction tiles first, 16 elements of C per lane in flight together (read at its nearest
    // element where a tile hangs over it, so that no load waits behind a branch), then their stores
    constexpr int ROWS = TN * 4 >= 16 ? 1 : 16 / (TN * 4);
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += ROWS) {
        auto each = [&](auto element) {
#pragma unroll
            for (int i = i0; i < i0 + ROWS && i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        element(m0 + wm * (16 * TM) + 16 * i + 4 * r + kq, n0 + wn * (16 * TN) + 16 * j + l16, acc[i][j], r);
        };
        if (beta == 0.0)
            each([&](int, int, f64x4 &v, int r) { v[r] = alpha * v[r]; });
        else
            each([&](int row, int col, f64x4 &v, int r) {
                v[r] = alpha * v[r] + beta * C[(long)(row < M ? row : M - 1) * ldc + (col < N ? col : N - 1)];
            });
        each([&](int row, int col, f64x4 &v, int r) {
            if (row < M && col < N) C[(long)row * ldc + col] = v[r];
        });
    }
}

}  // namespace tgemm64
#endif
