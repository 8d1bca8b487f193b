// fp64 GEMM on the matrix cores of gfx950 (v_mfma_f64_16x16x4_f64): C = alpha * op(A) * op(B) + beta * C with
// every operand addressed through two strides, so that one kernel serves all four transposition cases of the
// library call, leading dimensions and offsets included.
//
// A workgroup of WGM x WGN wavefronts computes a tile of (16 TM WGM) x (16 TN WGN) elements, TM x TN instruction
// tiles of 16 x 16 per wavefront.  K is walked in slices of BK: the slice's A and B parts go from
// global memory to registers (8-byte loads, the thread-to-element mapping chosen so that consecutive lanes follow
// the operand's unit stride), from there to one of two LDS stages as [k][m] and [k][n], and each k-step (4) of a slice reads
// TM + TN operand fragments for TM * TN matrix instructions.  The next slice's global loads are issued before the
// current slice is multiplied and stored to the other stage after it: one barrier per slice.
//
// What bounds it: with tiles enough, the fp64 matrix instruction (64 cycles each, so LDS is never short); with few, the chain of
// one tile's slices, each a trip to memory, two LDS accesses and a barrier.  Hence tiles from 128 x 128 down to 16 x 16, and, in
// tiles that cannot fill the chip, groups of wavefronts that share a slice's k (WGK).  us before and after (before: 128 x 128,
// 64 x 64 or 32 x 32 by the number of tiles, slices of 16, every element guarded in all slices and in the epilogue):
//   1500 x 1430 x 250 62 -> 33, 2000 x 1100 x 700 112 -> 78, 1000^3 62 -> 48, 500^3 15.6 -> 11.6, 64 x 2048 x 512 14.8 -> 8.2,
//   180^3 7.6 -> 5.2, 16 x 16 x 2000 47 -> 14.3; 2048^3 314 (55 TFLOP/s) either way.
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
template <int TM_, int TN_, int WGM_, int WGN_, int BK_, int WGK_ = 1, int PAD = 2>
struct shape {
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
// `further` for each of several, whichever is more.  Fits to whole launches of 16 ... 2048 in each size (measured / modelled:
// 1500 x 1430 x 250 32.5 / 34.1 with 32 x 32, 34.3 / 34.7 with 96 x 96, 46 / 47 with 128 x 128; x 1000 114 / 120, 107 / 108,
// 155 / 155; 2080 x 4832 x 32 25 / 29, 30 / 29, 27 / 29; 1000^3 48 / 46 with 64 x 64, 55 / 55 with 32 x 32; 700 x 900 x 1000 45.5 / 42.1 without and 42.4 / 41.9 with
// shared slices; 200 x 300 x 1000 9.7 / 8.6 with 16 x 16, 18.6 / 18 with 32 x 32).
enum tile { TILE_128, TILE_96, TILE_64, TILE_32, TILE_32_SHARED, TILE_16, TILES };
typedef shape<4, 2, 2, 4, 16> shape_128;             // 2 x 4 wavefronts: two per SIMD cover each other's waits
typedef shape<3, 3, 2, 2, 16> shape_96;
typedef shape<2, 2, 2, 2, 64, 4> shape_64;
typedef shape<1, 1, 2, 2, 16> shape_32;              // eight workgroups to a compute unit: short reductions, many tiles
typedef shape<1, 1, 2, 2, 64, 4> shape_32_shared;
typedef shape<1, 1, 1, 1, 128, 8> shape_16;
// For at most 32 k, which two groups hold sixteen each of, as in the slices above (the sums are the same ones): the other groups'
// wavefronts only cost their start.  us of a call with 32 x 32 tiles without shared slices, with all groups, with two:
// 384 x 512 x 32 3.9, 4.2, 3.9; 345 x 533 x 11 3.8, 4.3, 4.0; 1184 x 160 x 32 3.8, 4.3, 3.9.
typedef shape<1, 1, 2, 2, 32, 2> shape_32_short;
typedef shape<1, 1, 1, 1, 32, 2> shape_16_short;

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

    const int slices = (K + BK - 1) / BK;
    if (slices > 0) {
        load_slice(0);
        store_slice(0);
    }
    __syncthreads();
    for (int s = 0; s < slices; s++) {
        const int stage = s & 1;
        if (s + 1 < slices) load_slice((s + 1) * BK);
        const double *la = lds64 + stage * S::STAGE + wm * (16 * TM) + l16;
        const double *lb = lds64 + stage * S::STAGE + BK * S::A_ROW + wn * (16 * TN) + l16;
#pragma unroll
        for (int ks = 0; ks < BK / 4 / S::WGK; ks++) {
            double fa[TM], fb[TN];
            const int k = 4 * (wk * (BK / 4 / S::WGK) + ks) + kq;
#pragma unroll
            for (int i = 0; i < TM; i++) fa[i] = la[k * S::A_ROW + 16 * i];
#pragma unroll
            for (int j = 0; j < TN; j++) fb[j] = lb[k * S::B_ROW + 16 * j];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (s + 1 < slices) store_slice(stage ^ 1);
        __syncthreads();
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
