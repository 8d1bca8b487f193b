// The implicit GEMM of a convolution (gemm_mfma_window.hip.h) on the bf16 matrix cores, every fp32 operand element as three bf16 parts
// (gemm_mfma_split.hip.h):
//     C[m, p] = sum over (c, t) of  A[m, c * TAPS + t] * X[ f(p) + c * chan_stride + tap_offset(t) ]
// A block of 8 channels is split once per tile on its way to LDS, in granules of 16 bytes that hold the 8 channels of one place in
// bf16: of one position of the window (X) or one row and tap (A).  A granule is a lane's whole operand of
// v_mfma_f32_32x32x16_bf16, whose sixteen k are the 8 channels of two taps, one for each half of the wavefront; shifting the window by
// a tap is an offset of whole granules.  An odd number of taps is followed by one of zeros.
//
// One stage in LDS (51 KB for 3 x 3 taps and 256 positions), the next block travels into registers while this one is multiplied; two
// workgroups of four wavefronts share a compute unit and cover each other's splitting, barriers and epilogues.  LDS accesses
// are free of bank conflicts: lanes store and read granules of neighbouring positions, and rows of A lie an odd number of
// granules apart.  (One workgroup of eight wavefronts with two stages, 512 positions and one barrier per block, the split dealt out
// between the matrix instructions: 229 us where this form took 181; it needs more registers than there are.)
//
// 32 images of 112 x 112, 64 to 64 channels: 250 us with the fp32 instruction, 172 so (median launches); matrix cores 58 % busy at the 1.8 GHz that
// the power limit leaves.  The error against 64 bits is smaller (gemm_mfma_split.hip.h), and sums that are not finite are
// computed again with the fp32 instruction (operands of 2^60, every sum: 454 us a call, 198 without, 276 with that instruction alone).
//
// Requirements (checked by the emitter): those of contraction_window, and whole blocks of 8 channels.  Work distribution, pieces of
// the last tiles and their hand-over are contraction_window's.
#ifndef TIRAMISU_AMD_GEMM_MFMA_WINDOW_SPLIT_HIP_H
#define TIRAMISU_AMD_GEMM_MFMA_WINDOW_SPLIT_HIP_H
#include "gemm_mfma_split.hip.h"

namespace tgemm {

template <int BM_, int BN_, int WGM_, int WGN_>
struct config_window {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, WGK = 1, NT = 64 * WGM * WGN;
    static constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    static constexpr bool EDGE = false;
};

// TAP_OFFSETS, POS, VALUE, STORE, scratch: as in contraction_window.  WIN: positions of a tile's window at most.
template <class CFG, int TAPS, int WIN, int SPLITS, class TAP_OFFSETS, class POS, class VALUE, class STORE>
__device__ __forceinline__ void contraction_window_split(const float *__restrict__ A, long lda, const float *__restrict__ X, long x_elements, const POS &pos,
                                                         long chan_stride, int channels, int M, int N, float *__restrict__ scratch, float *lds_, VALUE value,
                                                         STORE store) {
    constexpr int BM = CFG::BM, BN = CFG::BN, NT = CFG::NT, TM = CFG::TM, TN = CFG::TN;
    constexpr int CB = 8, STEPS = (TAPS + 1) / 2, ROW = TAPS | 1;                 // granules from one row of A to the next
    constexpr int A_GRANULES = BM * ROW + 1, X_GRANULES = WIN;                     // (one of zeros behind the rows)
    constexpr int A_UNITS = BM * TAPS, NVA = (A_UNITS + NT - 1) / NT, NVX = (WIN + NT - 1) / NT;
    static_assert(3 * 16 * (A_GRANULES + X_GRANULES) == ttarget::window_split_lds_bytes(BM, TAPS, WIN), "LDS of a workgroup");
    __shared__ unsigned ticket;
    __shared__ int next_item;
    uint32_t *const la = reinterpret_cast<uint32_t *>(lds_), *const lx = la + 3 * A_GRANULES * 4;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / CFG::WGN, wn = wave % CFG::WGN;
    const int l32 = lane & 31, h = lane >> 5;

    // ---- work items: whole tiles [0, whole), then pieces of the remaining tiles
    const int tiles_m = M / BM, tiles = tiles_m * (N / BN), G = gridDim.x, w = blockIdx.x;
    const int blocks = channels / CB;
    constexpr int splits = SPLITS;
    constexpr bool split = splits > 1;
    const int rest = split ? tiles % G : 0, whole = tiles - rest, items = whole + rest * splits;
    auto is_piece = [&](int q) { return q >= whole; };
    auto item_tile = [&](int q) { return is_piece(q) ? whole + (q - whole) / splits : q; };
    auto item_first = [&](int q) { return is_piece(q) ? (int)((long)((q - whole) % splits) * blocks / splits) : 0; };
    auto item_end = [&](int q) { return is_piece(q) ? (int)((long)((q - whole) % splits + 1) * blocks / splits) : blocks; };

    // ---- a tile: rows m0.., positions n0..; its window starts at f0
    struct place { int m0, n0; long f0; };
    auto place_of = [&](int tile) -> place {
        const int n0 = (tile / tiles_m) * BN;
        return {(tile % tiles_m) * BM, n0, (long)pos(n0)};
    };

    // ---- the block that travels: 8 channels of a position, or of a row and tap, per unit.  Addresses are a scalar part, channel by
    // channel, and a thread's own 32 bits.
    const split_constants sc;
    float rx[NVX][CB], ra[NVA][CB];
    auto load = [&](const place &p, int b) {
        const float *const from_a = A + (long)p.m0 * lda + (long)b * CB * TAPS;
#pragma unroll
        for (int c = 0; c < CB; c++) {
            const long first = p.f0 + ((long)b * CB + c) * chan_stride;
            const int behind = (int)min(x_elements - 1 - first, (long)WIN);       // the tail of a window may lie beyond the tensor: never used
#pragma unroll
            for (int v = 0; v < NVX; v++) {
                const int u = t + NT * v;
                if (WIN % NT != 0 && u >= WIN) break;
                rx[v][c] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(X + first) + 4u * (uint32_t)min(u, behind));
            }
        }
#pragma unroll
        for (int v = 0; v < NVA; v++) {
            const int u = t + NT * v;
            if (A_UNITS % NT != 0 && u >= A_UNITS) break;
            const uint32_t own = 4u * ((uint32_t)(u / TAPS) * (uint32_t)lda + (uint32_t)(u % TAPS));
#pragma unroll
            for (int c = 0; c < CB; c++) ra[v][c] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(from_a + c * TAPS) + own);
        }
    };
    auto put = [&](uint32_t *to, int plane, const float (&e)[CB]) {
        uint32_t word[3][4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            uint32_t part[3];
            split_pair(sc, e[2 * q], e[2 * q + 1], part);
#pragma unroll
            for (int s = 0; s < 3; s++) word[s][q] = part[s];
        }
#pragma unroll
        for (int s = 0; s < 3; s++) *reinterpret_cast<split_u4 *>(to + s * plane * 4) = split_u4{word[s][0], word[s][1], word[s][2], word[s][3]};
    };
    auto write = [&]() {
#pragma unroll
        for (int v = 0; v < NVX; v++) {
            const int u = t + NT * v;
            if (WIN % NT != 0 && u >= WIN) break;
            put(lx + u * 4, X_GRANULES, rx[v]);
        }
#pragma unroll
        for (int v = 0; v < NVA; v++) {
            const int u = t + NT * v;
            if (A_UNITS % NT != 0 && u >= A_UNITS) break;
            put(la + ((u / TAPS) * ROW + u % TAPS) * 4, A_GRANULES, ra[v]);
        }
    };

    // ---- the block in LDS
    accumulators<CFG> acc;
    int fp[TN];                                               // lane's positions in the current tile's window
    auto multiply = [&]() {
#pragma unroll
        for (int st = 0; st < STEPS; st++) {
            // the half's tap is 2 st + h
            const bool odd = 2 * st + 1 == TAPS;              // ... or, behind the last one, the tap of zeros (times the last one's positions)
            const int off = h && !odd ? TAP_OFFSETS::at(odd ? 0 : 2 * st + 1) : TAP_OFFSETS::at(2 * st);
            split_x8 fa[3][TM], fb[3][TN];
#pragma unroll
            for (int o = 0; o < 3; o++) {
                const int s = SPLIT_READ[o];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const int own = (wm * CFG::WM + i * 32 + l32) * ROW + h + 2 * st, at = odd && h ? BM * ROW : own;
                    fa[s][i] = __builtin_bit_cast(split_x8, *reinterpret_cast<const split_u4 *>(la + (s * A_GRANULES + at) * 4));
                }
#pragma unroll
                for (int j = 0; j < TN; j++)
                    fb[s][j] = __builtin_bit_cast(split_x8, *reinterpret_cast<const split_u4 *>(lx + (s * X_GRANULES + fp[j] + off) * 4));
            }
#pragma unroll
            for (int c = 0; c < 6; c++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc.t[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[SPLIT_A[c]][i], fb[SPLIT_B[c]][j], acc.t[i][j], 0, 0, 0);
        }
    };
    // sums that are not finite: the wavefront's part of the item again, with the fp32 instruction from global memory
    auto finish = [&](const place &p, int first, int end) {
        if (!__any(unscale(acc, 0, 0, 0, 0))) return;
        acc.clear();
#pragma unroll 1
        for (int c = first * CB; c < end * CB; c += 2)
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++) {
                if (tap % 9 == 0) __builtin_amdgcn_sched_barrier(0);       // nine taps' operands at a time
                float a[TM], b[TN];
#pragma unroll
                for (int i = 0; i < TM; i++) a[i] = A[(long)(p.m0 + wm * CFG::WM + i * 32 + l32) * lda + (long)(c + h) * TAPS + tap];
#pragma unroll
                for (int j = 0; j < TN; j++) b[j] = X[p.f0 + fp[j] + (long)(c + h) * chan_stride + TAP_OFFSETS::at(tap)];
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc.t[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc.t[i][j], 0, 0, 0);
            }
    };

    // ---- a piece of a remaining tile: park it in scratch; the last piece to arrive adds all of them
    constexpr int QUADS = TM * TN * 4;
    f32x4 *pieces = reinterpret_cast<f32x4 *>(scratch);
    unsigned *counters = reinterpret_cast<unsigned *>(scratch + (long)rest * splits * BM * BN);
    unsigned *piece_queue = counters + rest, *finished = piece_queue + 1, *xcd_queue = finished + 1;
    auto finish_piece = [&](int q, const place &p) {
        const int rt = (q - whole) / splits, z = (q - whole) % splits;
        f32x4 *mine = pieces + ((long)rt * splits + z) * QUADS * NT;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    store_handed_over(mine + ((i * TN + j) * 4 + r) * NT + t, f32x4{acc.t[i][j][4 * r], acc.t[i][j][4 * r + 1], acc.t[i][j][4 * r + 2], acc.t[i][j][4 * r + 3]});
        handed_over_stores_done();         // the piece is in memory before the ticket is taken
        __syncthreads();
        if (t == 0) ticket = atomicAdd(&counters[rt], 1u);
        __syncthreads();
        if (ticket != (unsigned)(splits - 1)) return;
        handed_over_loads_begin();
        const f32x4 *all = pieces + (long)rt * splits * QUADS * NT;
#pragma unroll 1
        for (int q0 = 0; q0 < QUADS; q0 += 2) {
            f32x4 part[2][SPLITS];
#pragma unroll
            for (int c = 0; c < SPLITS; c++)
#pragma unroll
                for (int d = 0; d < 2; d++) part[d][c] = load_handed_over(all + ((long)c * QUADS + q0 + d) * NT + t);
#pragma unroll
            for (int d = 0; d < 2; d++) {
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < SPLITS; c++) sum += part[d][c];
                const int qq = q0 + d, i = qq / (4 * TN), j = (qq / 4) % TN, r = qq % 4;
                const int row = p.m0 + wm * CFG::WM + i * 32 + 8 * r + 4 * h, col = p.n0 + wn * CFG::WN + j * 32 + l32;
#pragma unroll
                for (int e = 0; e < 4; e++) sum[e] = value(row + e, col, sum[e]);
#pragma unroll
                for (int e = 0; e < 4; e++) store(row + e, col, sum[e]);
            }
        }
        if (t == 0) counters[rt] = 0;      // zero again for the next launch
    };

    // this workgroup's queue (its XCD's range of whole tiles, then the pieces)
    const int queues = G % ttarget::XCDS == 0 ? ttarget::XCDS : 1, x = w % queues, in_queue = G / queues;
    const int lo = (int)((long)x * whole / queues), hi = (int)((long)(x + 1) * whole / queues);
    auto take_item = [&]() {
        const int i = in_queue + (int)atomicAdd(xcd_queue + x, 1u);
        return lo + i < hi ? lo + i : whole + (int)atomicAdd(piece_queue, 1u);
    };
    int cur = lo + w / queues;                     // G <= whole: every workgroup has a first item
    place here = place_of(item_tile(cur));
    auto aim = [&]() {
#pragma unroll
        for (int j = 0; j < TN; j++) fp[j] = (int)(pos(here.n0 + wn * CFG::WN + j * 32 + l32) - here.f0);
    };
    aim();
    acc.clear();
    if (t < 12) la[((t / 4) * A_GRANULES + BM * ROW) * 4 + t % 4] = 0;      // the tap of zeros
    load(here, item_first(cur));
    write();
    __syncthreads();
    while (cur < items) {
        if (t == 0) next_item = take_item();
        __syncthreads();
        const int next = __builtin_amdgcn_readfirstlane(next_item);
        // behind the last block the first one of the next item travels (of this item again when there is none: never used)
        const int then = next < items ? next : cur;
        const place there = place_of(item_tile(then));
        const int b_first = item_first(cur), b_end = item_end(cur);
        for (int b = b_first; b < b_end; b++) {
            place from = there;
            if (b + 1 < b_end) from = here;
            load(from, b + 1 < b_end ? b + 1 : item_first(then));
            __builtin_amdgcn_sched_barrier(0);
            multiply();
            __syncthreads();                       // every wavefront has read the block
            write();
            __syncthreads();
        }
        finish(here, b_first, b_end);
        if (!is_piece(cur)) tile_epilogue<CFG>(acc, M, N, here.m0, here.n0, value, store);
        else finish_piece(cur, here);
        acc.clear();
        here = there;
        aim();
        cur = next;
    }
    // the last workgroup to run out of items leaves the queues ready for the next launch
    if (t == 0 && atomicAdd(finished, 1u) == (unsigned)(G - 1)) {
        *piece_queue = 0;
        *finished = 0;
        for (int g = 0; g < queues; g++) xcd_queue[g] = 0;
    }
}

}  // namespace tgemm
#endif
