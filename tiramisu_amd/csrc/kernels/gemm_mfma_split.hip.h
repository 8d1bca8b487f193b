// fp32 dense contraction on the bf16 matrix cores of gfx950, without giving up a bit of the operands:
// C[m,n] = epilogue(sum_k A[m,k] * B[k,n]) with every fp32 operand element written as the exact sum of three bf16 numbers.
//
// A float has 24 significant bits, a bf16 number 8 and the same exponents.  With h = bf16(x), m = bf16(x - h), l = x - h - m
// (both differences are exact) l has at most 8 significant bits again: x = h + m + l.  A product is then nine products of
// bf16 numbers, which the matrix cores form exactly and add in fp32.  The six of them down to 2^-18 of the largest are taken,
//     mA*mB, mA*hB, lA*hB, hA*lB, hA*mB, hA*hB;
// the other three together are below 2^-24 of the product (they come near it: both operands 1 + 2^-8 - 2^-17), as much as one fp32
// multiplication may round by, and they are zero wherever the product has 24 significant bits or fewer (products of small whole
// numbers stay exact).  The largest comes last: a sum that one product dominates is then rounded at its full size once.  One product
// alone is within 1.45 units in the last place, 0.39 rms (fp32 instruction 0.5 and 0.29; with the largest first, rounded again
// by each of the five that follow, 3.4 and 0.60).  The order of the five costs nothing in accuracy; in this one neighbours share an operand
// where they can, which the power limit rewards (4096^3 590 us; smallest first 609, largest first 602; a convolution 64 to 64 channels, which
// waits for the parts from LDS, 170.5, 173 and 169).
// v_mfma_f32_32x32x16_bf16 does sixteen times the work of v_mfma_f32_32x32x2_f32 per cycle, so that six of it take 3/8 of the
// fp32 instruction's time; and an accumulator is rounded six times per sixteen k instead of eight times or more, which is why
// the error against 64 bits is smaller (uniform random operands, 2-norm: 4096^3 1.00e-6 against 1.15e-6, with partial sums
// 2048^3 4.9e-7 against 8.1e-7, 1024^3 1.7e-7 against 4.1e-7).
//
// What three bf16 numbers cannot hold is multiplied by the fp32 instruction.  Operands are scaled by 2^16 on the way (exactly;
// the sums are scaled back), so that the last part of the smallest fp32 number, 2^-149, is still a bf16 number, 2^-133.  What is
// left are infinities, NaNs and numbers that overflow, from 2^111 on, or whose products do: they all show as sums that are
// not finite, and a wavefront that finds one computes its part of the tile again from global memory (recompute_fp32): 4096^3 with one row
// of NaN 1150 us, with operands of 2^60, whose every product overflows, 2030 (bound by the L2; 600 without, 960 with the fp32 instruction),
// 1024^3 38 (18; 20).
//
// What bounds it: at 4096^3 the power limit (596 to 625 us on random operands, machines differ, 470 on zeros; 948 to 964 with the fp32 instruction), on small tiles the
// vector work of the split, seven instructions per element, each done once per tile (1024^3 17 to 19 us, 20.6 to 22.5 with the fp32 instruction).
#ifndef TIRAMISU_AMD_GEMM_MFMA_SPLIT_HIP_H
#define TIRAMISU_AMD_GEMM_MFMA_SPLIT_HIP_H
#include "gemm_mfma.hip.h"

namespace tgemm {

typedef __bf16 split_x8 __attribute__((ext_vector_type(8)));       // one operand of the matrix instruction
typedef __bf16 split_x2 __attribute__((ext_vector_type(2)));
typedef float split_f2 __attribute__((ext_vector_type(2)));
typedef uint32_t split_u4 __attribute__((ext_vector_type(4)));

// The constants of the split live in vector registers: the vector ALUs take almost twice as long for an operand from a scalar
// register or the instruction word (measured: and, multiply 1.75 ns per instruction and SIMD against 1.0).
constexpr float SPLIT_SCALE = 65536.f, SPLIT_UNSCALE = 1.f / (65536.f * 65536.f);
struct split_constants {
    float scale;
    uint32_t high;
    __device__ __forceinline__ split_constants() : scale(SPLIT_SCALE), high(0xffff0000u) { asm("" : "+v"(scale), "+v"(high)); }
};
__device__ __forceinline__ uint32_t split_pack(float a, float b) {
    const split_f2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, split_x2));     // v_cvt_pk_bf16_f32, to nearest even
}
// The three parts of two elements times 2^16, packed.
__device__ __forceinline__ void split_pair(const split_constants &c, float a, float b, uint32_t (&part)[3]) {
    a *= c.scale;
    b *= c.scale;
    part[0] = split_pack(a, b);
    a -= __builtin_bit_cast(float, part[0] << 16);
    b -= __builtin_bit_cast(float, part[0] & c.high);
    part[1] = split_pack(a, b);
    a -= __builtin_bit_cast(float, part[1] << 16);
    b -= __builtin_bit_cast(float, part[1] & c.high);
    part[2] = split_pack(a, b);
}
// The products taken: part of A, part of B; and the parts in the order in which they are needed.
constexpr int SPLIT_A[6] = {1, 1, 2, 0, 0, 0}, SPLIT_B[6] = {1, 0, 0, 2, 1, 0}, SPLIT_READ[3] = {1, 0, 2};

// Takes the scale out of the sums of the wavefront's rows from m0 and columns from n0; whether one that is in C is not finite.
template <class CFG>
__device__ __forceinline__ bool unscale(accumulators<CFG> &acc, int M, int N, int m0, int n0) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    float zero[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < CFG::TM; i++)
#pragma unroll
        for (int j = 0; j < CFG::TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc.t[i][j][r] *= SPLIT_UNSCALE;
                const bool inside = !CFG::EDGE || (m0 + i * 32 + 8 * (r / 4) + 4 * h + (r % 4) < M && n0 + j * 32 + l32 < N);
                zero[r % 4] = __builtin_fmaf(inside ? acc.t[i][j][r] : 0.f, 0.f, zero[r % 4]);
            }
    return !(zero[0] + zero[1] + zero[2] + zero[3] == 0.f);
}

// An operand: element (x, k) at base[x * ld + k] (KMAJOR) or base[k * ld + x]; XE, KE >= 4, 4 <= ld < 2^22.  As in linear_source
// (gemm_mfma.hip.h) loads are moved to four elements inside where the tile hangs over the operand (EDGE) and shifted afterwards, but
// only in the slice that holds the last k (LAST): in the others another row follows, and what is read behind XE only reaches
// elements of C that nobody stores.  An address is a scalar part (first row of the tile, first k of the slice, `i`) and a 32-bit
// part that a thread keeps from slice to slice (place): 64-bit vector additions for every load were a tenth of the vector work.
template <bool KMAJOR, bool EDGE>
struct split_source {
    const float *__restrict__ base;
    long ld;
    int XE, KE;
    __device__ __forceinline__ uint32_t place(int x0, int x, int k) const {
        if (EDGE) x = min(x, XE - 1 - x0);
        return 4u * (KMAJOR ? (uint32_t)x * (uint32_t)ld + (uint32_t)k : (uint32_t)k * (uint32_t)ld + (uint32_t)x);
    }
    // (x0 + x, k0 + k + i) and the three behind it; x0, k0, i uniform, `at` = place(x0, x, k)
    template <class LAST>
    __device__ __forceinline__ f32x4 load(int x0, int x, int k0, int k, int i, uint32_t at, LAST) const {
        const float *from;
        if (!EDGE || !LAST::value) {
            const float *scalar = base + (KMAJOR ? (long)x0 * ld + (k0 + i) : (long)(k0 + i) * ld + x0);
            from = reinterpret_cast<const float *>(reinterpret_cast<const char *>(scalar) + at);
        } else if (KMAJOR) {
            from = base + (long)min(x0 + x, XE - 1) * ld + min(k0 + k + i, KE - 4);
        } else {
            from = base + (long)min(k0 + k + i, KE - 1) * ld + min(x0 + x, XE - 4);
        }
        const f32x4_u v = *reinterpret_cast<const f32x4_u *>(from);
        return f32x4{v[0], v[1], v[2], v[3]};
    }
    template <class LAST>
    __device__ __forceinline__ f32x4 finish(f32x4 v, int x, int k, LAST) const {
        if (!EDGE || !LAST::value) return v;
        if (KMAJOR) return shifted_down(v, max(k - (KE - 4), 0));
        const f32x4 none = {0.f, 0.f, 0.f, 0.f};
        return k < KE ? shifted_down(v, max(x - (XE - 4), 0)) : none;
    }
    // the four elements (x0 + x, k0 + k + i ..), `at` = place(x0, x, k), i uniform: all there (WHOLE), or zero behind KE
    template <bool WHOLE>
    __device__ __forceinline__ f32x4 four(int x0, int k0, int k, int i, uint32_t at) const {
        const float *const scalar = base + (KMAJOR ? (long)x0 * ld + k0 : (long)k0 * ld + x0);
        auto element = [&](const float *from, int d) {          // d k further
            return reinterpret_cast<const char *>(from) + (at + 4u * (uint32_t)(KMAJOR ? d : d * (int)ld));
        };
        f32x4 v;
        if (WHOLE && KMAJOR) {
            const f32x4_u q = *reinterpret_cast<const f32x4_u *>(element(scalar + i, 0));
            return f32x4{q[0], q[1], q[2], q[3]};
        }
#pragma unroll
        for (int e = i; e < i + 4; e++) {
            const int last = KE - 1 - k0 - k;                     // (negative where k0 + k lies behind KE)
            if (WHOLE) v[e - i] = *reinterpret_cast<const float *>(element(scalar + (long)e * ld, 0));
            else v[e - i] = *reinterpret_cast<const float *>(element(scalar, min(e, last)));
            if (!WHOLE && e > last) v[e - i] = 0.f;
        }
        return v;
    }
};

// The wavefront's part of a tile with the fp32 instruction, operands straight from global memory: of the slices first, first + step, ...
// of BK k the k in [from, from + 16), eight of them on each half of the wavefront, so that a row is read 64 bytes at a time.
template <class CFG, class SRCA, class SRCB>
__device__ __forceinline__ void recompute_fp32(accumulators<CFG> &acc, const SRCA &A, const SRCB &B, int K, int m0, int n0, int first, int step, int from) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    uint32_t ata[CFG::TM], atb[CFG::TN];
#pragma unroll
    for (int i = 0; i < CFG::TM; i++) ata[i] = A.place(m0, i * 32 + l32, 8 * h);
#pragma unroll
    for (int j = 0; j < CFG::TN; j++) atb[j] = B.place(n0, j * 32 + l32, 8 * h);
    auto slice = [&](int k, auto whole) {
        constexpr bool WHOLE = decltype(whole)::value;
        f32x4 a[2][CFG::TM], b[2][CFG::TN];
#pragma unroll
        for (int q = 0; q < 2; q++) {
#pragma unroll
            for (int i = 0; i < CFG::TM; i++) a[q][i] = A.template four<WHOLE>(m0, k, 8 * h, 4 * q, ata[i]);
#pragma unroll
            for (int j = 0; j < CFG::TN; j++) b[q][j] = B.template four<WHOLE>(n0, k, 8 * h, 4 * q, atb[j]);
        }
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < CFG::TM; i++)
#pragma unroll
                    for (int j = 0; j < CFG::TN; j++)
                        acc.t[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q][i][e], b[q][j][e], acc.t[i][j], 0, 0, 0);
    };
    acc.clear();
    int k = first * CFG::BK + from;
#pragma unroll 1
    for (; k + 16 <= K; k += step * CFG::BK) slice(k, std::true_type());
    if (CFG::EDGE && k < K) slice(k, std::false_type());
}

// ---------------------------------------------------------------------------------------------------------------------
// Large tiles: a slice is split once by the workgroup, on its way from registers to LDS.
//
// One operand's slice of X x BK elements as three planes of 16-byte granules, granule (kq, x) = the 8 consecutive k of k-group kq of
// row x in bf16: a lane's whole operand of the matrix instruction.  A thread loads units of KU k of one row (KMAJOR) or of
// four neighbouring rows, which needs no transposition: the conversion packs any two registers.
template <int X, int BK, int NT, bool KMAJOR>
struct split_tile {
    static constexpr int ROWS = KMAJOR ? 1 : 4;                   // rows of a unit
    static constexpr int KU = X * BK / (8 * ROWS) >= NT ? 8 : X * BK / (4 * ROWS) >= NT ? 4 : 2;
    static constexpr int UNITS = X * BK / (KU * ROWS), NV = UNITS / NT;      // units per slice, per thread
    static constexpr int LOADS = KMAJOR ? KU / 4 : KU;            // 16-byte loads per unit
    static constexpr int PARTS = 8 / KU;                          // units per granule (and row)
    // Positions: rows as they are (KMAJOR) or the four rows of a unit a class stride apart, so that lanes store to neighbouring
    // granules; the strides spread the k-groups (classes) that 16 lanes store or read together over the banks.
    static constexpr int CLASS = X / 4 + 4;
    static constexpr int GROUP = KMAJOR ? X + 16 / (BK / 8) : 4 * CLASS;
    static constexpr int PLANE_WORDS = (BK / 8) * GROUP * 4;
    static constexpr int WORDS = 3 * PLANE_WORDS;
    static_assert(NV * NT == UNITS && NV > 0 && LOADS > 0, "a slice must split evenly over the threads");

    static __device__ __forceinline__ int granule(int kq, int x) { return kq * GROUP + (KMAJOR ? x : (x >> 2) + (x & 3) * CLASS); }
    static __device__ __forceinline__ void unit(int idx, int &x, int &k) {
        if (KMAJOR) { k = KU * (idx % (BK / KU)); x = idx / (BK / KU); }
        else { x = 4 * ((idx / PARTS) % (X / 4)); k = KU * (idx % PARTS) + 8 * (idx / PARTS / (X / 4)); }
    }
    template <class SRC>
    static __device__ __forceinline__ void place(const SRC &src, int x0, uint32_t (&at)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int x, k;
            unit(threadIdx.x + NT * v, x, k);
            at[v] = src.place(x0, x, k);
        }
    }
    template <class SRC, class LAST>
    static __device__ __forceinline__ void load(const SRC &src, int x0, int k0, const uint32_t (&at)[NV], f32x4 (&regs)[NV][LOADS], LAST last) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int x, k;
            unit(threadIdx.x + NT * v, x, k);
#pragma unroll
            for (int i = 0; i < LOADS; i++) regs[v][i] = src.load(x0, x, k0, k, KMAJOR ? 4 * i : i, at[v], last);
        }
    }
    template <class SRC, class LAST>
    static __device__ __forceinline__ void store(uint32_t *lds, const f32x4 (&regs)[NV][LOADS], const SRC &src, int x0, int k0, LAST last, const split_constants &sc) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int x, k;
            unit(threadIdx.x + NT * v, x, k);
            f32x4 e[LOADS];
#pragma unroll
            for (int i = 0; i < LOADS; i++) e[i] = src.finish(regs[v][i], x0 + x, k0 + k + (KMAJOR ? 4 * i : i), last);
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                uint32_t w[3][KU / 2];
#pragma unroll
                for (int p = 0; p < KU / 2; p++) {
                    uint32_t part[3];
                    split_pair(sc, KMAJOR ? e[p / 2][2 * (p % 2)] : e[KMAJOR ? 0 : 2 * p][r], KMAJOR ? e[p / 2][2 * (p % 2) + 1] : e[KMAJOR ? 0 : 2 * p + 1][r], part);
#pragma unroll
                    for (int s = 0; s < 3; s++) w[s][p] = part[s];
                }
#pragma unroll
                for (int s = 0; s < 3; s++) {
                    uint32_t *to = lds + s * PLANE_WORDS + granule(k / 8, x + r) * 4 + (k % 8) / 2;
                    if constexpr (KU == 8) *reinterpret_cast<split_u4 *>(to) = split_u4{w[s][0], w[s][1], w[s][2], w[s][3]};
                    else if constexpr (KU == 4) *reinterpret_cast<uint64_t *>(to) = ((uint64_t)w[s][1] << 32) | w[s][0];
                    else *to = w[s][0];
                }
            }
        }
    }
    static __device__ __forceinline__ split_x8 read(const uint32_t *lds, int part, int x, int kq) {
        return __builtin_bit_cast(split_x8, *reinterpret_cast<const split_u4 *>(lds + part * PLANE_WORDS + granule(kq, x) * 4));
    }
};

// As config (gemm_mfma.hip.h): WGM x WGN wavefronts tile the block, WGK groups of them take 1/WGK of every slice.  AHEAD: the parts of
// the next slice are read while one is multiplied (one step per wavefront and slice; tiles whose registers hold two sets).
template <int BM_, int BN_, int BK_, int WGM_, int WGN_, bool A_KMAJOR_, bool B_KMAJOR_, bool EDGE_, int WGK_, bool AHEAD_>
struct config_split {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WGM = WGM_, WGN = WGN_, WGK = WGK_;
    static constexpr bool A_KMAJOR = A_KMAJOR_, B_KMAJOR = B_KMAJOR_, EDGE = EDGE_, AHEAD = AHEAD_;
    static constexpr int NT = 64 * WGM * WGN * WGK;
    static constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    typedef split_tile<BM, BK, NT, A_KMAJOR> opA;
    typedef split_tile<BN, BK, NT, B_KMAJOR> opB;
    static constexpr int STAGE_FLOATS = opA::WORDS + opB::WORDS;
    static constexpr int LDS_BYTES = 2 * STAGE_FLOATS * 4;
    static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be made of 32x32 MFMA tiles");
    static_assert(BK == 16 * WGK, "one step per wavefront and slice");
    static_assert(LDS_BYTES == ttarget::split_lds_bytes(BM, A_KMAJOR, B_KMAJOR) && LDS_BYTES <= ttarget::LDS_BYTES_PER_CU, "two stages must fit");
    static_assert(BK == ttarget::split_slice(BM), "slice");
    static_assert(WGK == 1 || (WGK - 1) * WGM * WGN * TM * TN * 16 * 64 <= 2 * STAGE_FLOATS, "LDS too small for the K reduction");
};

// acc += A(m0.., :) * B(:, n0..) over K > BK.  All threads of the workgroup call this together; the last access to LDS is behind a barrier.
template <class CFG, class SRCA, class SRCB>
__device__ __forceinline__ void tile_accumulate_split(accumulators<CFG> &acc, const SRCA &A, const SRCB &B, int M, int N, int K, int m0, int n0, float *lds_) {
    typedef typename CFG::opA opA;
    typedef typename CFG::opB opB;
    constexpr int TM = CFG::TM, TN = CFG::TN, BK = CFG::BK;
    uint32_t *lds = reinterpret_cast<uint32_t *>(lds_);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wk = wave / (CFG::WGM * CFG::WGN), wmn = wave % (CFG::WGM * CFG::WGN);
    const int wm = wmn / CFG::WGN, wn = wmn % CFG::WGN;
    const int l32 = lane & 31, h = lane >> 5;

    f32x4 ra[opA::NV][opA::LOADS], rb[opB::NV][opB::LOADS];
    uint32_t ata[opA::NV], atb[opB::NV];
    opA::place(A, m0, ata);
    opB::place(B, n0, atb);
    const split_constants sc;
    auto stage_a = [&](int stage) -> uint32_t * { return lds + stage * CFG::STAGE_FLOATS; };
    auto stage_b = [&](int stage) -> uint32_t * { return lds + stage * CFG::STAGE_FLOATS + opA::WORDS; };
    const int KT = (K + BK - 1) / BK;
    // The slice that holds the last k comes first (number 0), ahead of the loop: the loop then has no guards and no branches.
    // Behind the last number the first slice of K is loaded and stored again and never multiplied: where a path without
    // loads joins, the compiler would wait for all loads in flight instead of those it needs.
    auto slice_of = [&](int n) -> int { return n < KT ? n - 1 : 0; };
    auto load = [&](int n, auto last) {
        const int s = decltype(last)::value ? KT - 1 : slice_of(n);
        opA::load(A, m0, s * BK, ata, ra, last);
        opB::load(B, n0, s * BK, atb, rb, last);
    };
    auto store = [&](int n, int stage, auto last) {
        const int s = decltype(last)::value ? KT - 1 : slice_of(n);
        opA::store(stage_a(stage), ra, A, m0, s * BK, last, sc);
        opB::store(stage_b(stage), rb, B, n0, s * BK, last, sc);
    };
    auto read = [&](int stage, split_x8 (&fa)[3][TM], split_x8 (&fb)[3][TN]) {
        const int kq = 2 * wk + h;
#pragma unroll
        for (int o = 0; o < 3; o++) {
            const int p = SPLIT_READ[o];
#pragma unroll
            for (int i = 0; i < TM; i++) fa[p][i] = opA::read(stage_a(stage), p, wm * CFG::WM + i * 32 + l32, kq);
#pragma unroll
            for (int j = 0; j < TN; j++) fb[p][j] = opB::read(stage_b(stage), p, wn * CFG::WN + j * 32 + l32, kq);
        }
    };
    auto multiply = [&](const split_x8 (&fa)[3][TM], const split_x8 (&fb)[3][TN]) {
#pragma unroll
        for (int c = 0; c < 6; c++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    acc.t[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[SPLIT_A[c]][i], fb[SPLIT_B[c]][j], acc.t[i][j], 0, 0, 0);
    };
    typedef std::true_type yes;
    typedef std::false_type no;
    load(0, yes());
    store(0, 0, yes());
    load(1, no());
    if constexpr (!CFG::AHEAD) {
        // the two wavefronts of a SIMD cover each other's LDS reads
        __syncthreads();
        for (int n = 0; n < KT; n++) {
            store(n + 1, (n + 1) & 1, no());
            load(n + 2, no());
            split_x8 fa[3][TM], fb[3][TN];
            read(n & 1, fa, fb);
            multiply(fa, fb);
            __syncthreads();
        }
    } else {
        // While a slice is multiplied the next one's parts are read from their stage and the one after that is split and stored into
        // this slice's own, which every wavefront has read: nothing in an iteration waits for anything else in it, and the
        // scheduling groups deal vector, LDS and matrix instructions out evenly (2048^3 with 128 x 128 tiles 94 us; with
        // the reads at the head of the slice that needs them 105).
        split_x8 fa[2][3][TM], fb[2][3][TN];
        store(1, 1, no());
        load(2, no());
        __syncthreads();
        read(0, fa[0], fb[0]);
        __syncthreads();
        for (int b = 0; b < KT; b += 2) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if (b + u >= KT) break;
                store(b + u + 2, u, no());
                load(b + u + 3, no());
                read(u ^ 1, fa[u ^ 1], fb[u ^ 1]);
                multiply(fa[u], fb[u]);
                constexpr int MFMAS = 6 * TM * TN, READS = 3 * (TM + TN), ELEMENTS = 4 * (opA::NV * opA::LOADS + opB::NV * opB::LOADS);
#pragma unroll
                for (int i = 0; i < MFMAS; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (i < READS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, ELEMENTS * 7 / MFMAS + 1, 0);
                    if (i > MFMAS / 4) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
            }
        }
    }
    m0 += wm * CFG::WM;
    n0 += wn * CFG::WN;
    if (__any(unscale(acc, M, N, m0, n0))) recompute_fp32(acc, A, B, K, m0, n0, 0, 1, wk * 16);
}

// ---------------------------------------------------------------------------------------------------------------------
// 64 x 64 tiles (whole ones only): every wavefront of a workgroup multiplies the whole tile over its own k (slices of 16, dealt round robin) and
// nothing is shared until the sums are added: no barrier in the loop, and every element is read from LDS and split once.
template <bool A_KMAJOR_, bool B_KMAJOR_>
struct config_waves {
    static constexpr int BM = 64, BN = 64, BK = 16, WAVES = 8;
    static constexpr bool A_KMAJOR = A_KMAJOR_, B_KMAJOR = B_KMAJOR_, EDGE = false;
    static constexpr int NT = 64 * WAVES, TM = BM / 32, TN = BN / 32;
    static constexpr int A_WORDS = BM * BK + (A_KMAJOR ? 0 : 4 * BK), B_WORDS = BN * BK + (B_KMAJOR ? 0 : 4 * BK);
    static constexpr int WAVE_WORDS = A_WORDS + B_WORDS;
    static constexpr int STAGING = 2 * WAVES * WAVE_WORDS * 4, SUMS = WAVES * TM * TN * 16 * 64 * 4;
    static constexpr int LDS_BYTES = STAGING > SUMS ? STAGING : SUMS;
    static constexpr int QUADS = TM * TN * 4, SHARE = QUADS / WAVES;       // of four accumulator registers; those a wavefront finishes
    static_assert(LDS_BYTES == ttarget::split_lds_bytes(BM, A_KMAJOR, B_KMAJOR), "two stages of every wavefront's slices");
};

// Between the accesses of a wavefront's lanes to LDS that only they use: what was written or read before is done for what is written or
// read behind.  The LDS executes a wavefront's accesses in order, so this holds the compiler alone and is no instruction.
__device__ __forceinline__ void wave_lds_in_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// One operand's X x 16 slice of one wavefront, in fp32.
template <int X, bool KMAJOR>
struct wave_operand {
    static constexpr int NV = X / 16;                  // 16-byte loads per lane
    static __device__ __forceinline__ void unit(int idx, int &x, int &k) {
        if (KMAJOR) { k = 4 * (idx % 4); x = idx / 4; }
        else { x = 4 * (idx % (X / 4)); k = idx / (X / 4); }
    }
    // (K-major: rows of 64 bytes, the granules of a row exchanged so that 16 rows' reads hit different banks; else rows of X floats,
    // the second eight half the banks further)
    static __device__ __forceinline__ int word(int x, int k) {
        return KMAJOR ? x * 16 + ((k >> 2) ^ ((x >> 2) & 3)) * 4 : k * X + x + (k >> 3) * 32;
    }
    template <class SRC>
    static __device__ __forceinline__ void place(const SRC &src, int x0, uint32_t (&at)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int x, k;
            unit((threadIdx.x & 63) + 64 * v, x, k);
            at[v] = src.place(x0, x, k);
        }
    }
    template <class SRC>
    static __device__ __forceinline__ void load(const SRC &src, int x0, int k0, const uint32_t (&at)[NV], f32x4 (&regs)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int x, k;
            unit((threadIdx.x & 63) + 64 * v, x, k);
            regs[v] = src.load(x0, x, k0, k, 0, at[v], std::false_type());
        }
    }
    static __device__ __forceinline__ void store(uint32_t *lds, const f32x4 (&regs)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int x, k;
            unit((threadIdx.x & 63) + 64 * v, x, k);
            *reinterpret_cast<f32x4 *>(lds + word(x, k)) = regs[v];
        }
    }
    // the eight k of a lane's row
    static __device__ __forceinline__ void read(const uint32_t *lds, int x, int h, float (&e)[8]) {
        if (KMAJOR) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(lds + word(x, 8 * h + 4 * i));
#pragma unroll
                for (int c = 0; c < 4; c++) e[4 * i + c] = v[c];
            }
        } else {
            const float *p = reinterpret_cast<const float *>(lds) + h * (8 * X + 32) + x;
#pragma unroll
            for (int i = 0; i < 8; i++) e[i] = p[i * X];
        }
    }
};

__device__ __forceinline__ void split_eight(const split_constants &sc, const float (&e)[8], split_x8 (&out)[3]) {
    uint32_t w[3][4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        uint32_t part[3];
        split_pair(sc, e[2 * p], e[2 * p + 1], part);
#pragma unroll
        for (int s = 0; s < 3; s++) w[s][p] = part[s];
    }
#pragma unroll
    for (int s = 0; s < 3; s++) out[s] = __builtin_bit_cast(split_x8, split_u4{w[s][0], w[s][1], w[s][2], w[s][3]});
}

// acc += the wavefront's share of A(m0.., :) * B(:, n0..) over K, whole tiles and slices
template <class CFG, class SRCA, class SRCB>
__device__ __forceinline__ void tile_accumulate_waves(accumulators<CFG> &acc, const SRCA &A, const SRCB &B, int M, int N, int K, int m0, int n0, float *lds_) {
    typedef wave_operand<CFG::BM, CFG::A_KMAJOR> opA;
    typedef wave_operand<CFG::BN, CFG::B_KMAJOR> opB;
    constexpr int TM = CFG::TM, TN = CFG::TN, W = CFG::WAVES, BK = CFG::BK, T = TM * TN;
    static_assert(TM == 2 && TN == 2, "four tile products");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    uint32_t *lds = reinterpret_cast<uint32_t *>(lds_) + 2 * wave * CFG::WAVE_WORDS;      // two stages of the wavefront's own
    const int KT = K / BK;
    const int mine = KT > wave ? (KT - wave + W - 1) / W : 0;     // the wavefront's slices: wave, wave + W, ...
    f32x4 ra[opA::NV], rb[opB::NV];
    uint32_t ata[opA::NV], atb[opB::NV];
    opA::place(A, m0, ata);
    opB::place(B, n0, atb);
    const split_constants sc;
    // (behind its end the wavefront's last slice again: see tile_accumulate_split)
    auto load = [&](int n) {
        const int s = wave + min(n, mine - 1) * W;
        opA::load(A, m0, s * BK, ata, ra);
        opB::load(B, n0, s * BK, atb, rb);
    };
    auto store = [&](int stage) {
        wave_lds_in_order();                 // the lanes have read what the stage held
        opA::store(lds + stage * CFG::WAVE_WORDS, ra);
        opB::store(lds + stage * CFG::WAVE_WORDS + CFG::A_WORDS, rb);
        wave_lds_in_order();                 // the lanes read what the others stored
    };
    // A slice is four tile products; while the matrix cores work on one, the vector ALUs split the block of 32 rows or columns that
    // the next one needs, requested from LDS one product earlier: column block 1, row block 1, then the first row and
    // column block of the next slice.
    auto read_block = [&](int block, int stage, float (&to)[8]) {       // row blocks 0, 1, column blocks 2, 3
        const uint32_t *la = lds + stage * CFG::WAVE_WORDS;
        if (block < TM) opA::read(la, block * 32 + l32, h, to);
        else opB::read(la + CFG::A_WORDS, (block - TM) * 32 + l32, h, to);
    };
    split_x8 fa[TM][3], fb[TN][3];
    float e[2][8];                           // elements on the way from LDS, by the parity of the tile product that splits them
    auto slice = [&](int stage) {
        split_x8 na[3], nb[3];
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int i = t / TN, j = t % TN;
            if (t == 0) read_block(1, stage, e[1]);
            else if (t == 1) read_block(0, stage ^ 1, e[0]);
            else if (t == 2) read_block(2, stage ^ 1, e[1]);
            else read_block(3, stage ^ 1, e[0]);
            if (t == 0) split_eight(sc, e[0], fb[1]);
            else if (t == 1) split_eight(sc, e[1], fa[1]);
            else if (t == 2) split_eight(sc, e[0], na);
            else split_eight(sc, e[1], nb);
#pragma unroll
            for (int c = 0; c < 6; c++) acc.t[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][SPLIT_A[c]], fb[j][SPLIT_B[c]], acc.t[i][j], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < 6; c++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int p = 0; p < 3; p++) { fa[0][p] = na[p]; fb[0][p] = nb[p]; }
    };
    if (mine > 0) {
        load(0);
        store(0);
        load(1);
        float e0[8], e1[8];
        read_block(0, 0, e0);
        read_block(TM, 0, e1);
        read_block(TM + 1, 0, e[0]);
        split_eight(sc, e0, fa[0]);
        split_eight(sc, e1, fb[0]);
        for (int b = 0; b < mine; b += 2) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if (b + u >= mine) break;
                store(u ^ 1);
                load(b + u + 2);
                __builtin_amdgcn_sched_barrier(0);
                slice(u);
            }
        }
    }
    if (__any(unscale(acc, M, N, m0, n0))) recompute_fp32(acc, A, B, K, m0, n0, wave, W, 0);
}

// The sums of the wavefronts, added in their order; each finishes its SHARE of the tile's quads.  value and store as in tile_epilogue.
template <class CFG, class VALUE, class STORE>
__device__ __forceinline__ void tile_finish_waves(const accumulators<CFG> &acc, int m0, int n0, float *lds, VALUE value, STORE store) {
    constexpr int W = CFG::WAVES, Q = CFG::QUADS, SHARE = CFG::SHARE;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    f32x4 *slots = reinterpret_cast<f32x4 *>(lds);
    __syncthreads();                         // every wavefront has read its slices
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const f32x16 &t = acc.t[q / 4 / CFG::TN][q / 4 % CFG::TN];
        slots[(wave * Q + q) * 64 + lane] = f32x4{t[4 * (q % 4)], t[4 * (q % 4) + 1], t[4 * (q % 4) + 2], t[4 * (q % 4) + 3]};
    }
    __syncthreads();
    f32x4 sum[SHARE];
#pragma unroll
    for (int c = 0; c < SHARE; c++) {
        sum[c] = slots[(wave * SHARE + c) * 64 + lane];
#pragma unroll
        for (int g = 1; g < W; g++) sum[c] += slots[(g * Q + wave * SHARE + c) * 64 + lane];
    }
#pragma unroll
    for (int pass = 0; pass < 2; pass++)
#pragma unroll
        for (int c = 0; c < SHARE; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int q = wave * SHARE + c;
                const int row = m0 + (q / 4 / CFG::TN) * 32 + 8 * (q % 4) + 4 * h + e, col = n0 + (q / 4 % CFG::TN) * 32 + l32;
                if (pass == 0) sum[c][e] = value(row, col, sum[c][e]);
                else store(row, col, sum[c][e]);
            }
}

// ---- a tile from the first load to the last store.  The tiles that are used, whichever of the two kinds they are:
template <int EDGE_LENGTH, bool A_KMAJOR, bool B_KMAJOR, bool GUARDED> struct split_config;
template <bool AK, bool BK_, bool G> struct split_config<256, AK, BK_, G> { typedef config_split<256, 256, 16, 2, 4, AK, BK_, G, 1, false> type; };
template <bool AK, bool BK_, bool G> struct split_config<128, AK, BK_, G> { typedef config_split<128, 128, 32, 2, 2, AK, BK_, G, 2, true> type; };
template <bool AK, bool BK_> struct split_config<64, AK, BK_, false> { typedef config_waves<AK, BK_> type; };

template <class CFG, class VALUE, class STORE>
__device__ __forceinline__ void split_mainloop(const float *__restrict__ A, long lda, const float *__restrict__ B, long ldb, int M, int N, int K, int m0, int n0,
                                               float *lds, VALUE value, STORE store) {
    accumulators<CFG> acc;
    acc.clear();
    const split_source<CFG::A_KMAJOR, CFG::EDGE> sa{A, lda, M, K};
    const split_source<CFG::B_KMAJOR, CFG::EDGE> sb{B, ldb, N, K};
    if constexpr (CFG::BM == 64) {
        tile_accumulate_waves<CFG>(acc, sa, sb, M, N, K, m0, n0, lds);
        tile_finish_waves<CFG>(acc, m0, n0, lds, value, store);
    } else {
        tile_accumulate_split<CFG>(acc, sa, sb, M, N, K, m0, n0, lds);
        if (tile_reduce_k<CFG>(acc, lds)) tile_epilogue<CFG>(acc, M, N, m0, n0, value, store);
    }
}

template <class CFG>
__global__ void __launch_bounds__(CFG::NT) sgemm_split_kernel(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int M, int N, int K,
                                                              long lda, long ldb, long ldc, float alpha, float beta) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    int tm, tn;
    tile_of_block((M + CFG::BM - 1) / CFG::BM, (N + CFG::BN - 1) / CFG::BN, tm, tn);
    split_mainloop<CFG>(A, lda, B, ldb, M, N, K, tm * CFG::BM, tn * CFG::BN, lds, axpby_value{C, ldc, alpha, beta}, axpby_store{C, ldc});
}

template <class CFG>
__global__ void __launch_bounds__(CFG::NT) sgemm_split_batched_kernel(const sgemm_batch batch, int M, int N, int K, long lda, long ldb, long ldc, float alpha,
                                                                      float beta) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    int tm, tn;
    tile_of_block((M + CFG::BM - 1) / CFG::BM, (N + CFG::BN - 1) / CFG::BN, tm, tn);
    const float *A = batch.A[blockIdx.z], *B = batch.B[blockIdx.z];
    float *C = batch.C[blockIdx.z];
    split_mainloop<CFG>(A, lda, B, ldb, M, N, K, tm * CFG::BM, tn * CFG::BN, lds, axpby_value{C, ldc, alpha, beta}, axpby_store{C, ldc});
}

}  // namespace tgemm
#endif
