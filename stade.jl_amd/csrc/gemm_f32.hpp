// fp32 GEMM on CDNA4 matrix cores, with a fused per-element epilogue.
//
//   C(m, n) = sum over segments s of  sum_k A_s(m, k) * B_s(k, n),   epi(m, n, C(m, n), epi.load(m, n))
//
// An epilogue functor reads what it needs of the old output in load(m, n) (gathered for the
// whole tile before any store) and writes in operator()(m, n, v, loaded).
//
// A_s is M x K_s and B_s is K_s x N, column-major (Julia) with either storage order:
//   A_KM = false: A(m, k) at A[m + k * lda] (m contiguous);  A_KM = true: at A[k + m * lda]
//   B_KM = true:  B(k, n) at B[k + n * ldb] (k contiguous);  B_KM = false: at B[n + k * ldb]
// Up to two segments accumulate into one tile, so a tangent product such as
// W1d * X + W1 * Xd is one launch.  A dual launch instead reads both segments in the same K
// steps and writes two outputs, P = A0 B0 and Q = A0 B1 + A1 B0 (a product with its tangent).
//
// Arithmetic: six bf16 products of operands split into three bf16 parts (split_bf16.hpp).  A
// step's products are summed from zero and then added to the tile's total: one rounding at the
// total's size per 16 k, where v_mfma_f32_32x32x2_f32 rounds every 2 k (and where the six
// products accumulated straight into the total would round six times).  Against 64 bits (N(0, 1)
// times U(0, 1) operands) the normwise error is 1.4e-7 at K = 784 and 3.1e-7 at K = 4096; of
// v_mfma_f32_32x32x2_f32 5.0e-7 and 1.1e-6, accumulated straight 4.0e-7 and 9.9e-7.
// The matrix cores run bf16 at 16 times the fp32 rate, so six products leave a factor of 2.7.
// Measured, us with fp32 MFMAs -> split: 1024 x 4096 x 784 64 -> 55, its dual 179 -> 121;
// 1024 x 784 x 4096 (atomic K slices) 77 -> 60, dual 204 -> 149.  What bounds the loop now is
// the splitting (12 vector instructions a pair of elements, 100 a wave and step beside 24 MFMAs)
// and the loads and barriers that a block's two waves a SIMD do not hide wholly: without the
// splitting and the loads the same loop runs at 270 TFLOP/s, with them at 165-180.
// A block that meets an element the split cannot hold forms its tile again with fp32 matrix
// instructions (fp32_loop): the results there are those of plain fp32.
//
// Tiling: a 256-thread block (4 waves) computes a 128 x BNT tile of C (BNT = 128 or 64);
// each wave a 64 x BNT/2 part as 2 x BNT/64 MFMA 32 x 32 tiles.  K advances 16 at a time
// through two LDS buffers: while a step's MFMAs run from one, the next step is split and stored to
// the other and the step after that is being loaded; one barrier a step, and two blocks a CU,
// so that one block's splitting overlaps the other's MFMAs.  The partial K steps (K % 16, one a
// segment) come first, in the prologue, so that the steps of the loop load without tests.
// The MFMA operands are swapped (B tile as the matrix-core A operand) so that the
// accumulator's lane index runs along m: each epilogue store of a wave covers 32 consecutive
// rows of a column-major C, a 128-byte segment.
//
// Split K: with `ksplit` > 1 the K steps (of all segments, in order) are cut into ksplit
// contiguous ranges, one per blockIdx.z; each writes its partial tile to a scratch slice
// and a second kernel adds the slices in slice order and applies the epilogue.  An epilogue
// that only accumulates (C += v: a shadow, as the generated adjoint code accumulates it)
// can instead take the slices by atomic addition straight into C (`Epi::kAtomic`): no
// partial tiles and no second kernel, with the slices' order left to the hardware.  The host
// picks the tile width and the split from a cost model (plan()).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "split_bf16.hpp"

namespace stade {
namespace gemm {

constexpr int BM = 128, KT = 16, NT = 256;
constexpr int KQ = KT / 4;  // k-planes per step of the fp32 loop

// The fp32 loop's LDS tiles use a "quad" layout: element (k, r) of a ROWS x KT tile sits at
// S[(k / 4) * ldq(ROWS) + r * 4 + k % 4], i.e. KT / 4 k-planes each holding, per row, that
// row's four consecutive k values as one 16-byte cell: a matrix-core fragment is one 128-bit
// LDS read per 32 rows and 4 k values.
template <int ROWS>
constexpr int ldq() {
    return ROWS * 4 + 128 / KT;
}

struct Seg {
    const float* A;
    const float* B;
    long lda, ldb;
    int K;
};

struct Args {
    Seg seg[2];
    int nseg;
    int M, N;
    int ksplit;     // blockIdx.z ranges over ksplit slices of the K steps
    bool atomic;    // ksplit > 1: slices added into the output by atomics (Epi::kAtomic)
    float* part;    // ksplit > 1, !atomic: partial tiles, slice z at part + z * M * N, column-major
    bool bufok;     // set by prepare(): every operand's byte extent fits 31 bits
    uint32_t abytes[2], bbytes[2];  // set by prepare(): the operands' byte extents
};

// The cells (row, k-plane) of a ROWS x KT tile are shared out over the block: cell
// e = threadIdx.x + NT * q of this thread is
//   KMAJ (k contiguous in memory):    row e / KQ,   plane e % KQ
//   !KMAJ (rows contiguous in memory): row e % ROWS, plane e / ROWS (four 4-byte loads per
//                                     cell, one per k; a wave reads 64 consecutive rows of a k)
template <int ROWS>
struct Stage {
    float4 v[ROWS * KQ / NT];
};

template <bool KMAJ, int ROWS>
__device__ __forceinline__ void cell_of(int e, int& r, int& kq) {
    if (KMAJ) {
        r = e / KQ;
        kq = e % KQ;
    } else {
        r = e % ROWS;
        kq = e / ROWS;
    }
}

// A tile (r 0..ROWS-1, k 0..KT-1) at (r0, k0) into registers; zero outside rows x K.
template <bool KMAJ, int ROWS>
__device__ __forceinline__ void load_tile(Stage<ROWS>& st, const float* __restrict__ P, long ld, int rows, int K, int r0,
                                          int k0) {
#pragma unroll
    for (int q = 0; q < ROWS * KQ / NT; ++q) {
        int rr, kq;
        cell_of<KMAJ, ROWS>(threadIdx.x + NT * q, rr, kq);
        const int r = r0 + rr, k = k0 + 4 * kq;
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < rows) {
            if (KMAJ) {
                const float* p = P + (long)k + (long)r * ld;
                if (k + 0 < K) x.x = p[0];
                if (k + 1 < K) x.y = p[1];
                if (k + 2 < K) x.z = p[2];
                if (k + 3 < K) x.w = p[3];
            } else {
                const float* p = P + (long)r + (long)k * ld;
                if (k + 0 < K) x.x = p[0];
                if (k + 1 < K) x.y = p[ld];
                if (k + 2 < K) x.z = p[2 * ld];
                if (k + 3 < K) x.w = p[3 * ld];
            }
        }
        st.v[q] = x;
    }
}

// Registers -> LDS tile in the quad layout (one 16-byte store per cell)
template <bool KMAJ, int ROWS>
__device__ __forceinline__ void store_tile(const Stage<ROWS>& st, float* __restrict__ S) {
#pragma unroll
    for (int q = 0; q < ROWS * KQ / NT; ++q) {
        int rr, kq;
        cell_of<KMAJ, ROWS>(threadIdx.x + NT * q, rr, kq);
        *reinterpret_cast<float4*>(S + kq * ldq<ROWS>() + rr * 4) = st.v[q];
    }
}

// an epilogue that only accumulates declares `static constexpr bool kAtomic = true` and an
// atomic(m, n, v) (dual: atomic(m, n, p, q)) adding into its output
template <class E, class = void>
struct has_atomic : std::false_type {};
template <class E>
struct has_atomic<E, std::void_t<decltype(E::kAtomic)>> : std::integral_constant<bool, E::kAtomic> {};
// an epilogue whose load(m, n) depends on m only (a bias per row) declares
// `static constexpr bool kRowLoad = true`: the block reads its rows' values before the main
// loop, so that their latency is hidden under the products
template <class E, class = void>
struct has_row_load : std::false_type {};
template <class E>
struct has_row_load<E, std::void_t<decltype(E::kRowLoad)>> : std::integral_constant<bool, E::kRowLoad> {};

template <int... U, class F>
__device__ __forceinline__ void unroll_seq(std::integer_sequence<int, U...>, F&& f) {
    (f(std::integral_constant<int, U>{}), ...);
}

// K steps in the order the blocks take them: the partial steps (K % 16 of a segment) first,
// then the segments' whole steps.  DUAL: the segments share K, and so their steps.
template <bool DUAL>
__device__ __forceinline__ int step_count(const Args& g) {
    int n = (g.seg[0].K + KT - 1) / KT;
    if (!DUAL && g.nseg > 1) n += (g.seg[1].K + KT - 1) / KT;
    return n;
}
template <bool DUAL>
__device__ __forceinline__ void step_of(const Args& g, int t, int& s, int& k0) {
    const int p0 = g.seg[0].K % KT != 0, p1 = !DUAL && g.nseg > 1 && g.seg[1].K % KT != 0;
    if (t < p0 + p1) {
        s = t >= p0;
        k0 = g.seg[s].K / KT * KT;
        return;
    }
    const int u = t - p0 - p1, f0 = g.seg[0].K / KT;
    s = !DUAL && u >= f0;
    k0 = (s ? u - f0 : u) * KT;
}

// ------------------------------------------------------------------------------------------
// split-bf16 staging.  A cell is one row's (of A: m; of B: n) eight k values of a step, octet
// o in {0, 1} holding k = 4 o + {0..3} and 8 + 4 o + {0..3} (any order will do that both
// operands share; with this one two lanes read a k-contiguous row's 16 values as two
// 32-byte segments).  In LDS a cell is one 16-byte block per part (h, m, l), at
//   (part * 2 + o) * plane + row * 16:
// a fragment of v_mfma_f32_32x32x16_bf16 (lane: row lane % 32, octet lane / 32) is one 128-bit
// read of consecutive addresses, and the 64 bytes between the planes put the two octets that
// neighbouring lanes of a k-contiguous operand store on different banks.
// ------------------------------------------------------------------------------------------
template <int ROWS>
constexpr int plane_bytes() {
    return ROWS * 16 + 64;
}
template <int ROWS>
constexpr int tile_bytes() {
    return 6 * plane_bytes<ROWS>();
}

// this thread's cell of a ROWS x 16 tile (ROWS = 64: threads 0..127, or, of two such tiles,
// threads 0..127 the first's and 128..255 the second's)
template <bool KMAJ, int ROWS>
__device__ __forceinline__ void my_cell(int& row, int& oct) {
    const int e = threadIdx.x & (2 * ROWS - 1);
    row = KMAJ ? e >> 1 : e & (ROWS - 1);
    oct = KMAJ ? e & 1 : e / ROWS;
}

constexpr int kBufWord3 = 0x00020000;  // gfx9-family buffer resource word 3 (raw, 32-bit data)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t operand_rsrc(const float* P, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(P), (short)0, bytes, kBufWord3);
}

// the cell's byte offset at k step 0; a row past the operand gets an offset past every buffer
// (its loads return zero)
template <bool KMAJ, int ROWS>
__device__ __forceinline__ uint32_t cell_offset(long ld, int r0, int rows) {
    int row, oct;
    my_cell<KMAJ, ROWS>(row, oct);
    if (r0 + row >= rows) return 0x80000000u;
    return (uint32_t)((KMAJ ? (long)(r0 + row) * ld + 4 * oct : (long)(r0 + row) + 4L * oct * ld) * 4);
}

// a whole k step's cell by buffer loads (soff: the step's byte offset; ld4 = ld * 4).  The
// 128-bit loads need 4-byte alignment only.
template <bool KMAJ>
__device__ __forceinline__ void load_cell(float (&v)[8], __amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff, uint32_t ld4) {
    if constexpr (KMAJ) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const v4f x = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff + 32u * b, 0));
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * b + i] = x[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff + ld4 * (uint32_t)(i < 4 ? i : i + 4), 0));
    }
}

// the same for a step that K cuts short: element by element, zero past the operand
template <bool KMAJ, int ROWS>
__device__ __forceinline__ void load_cell_part(float (&v)[8], const float* __restrict__ P, long ld, int r0, int rows, int k0, int K) {
    int row, oct;
    my_cell<KMAJ, ROWS>(row, oct);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int k = k0 + 4 * oct + (i < 4 ? i : i + 4);
        float x = 0.f;
        if (r0 + row < rows && k < K) x = KMAJ ? P[(long)(r0 + row) * ld + k] : P[(long)(r0 + row) + (long)k * ld];
        v[i] = x;
    }
}

template <bool KMAJ, int ROWS>
__device__ __forceinline__ void store_cell(const u32x4 (&c)[3], char* S) {
    int row, oct;
    my_cell<KMAJ, ROWS>(row, oct);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(S + (2 * p + oct) * plane_bytes<ROWS>() + row * 16) = c[p];
}

// DUAL: the two segments share K and their operands are read in the same K steps, giving two
// outputs from three products,
//   P = A0 B0,   Q = A0 B1 + A1 B0,
// (a tangent pair such as s1 = W1 x, s1d = W1 xd + W1d x) with each operand tile loaded once.
// The epilogue then takes both: load(m, n) returns a float2 of old values and
// operator()(m, n, p, q, old) writes.
// LDS bytes of one block: two buffers of the A and B operand tiles (DUAL: two of each)
template <int BNT, bool DUAL>
constexpr int smem_bytes() {
    return 2 * (DUAL ? 2 : 1) * (tile_bytes<BM>() + tile_bytes<BNT>());
}

// The tile again with fp32 matrix instructions (v_mfma_f32_32x32x2_f32), for operands that the
// split cannot hold: one LDS buffer, a step's loads after the step before (such tiles are rare).
// The MFMA's k index (lane / 32) selects the k-plane: MFMA 4 h + c of a step takes
// k = 4 (2 h + lane / 32) + c, the same for both operands.
template <bool A_KM, bool B_KM, int BNT, bool DUAL>
__device__ __forceinline__ void fp32_loop(const Args& g, int m0, int n0, int t_begin, int t_end, float* smem,
                                                    floatx16 (&acc)[DUAL ? 2 : 1][2][BNT / 64]) {
    constexpr int NJ = BNT / 64, LQA = ldq<BM>(), LQB = ldq<BNT>(), NOP = DUAL ? 2 : 1;
    auto As = reinterpret_cast<float(*)[KQ * LQA]>(smem);
    auto Bs = reinterpret_cast<float(*)[KQ * LQB]>(smem + NOP * KQ * LQA);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * (BNT / 2);
#pragma unroll
    for (int o = 0; o < NOP; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[o][i][j][r] = 0.f;
    for (int t = t_begin; t < t_end; ++t) {
        int s, k0;
        step_of<DUAL>(g, t, s, k0);
        __syncthreads();
#pragma unroll
        for (int o = 0; o < NOP; ++o) {
            const Seg& sg = g.seg[DUAL ? o : s];
            Stage<BM> sa;
            Stage<BNT> sb;
            load_tile<A_KM, BM>(sa, sg.A, sg.lda, g.M, sg.K, m0, k0);
            load_tile<B_KM, BNT>(sb, sg.B, sg.ldb, g.N, sg.K, n0, k0);
            store_tile<A_KM, BM>(sa, As[o]);
            store_tile<B_KM, BNT>(sb, Bs[o]);
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < KT / 8; ++h) {
            const int kq = 2 * h + (lane >> 5);
            v4f fa[NOP][2], fb[NOP][NJ];
#pragma unroll
            for (int o = 0; o < NOP; ++o) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    fa[o][i] = *reinterpret_cast<const v4f*>(As[o] + kq * LQA + (wm + i * 32 + (lane & 31)) * 4);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    fb[o][j] = *reinterpret_cast<const v4f*>(Bs[o] + kq * LQB + (wn + j * 32 + (lane & 31)) * 4);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        acc[0][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[0][j][c], fa[0][i][c], acc[0][i][j], 0, 0, 0);
                        if constexpr (DUAL) {
                            acc[1][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[1][j][c], fa[0][i][c], acc[1][i][j], 0, 0, 0);
                            acc[1][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[0][j][c], fa[1][i][c], acc[1][i][j], 0, 0, 0);
                        }
                    }
        }
    }
}

// One block of the product: the tile at (bx, by) of slice bz, with its LDS at smem.
template <bool A_KM, bool B_KM, int BNT, class Epi, bool DUAL>
__device__ __forceinline__ void gemm_block(const Args& g, const Epi& epi, int bx, int by, int bz, float* smem) {
    constexpr int NJ = BNT / 64;
    constexpr int NOP = DUAL ? 2 : 1;  // operand pairs staged per step
    static_assert(!DUAL || BNT == 64, "a dual block stages its two 64-row B tiles with half its threads each");
    constexpr int TA = tile_bytes<BM>(), TB = tile_bytes<BNT>(), PA = plane_bytes<BM>(), PB = plane_bytes<BNT>();
    char* const lds = reinterpret_cast<char*>(smem);
    // buffer b: A tiles at lds + b * BUF + o * TA, then the B tiles
    constexpr int BUF = NOP * (TA + TB);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 7);  // of the block's threads
    const int m0 = bx * BM, n0 = by * BNT;
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * (BNT / 2);

    // the K steps of all segments (DUAL: of the shared K), partial ones first; this block's slice
    const bool two = g.nseg > 1;
    const int total = step_count<DUAL>(g);
    const int t_begin = (int)((long)total * bz / g.ksplit);
    const int t_end = (int)((long)total * (bz + 1) / g.ksplit);
    const int npart = (g.seg[0].K % KT != 0) + (!DUAL && two && g.seg[1].K % KT != 0);
    const int full0 = g.seg[0].K / KT;
    // Both segments' operands in registers (indexing g.seg[s] with a runtime s would reload
    // them from the kernel-argument segment at every step).  A slice without a whole step (a
    // short K) loads none: its whole-step loads all fall past the buffers and return zero.
    const bool whole = t_end > npart;
    const long lda0 = whole ? g.seg[0].lda : 0, ldb0 = whole ? g.seg[0].ldb : 0;
    const long lda1 = whole && two ? g.seg[1].lda : lda0, ldb1 = whole && two ? g.seg[1].ldb : ldb0;
    const __amdgpu_buffer_rsrc_t rA0 = operand_rsrc(g.seg[0].A, g.abytes[0]), rA1 = operand_rsrc(g.seg[two].A, g.abytes[two]);
    const __amdgpu_buffer_rsrc_t rB0 = operand_rsrc(g.seg[0].B, g.bbytes[0]), rB1 = operand_rsrc(g.seg[two].B, g.bbytes[two]);
    const int ma = whole ? g.M : 0, nb = whole ? g.N : 0;
    const uint32_t oA0 = cell_offset<A_KM, BM>(lda0, m0, ma), oA1 = cell_offset<A_KM, BM>(lda1, m0, ma);
    const uint32_t oB0 = cell_offset<B_KM, BNT>(ldb0, n0, nb), oB1 = cell_offset<B_KM, BNT>(ldb1, n0, nb);

    floatx16 acc[NOP][2][NJ];  // DUAL: [0] P, [1] Q
#pragma unroll
    for (int o = 0; o < NOP; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[o][i][j][r] = 0.f;
    // the epilogue's per-row values, read now when they depend on the row only (kRowLoad)
    using Pre = decltype(epi.load(0, 0));
    Pre prow[2] = {};
    if constexpr (has_row_load<Epi>::value) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int m = m0 + wm + i * 32 + (lane & 31);
            if (m < g.M) prow[i] = epi.load(m, 0);
        }
    }
    u16x2 tiny = {0xffff, 0xffff};

    // one register stage of a cell per operand: a step's loads are issued a step before it is
    // split and stored.  Loads and stores are unconditional (a step past the slice reloads a
    // whole step inside the buffers' extents; its data is never multiplied).
    float va[NOP][8], vb[8];
    // a whole step t >= npart
    auto load = [&](int t) {
        const int u = max(min(t, t_end - 1) - npart, 0);
        if constexpr (DUAL) {
            const uint32_t sa = (uint32_t)((A_KM ? (long)u * KT : (long)u * KT * lda0) * 4);
            load_cell<A_KM>(va[0], rA0, oA0, sa, (uint32_t)(lda0 * 4));
            const uint32_t sa1 = (uint32_t)((A_KM ? (long)u * KT : (long)u * KT * lda1) * 4);
            load_cell<A_KM>(va[NOP - 1], rA1, oA1, sa1, (uint32_t)(lda1 * 4));
            const long ldb = half ? ldb1 : ldb0;
            const uint32_t sb = (uint32_t)((B_KM ? (long)u * KT : (long)u * KT * ldb) * 4);
            load_cell<B_KM>(vb, half ? rB1 : rB0, half ? oB1 : oB0, sb, (uint32_t)(ldb * 4));
        } else {
            const bool s1 = u >= full0;
            const long k0 = (long)(s1 ? u - full0 : u) * KT;
            const long lda = s1 ? lda1 : lda0, ldb = s1 ? ldb1 : ldb0;
            load_cell<A_KM>(va[0], s1 ? rA1 : rA0, s1 ? oA1 : oA0, (uint32_t)((A_KM ? k0 : k0 * lda) * 4), (uint32_t)(lda * 4));
            load_cell<B_KM>(vb, s1 ? rB1 : rB0, s1 ? oB1 : oB0, (uint32_t)((B_KM ? k0 : k0 * ldb) * 4), (uint32_t)(ldb * 4));
        }
    };
    // any step, in the prologue
    auto load_any = [&](int t) {
        if (t < npart && t < t_end) {
            int s, k0;
            step_of<DUAL>(g, t, s, k0);
#pragma unroll
            for (int o = 0; o < NOP; ++o) {
                const Seg& sg = g.seg[DUAL ? o : s];
                load_cell_part<A_KM, BM>(va[o], sg.A, sg.lda, m0, g.M, k0, sg.K);
            }
            const Seg& sg = g.seg[DUAL ? half : s];
            load_cell_part<B_KM, BNT>(vb, sg.B, sg.ldb, n0, g.N, k0, sg.K);
        } else {
            load(t);
        }
    };
    auto store = [&](int buf) {
        char* const S = lds + buf * BUF;
        u32x4 c[3];
#pragma unroll
        for (int o = 0; o < NOP; ++o) {
            split8(va[o], c, tiny);
            store_cell<A_KM, BM>(c, S + o * TA);
        }
        if (BNT == 128 || DUAL || half == 0) {
            split8(vb, c, tiny);
            store_cell<B_KM, BNT>(c, S + NOP * TA + (DUAL ? half * TB : 0));
        }
    };
    bf16x8 fa[NOP][2][3], fb[NOP][NJ][3];  // [operand][tile][part]
    auto read_frags = [&](int buf) {
        const char* const S = lds + buf * BUF;
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
            for (int o = 0; o < NOP; ++o) {
                const int pl = 2 * q + (lane >> 5);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    fa[o][i][q] = *reinterpret_cast<const bf16x8*>(S + o * TA + pl * PA + (wm + i * 32 + (lane & 31)) * 16);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    fb[o][j][q] = *reinterpret_cast<const bf16x8*>(S + NOP * TA + o * TB + pl * PB + (wn + j * 32 + (lane & 31)) * 16);
            }
    };
    // a tile edge block skips the MFMAs of its 32 x 32 tiles that lie wholly past M or N
    // (wave-uniform tests, compile-time true in whole blocks); those accumulators stay zero and
    // are never stored
    const bool li = m0 + wm + 32 < g.M, lj = n0 + wn + 32 < g.N, l0 = m0 + wm < g.M && n0 + wn < g.N;
    auto mma = [&](auto whole_tag) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
        if (!WHOLE && !l0) return;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (!WHOLE && i && !li) continue;
            floatx16 v[NOP][NJ];
#pragma unroll
            for (int o = 0; o < NOP; ++o)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) v[o][j][r] = 0.f;
#pragma unroll
            for (int x = 0; x < 6; ++x)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    if (!WHOLE && j && !lj) continue;
                    if constexpr (DUAL) v[1][j] = mfma_bf16(fb[1][j][kSplitB[x]], fa[0][i][kSplitA[x]], v[1][j]);
                    v[0][j] = mfma_bf16(fb[0][j][kSplitB[x]], fa[0][i][kSplitA[x]], v[0][j]);
                    if constexpr (DUAL) v[1][j] = mfma_bf16(fb[0][j][kSplitB[x]], fa[1][i][kSplitA[x]], v[1][j]);
                }
#pragma unroll
            for (int o = 0; o < NOP; ++o)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[o][i][j][r] += v[o][j][r];
        }
    };
    // step t (buffer p): its fragments from LDS, step t + 1 split and stored to the other
    // buffer, step t + 2's loads, t's MFMAs
    auto mainloop = [&](auto whole_tag) {
        auto step = [&](int t, int p) {
            read_frags(p);
            store(p ^ 1);
            load(t + 2);
            mma(whole_tag);
            __syncthreads();
        };
        for (int t = t_begin; t < t_end; t += 2) {
            step(t, 0);
            if (t + 1 < t_end) step(t + 1, 1);
        }
    };
    bool redo = !g.bufok;
    if (t_begin < t_end && g.bufok) {
        // partial steps are only t < npart <= 2: t_begin and t_begin + 1
        load_any(t_begin);
        store(0);
        load_any(t_begin + 1);
        __syncthreads();
        if (m0 + BM <= g.M && n0 + BNT <= g.N) mainloop(std::true_type{});
        else mainloop(std::false_type{});
        // a non-finite sum, or an element that the split cannot hold
        float z = 0.f;
#pragma unroll
        for (int o = 0; o < NOP; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) z = __builtin_fmaf(acc[o][i][j][r], 0.f, z);
        redo = z != 0.f || any_tiny(tiny);
    }
    if (__syncthreads_or(redo)) fp32_loop<A_KM, B_KM, BNT, DUAL>(g, m0, n0, t_begin, t_end, smem, acc);
    // accumulator (i, j, r): m = m0 + wm + 32 i + lane % 32,  n = n0 + wn + 32 j + 8 (r / 4) + 4 (lane / 32) + r % 4
    if constexpr (has_atomic<Epi>::value) {
        if (g.ksplit > 1 && g.atomic) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int m = m0 + wm + i * 32 + (lane & 31);
                if (m >= g.M) continue;
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int n = n0 + wn + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                        if (n < g.N) {
                            if constexpr (DUAL)
                                epi.atomic(m, n, acc[0][i][j][r], acc[NOP - 1][i][j][r]);
                            else
                                epi.atomic(m, n, acc[0][i][j][r]);
                        }
                    }
            }
            return;
        }
    }
    if (g.ksplit > 1) {
        // slice z at part + z * NOP * M * N (DUAL: P then Q)
        const long mn = (long)g.M * g.N;
        float* part = g.part + (long)bz * NOP * mn;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int m = m0 + wm + i * 32 + (lane & 31);
            if (m >= g.M) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int n = n0 + wn + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                    if (n < g.N) {
#pragma unroll
                        for (int o = 0; o < NOP; ++o) part[o * mn + m + (long)n * g.M] = acc[o][i][j][r];
                    }
                }
        }
        return;
    }
    // the epilogue's inputs (e.g. C of C += v) for the whole tile first, then the stores: the
    // output may alias them as far as the compiler knows, and interleaving would serialise one
    // memory round trip per element
    Pre pre[2][NJ][16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm + i * 32 + (lane & 31);
                const int n = n0 + wn + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if constexpr (has_row_load<Epi>::value)
                    pre[i][j][r] = prow[i];
                else
                    pre[i][j][r] = (m < g.M && n < g.N) ? epi.load(m, n) : Pre{};
            }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = m0 + wm + i * 32 + (lane & 31);
        if (m >= g.M) continue;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int n = n0 + wn + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (n < g.N) {
                    if constexpr (DUAL)
                        epi(m, n, acc[0][i][j][r], acc[NOP - 1][i][j][r], pre[i][j][r]);
                    else
                        epi(m, n, acc[0][i][j][r], pre[i][j][r]);
                }
            }
    }
}

template <bool A_KM, bool B_KM, int BNT, class Epi, bool DUAL = false>
__global__ __launch_bounds__(NT, 2) void gemm_kernel(Args g, Epi epi) {
    __shared__ __attribute__((aligned(16))) float smem[smem_bytes<BNT, DUAL>() / 4];
    gemm_block<A_KM, B_KM, BNT, Epi, DUAL>(g, epi, blockIdx.x, blockIdx.y, blockIdx.z, smem);
}

// Two products in one launch, each block one tile of one of them: blocks [0, nblocks(P0))
// are P0's (m tiles fastest, then n tiles, then K slices), the rest P1's.  Neither may need a
// second kernel (a K split adds by atomics).  The two share the CUs, so the tail of one is
// filled by blocks of the other.
template <bool A_KM, bool B_KM, class Epi>
struct Part {
    Args g;
    Epi epi;
    int gx, gy;  // tile grid: m tiles, n tiles (slices: g.ksplit)
};
//
// X: independent work that rides along as x.count extra blocks at the front of the grid, each
// calling x(block, smem) with NT threads and at least 1088 floats of LDS (NoExtra: none).
struct NoExtra {
    int count = 0;
    __device__ __forceinline__ void operator()(int, float*) const {}
};
template <class X>
__global__ __launch_bounds__(NT) void extra_kernel(X x) {
    __shared__ __attribute__((aligned(16))) float smem[1088];
    x(blockIdx.x, smem);
}
template <int BNT, bool DUAL, bool A0, bool B0, class E0, bool A1, bool B1, class E1, class X>
__global__ __launch_bounds__(NT, 2) void gemm_pair_kernel(Part<A0, B0, E0> p0, Part<A1, B1, E1> p1, X x) {
    static_assert(smem_bytes<BNT, DUAL>() >= 4 * 1088, "the extra blocks' LDS");
    __shared__ __attribute__((aligned(16))) float smem[smem_bytes<BNT, DUAL>() / 4];
    const int n0 = p0.gx * p0.gy * p0.g.ksplit;
    int b = blockIdx.x;
    if (b < x.count) {
        x(b, smem);
        return;
    }
    b -= x.count;
    if (b < n0) {
        const int per = p0.gx * p0.gy, r = b % per;
        gemm_block<A0, B0, BNT, E0, DUAL>(p0.g, p0.epi, r % p0.gx, r / p0.gx, b / per, smem);
    } else {
        b -= n0;
        const int per = p1.gx * p1.gy, r = b % per;
        gemm_block<A1, B1, BNT, E1, DUAL>(p1.g, p1.epi, r % p1.gx, r / p1.gx, b / per, smem);
    }
}

// second stage of a split-K product: C(m, n) = sum over slices in order, then the epilogue
// (DUAL: P and Q, each summed in slice order)
template <class Epi, bool DUAL = false>
__global__ __launch_bounds__(NT) void splitk_reduce_kernel(const float* __restrict__ part, int ksplit, int M, int N, Epi epi) {
    constexpr int NOP = DUAL ? 2 : 1;
    const long q = (long)blockIdx.x * NT + threadIdx.x;
    const long mn = (long)M * N;
    if (q >= mn) return;
    // every slice's value in flight at once (ksplit <= 16; indices past the last slice clamped
    // to it and never added), added in slice order
    const int m = (int)(q % M), n = (int)(q / M);
    float v[NOP][16];
#pragma unroll
    for (int o = 0; o < NOP; ++o)
#pragma unroll
        for (int z = 0; z < 16; ++z) v[o][z] = part[(long)min(z, ksplit - 1) * NOP * mn + o * mn + q];
    const auto old = epi.load(m, n);
    __builtin_amdgcn_sched_barrier(0);
    float s[NOP];
#pragma unroll
    for (int o = 0; o < NOP; ++o) {
        s[o] = v[o][0];
#pragma unroll
        for (int z = 1; z < 16; ++z)
            if (z < ksplit) s[o] += v[o][z];
    }
    if constexpr (DUAL)
        epi(m, n, s[0], s[NOP - 1], old);
    else
        epi(m, n, s[0], old);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Tile width and K split for an M x N x K product on `cus` compute units, from a cost model
// in microseconds: the CU with the most blocks sets the time: blocks per CU x K steps per block
// x the time of one block step with two blocks resident (128 x 128 x 16: 0.75 us, 128 x 64 x 16:
// 0.48, a dual 128 x 64 x 16: 1.2, measured on MI355X at K = 784..3920), longer by a half when
// the CU has one block only (one wave per SIMD: the splitting and the MFMAs of a wave do not
// overlap).  A K split costs its partial tiles' round trip through memory (8 bytes per element
// and slice at about 5 TB/s) plus the reduction launch, or, by atomics, their atomic traffic (4
// bytes per element and slice, overlapped with the other blocks' work: about 10 TB/s of issue).
// Every K slice keeps at least 8 steps.  Ties go to the narrow tile and the smaller split.
struct Plan {
    int bnt, ksplit;
    bool atomic;  // the slices are added into the output by atomics (an accumulate epilogue)
    double us;    // the model's time
};
// nout = 2 plans a dual product (three products per step over shared loads, two outputs; its
// tile is the narrow one).  atomic_ok: the epilogue only accumulates, so a split may add its
// slices by atomics (no partial tiles, no reduction launch).  bnt_only: 0, or the one tile
// width to consider.
inline Plan plan(int M, int N, int Ktot, int cus, int nout = 1, bool atomic_ok = false, int bnt_only = 0) {
    const long mt = (M + BM - 1) / BM;
    const long steps = (Ktot + KT - 1) / KT;
    Plan best{64, 1, false, 0.0};
    for (int bnt = 64; bnt <= (nout == 2 ? 64 : 128); bnt *= 2) {
        if (bnt_only && bnt != bnt_only) continue;
        const double step_us = nout == 2 ? 1.2 : bnt == 64 ? 0.48 : 0.75;
        const long tiles = mt * ((N + bnt - 1) / bnt);
        for (int ks = 1; ks <= 16; ++ks) {
            if (ks > 1 && steps / ks < 8) break;
            const long per_cu = (tiles * ks + cus - 1) / cus;
            const long st = (steps + ks - 1) / ks;
            // an atomic split is kept to two rounds of resident blocks (two per CU)
            if (atomic_ok && ks > 1 && per_cu > 4) break;
            double cost = (double)per_cu * st * step_us * (per_cu < 2 ? 1.5 : 1.0);
            if (ks > 1) cost += atomic_ok ? 4.0 * ks * nout * (double)M * N / 1e7 : 8.0 * ks * nout * (double)M * N / 5e6 + 3.0;
            if (cost < best.us || best.us == 0.0) best = Plan{bnt, ks, atomic_ok && ks > 1, cost};
        }
    }
    return best;
}

// Number of compute units of the current device (cached per process for device 0..15).
inline int device_cus() {
    static int cached[16] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
    if (!cached[dev]) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        cached[dev] = cus;
    }
    return cached[dev];
}

// the launch-time fields of g (split, atomic, byte extents)
template <bool A_KM, bool B_KM, class Epi, bool DUAL>
hipError_t prepare(Args& g, const Plan& p) {
    if (DUAL && (g.nseg != 2 || g.seg[0].K != g.seg[1].K)) return hipErrorInvalidValue;
    g.ksplit = p.ksplit;
    g.atomic = p.atomic && has_atomic<Epi>::value;
    if (p.ksplit > 1 && !g.atomic && !g.part) return hipErrorInvalidValue;
    // byte extent of each operand: A spans K columns of lda (A_KM = false) or M columns,
    // B spans N columns of ldb (B_KM = true) or K columns; the last column ends with its rows
    g.bufok = true;
    auto extent = [&](bool km, long ld, int rows, int K) -> uint32_t {
        const double e = K <= 0 ? 0.0 : 4.0 * (km ? (double)ld * (rows - 1) + K : (double)ld * (K - 1) + rows);
        g.bufok = g.bufok && e < 2147483648.0;
        return g.bufok ? (uint32_t)e : 0u;
    };
    for (int s = 0; s < g.nseg; ++s) {
        g.abytes[s] = extent(A_KM, g.seg[s].lda, g.M, g.seg[s].K);
        g.bbytes[s] = extent(B_KM, g.seg[s].ldb, g.N, g.seg[s].K);
    }
    return hipSuccess;
}

// Launch; returns the hipError of the launch.  `part` must hold ksplit * M * N floats (DUAL:
// twice that) when the plan splits K (ask with plan() first); it may be null otherwise.  A
// dual product takes two segments of the same K.
template <bool A_KM, bool B_KM, class Epi, bool DUAL = false>
hipError_t launch(Args g, Epi epi, hipStream_t stream, const Plan& p) {
    if (g.M <= 0 || g.N <= 0) return hipSuccess;
    if (hipError_t e = prepare<A_KM, B_KM, Epi, DUAL>(g, p)) return e;
    const dim3 grid((g.M + BM - 1) / BM, (g.N + p.bnt - 1) / p.bnt, p.ksplit);
    if constexpr (DUAL) {
        gemm_kernel<A_KM, B_KM, 64, Epi, true><<<grid, NT, 0, stream>>>(g, epi);
    } else {
        if (p.bnt == 128) gemm_kernel<A_KM, B_KM, 128, Epi><<<grid, NT, 0, stream>>>(g, epi);
        else gemm_kernel<A_KM, B_KM, 64, Epi><<<grid, NT, 0, stream>>>(g, epi);
    }
    if (p.ksplit > 1 && !g.atomic) {
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const long mn = (long)g.M * g.N;
        splitk_reduce_kernel<Epi, DUAL><<<(unsigned)((mn + NT - 1) / NT), NT, 0, stream>>>(g.part, p.ksplit, g.M, g.N, epi);
    }
    return hipGetLastError();
}

// Two products as one launch (gemm_pair_kernel) when both plans use one tile width and neither
// needs a second kernel; otherwise one launch each.  Both are enqueued on `stream`.
template <bool A0, bool B0, class E0, bool A1, bool B1, class E1, bool DUAL = false, class X = NoExtra>
hipError_t launch_pair(Args g0, E0 e0, const Plan& p0, Args g1, E1 e1, const Plan& p1, hipStream_t stream, X x = X{}) {
    const bool one0 = p0.ksplit == 1 || (p0.atomic && has_atomic<E0>::value);
    const bool one1 = p1.ksplit == 1 || (p1.atomic && has_atomic<E1>::value);
    if (g0.M <= 0 || g0.N <= 0 || g1.M <= 0 || g1.N <= 0 || p0.bnt != p1.bnt || !one0 || !one1) {
        if (x.count > 0) {
            extra_kernel<X><<<(unsigned)x.count, NT, 0, stream>>>(x);
            if (hipError_t e = hipGetLastError()) return e;
        }
        if (hipError_t e = launch<A0, B0, E0, DUAL>(g0, e0, stream, p0)) return e;
        return launch<A1, B1, E1, DUAL>(g1, e1, stream, p1);
    }
    Part<A0, B0, E0> q0{g0, e0, (g0.M + BM - 1) / BM, (g0.N + p0.bnt - 1) / p0.bnt};
    Part<A1, B1, E1> q1{g1, e1, (g1.M + BM - 1) / BM, (g1.N + p1.bnt - 1) / p1.bnt};
    if (hipError_t e = prepare<A0, B0, E0, DUAL>(q0.g, p0)) return e;
    if (hipError_t e = prepare<A1, B1, E1, DUAL>(q1.g, p1)) return e;
    const long nb = (long)x.count + (long)q0.gx * q0.gy * p0.ksplit + (long)q1.gx * q1.gy * p1.ksplit;
    if constexpr (DUAL) {
        gemm_pair_kernel<64, true, A0, B0, E0, A1, B1, E1, X><<<(unsigned)nb, NT, 0, stream>>>(q0, q1, x);
    } else {
        if (p0.bnt == 128) gemm_pair_kernel<128, false, A0, B0, E0, A1, B1, E1, X><<<(unsigned)nb, NT, 0, stream>>>(q0, q1, x);
        else gemm_pair_kernel<64, false, A0, B0, E0, A1, B1, E1, X><<<(unsigned)nb, NT, 0, stream>>>(q0, q1, x);
    }
    return hipGetLastError();
}

}  // namespace gemm
}  // namespace stade
