// The fp32 GEMM of gemm_f32.hpp by split bf16 (split_bf16.hpp), for pairs of large products that
// accumulate into their outputs: six bf16 products of operands split into three bf16 parts.  A
// step's products are summed from zero and then added to the tile's total: one rounding at the
// total's size per 16 k, where v_mfma_f32_32x32x2_f32 rounds every 2 k (and where the six
// products accumulated straight into the total would round six times).  Against 64 bits (N(0, 1)
// times U(0, 1) operands) the normwise error is 1.4e-7 at K = 784 and 3.1e-7 at K = 4096; of
// v_mfma_f32_32x32x2_f32 5.0e-7 and 1.1e-6, accumulated straight 4.0e-7 and 9.9e-7.
// The matrix cores run bf16 at 16 times the fp32 rate, so six products leave a factor of 2.7.
// Measured with fp32 MFMAs -> split, the evaluations that hold the pair (batch 4096, 784 x 1024):
// MLP adjoint 208 -> 179 us, HVP (dual products) 595 -> 479; HVP of 1000 x 500 x 700 168 -> 160.
// What bounds the loop is the splitting (12 vector instructions a pair of elements, 96 a
// wave and step beside 24 MFMAs) and the loads and barriers that a block's two waves a SIMD do not
// hide wholly: without the splitting and the loads the same loop runs at 270 TFLOP/s, with them
// at 165-180.
// A block that meets an element the split cannot hold forms its tile again with fp32 matrix
// instructions (fp32_loop): the results there are those of plain fp32.
//
// Tiling as in gemm_f32.hpp: a 256-thread block (4 waves) computes a 128 x BNT tile of C (BNT =
// 128 or 64), each wave a 64 x BNT/2 part as 2 x BNT/64 MFMA 32 x 32 tiles.  K advances 16 at a
// time through two LDS buffers: while a step's MFMAs run from one, the next step is split and
// stored to the other and the step after that is being loaded; one barrier a step, and two blocks
// a CU, so that one block's splitting overlaps the other's MFMAs.  A partial K step (K % 16)
// comes first, in the prologue, so that the steps of the loop load without tests.
#pragma once

#include "gemm_f32.hpp"
#include "split_bf16.hpp"

namespace stade {
namespace gemm {

// a product's operands with their byte extents (set by prepare_split)
struct SplitArgs {
    Args g;
    uint32_t abytes[2], bbytes[2];
};

// K steps in the order the blocks take them: the partial step first.  (A dual product's segments
// share K.)
__device__ __forceinline__ int step_k(int K, int t) {
    const int part = K % KT != 0;
    return t < part ? K / KT * KT : (t - part) * KT;
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

__device__ __forceinline__ __amdgpu_buffer_rsrc_t split_rsrc(const float* P, uint32_t bytes) {
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
// 128-bit loads need 4-byte alignment only.  The scalar offset never passes the buffer's end: the
// range check compares the lane's offset with what the scalar one leaves of the buffer, and that
// difference must not wrap (a buffer may be shorter than a step: then nothing but the lanes'
// offsets past every buffer is loaded, at scalar offset 0).
template <bool KMAJ>
__device__ __forceinline__ void load_cell(float (&v)[8], __amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff, uint32_t ld4) {
    if constexpr (KMAJ) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const v4f x = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, off + 32u * b, soff, 0));
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
        const int k0 = step_k(g.seg[0].K, t);
        __syncthreads();
#pragma unroll
        for (int o = 0; o < NOP; ++o) {
            const Seg& sg = g.seg[o];
            Stage<BM> sa;
            Stage<BNT> sb;
            load_tile<A_KM, BM>(sa, sg.A, sg.lda, g.M, sg.K, m0, k0, false);
            load_tile<B_KM, BNT>(sb, sg.B, sg.ldb, g.N, sg.K, n0, k0, false);
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

// One block of the product: the tile at (bx, by) of slice bz, with its LDS at smem.  The epilogue
// accumulates into its output, by atomics where K is split.
template <bool A_KM, bool B_KM, int BNT, class Epi, bool DUAL>
__device__ __forceinline__ void split_block(const SplitArgs& q, const Epi& epi, int bx, int by, int bz, float* smem) {
    const Args& g = q.g;
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

    const int K = g.seg[0].K, npart = K % KT != 0, total = (K + KT - 1) / KT;
    const int t_begin = (int)((long)total * bz / g.ksplit);
    const int t_end = (int)((long)total * (bz + 1) / g.ksplit);
    // A slice without a whole step (a short K) loads none: its whole-step loads all fall past
    // the buffers and return zero.
    const bool whole = t_end > npart;
    const long lda0 = whole ? g.seg[0].lda : 0, ldb0 = whole ? g.seg[0].ldb : 0;
    const long lda1 = whole && DUAL ? g.seg[1].lda : lda0, ldb1 = whole && DUAL ? g.seg[1].ldb : ldb0;
    const __amdgpu_buffer_rsrc_t rA0 = split_rsrc(g.seg[0].A, q.abytes[0]), rA1 = split_rsrc(g.seg[NOP - 1].A, q.abytes[NOP - 1]);
    const __amdgpu_buffer_rsrc_t rB0 = split_rsrc(g.seg[0].B, q.bbytes[0]), rB1 = split_rsrc(g.seg[NOP - 1].B, q.bbytes[NOP - 1]);
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
    uint32_t lost = 0;

    // one register stage of a cell per operand: a step's loads are issued a step before it is
    // split and stored.  Loads and stores are unconditional (a step past the slice reloads a
    // whole step inside the buffers' extents; its data is never multiplied).
    float va[NOP][8], vb[8];
    // a whole step t >= npart
    auto load = [&](int t) {
        const int u = max(min(t, t_end - 1) - npart, 0);
        auto at = [&](bool km, long ld) { return (uint32_t)((km ? (long)u * KT : (long)u * KT * ld) * 4); };
        load_cell<A_KM>(va[0], rA0, oA0, at(A_KM, lda0), (uint32_t)(lda0 * 4));
        if constexpr (DUAL) {
            load_cell<A_KM>(va[NOP - 1], rA1, oA1, at(A_KM, lda1), (uint32_t)(lda1 * 4));
            const long ldb = half ? ldb1 : ldb0;
            load_cell<B_KM>(vb, half ? rB1 : rB0, half ? oB1 : oB0, at(B_KM, ldb), (uint32_t)(ldb * 4));
        } else {
            load_cell<B_KM>(vb, rB0, oB0, at(B_KM, ldb0), (uint32_t)(ldb0 * 4));
        }
    };
    // any step, in the prologue
    auto load_any = [&](int t) {
        if (t < npart && t < t_end) {
            const int k0 = step_k(K, t);
#pragma unroll
            for (int o = 0; o < NOP; ++o) load_cell_part<A_KM, BM>(va[o], g.seg[o].A, g.seg[o].lda, m0, g.M, k0, K);
            const Seg& sg = g.seg[DUAL ? half : 0];
            load_cell_part<B_KM, BNT>(vb, sg.B, sg.ldb, n0, g.N, k0, K);
        } else {
            load(t);
        }
    };
    auto store = [&](int buf) {
        char* const S = lds + buf * BUF;
        u32x4 c[3];
#pragma unroll
        for (int o = 0; o < NOP; ++o) {
            split8(va[o], c, lost);
            store_cell<A_KM, BM>(c, S + o * TA);
        }
        if (BNT == 128 || DUAL || half == 0) {
            split8(vb, c, lost);
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
    bool redo = false;
    if (t_begin < t_end) {
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
        redo = z != 0.f || any_lost(lost);
    }
    if (__syncthreads_or(redo)) fp32_loop<A_KM, B_KM, BNT, DUAL>(g, m0, n0, t_begin, t_end, smem, acc);
    // accumulator (i, j, r): m = m0 + wm + 32 i + lane % 32,  n = n0 + wn + 32 j + 8 (r / 4) + 4 (lane / 32) + r % 4
    auto each = [&](auto&& f) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int m = m0 + wm + i * 32 + (lane & 31);
            if (m >= g.M) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int n = n0 + wn + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                    if (n < g.N) f(i, j, r, m, n);
                }
        }
    };
    if (g.ksplit > 1) {
        each([&](int i, int j, int r, int m, int n) {
            if constexpr (DUAL) epi.atomic(m, n, acc[0][i][j][r], acc[1][i][j][r]);
            else epi.atomic(m, n, acc[0][i][j][r]);
        });
        return;
    }
    // the old values of the whole tile first, then the stores: the output may alias them as far
    // as the compiler knows, and interleaving would serialise one memory round trip per element
    decltype(epi.load(0, 0)) pre[2][NJ][16];
    each([&](int i, int j, int r, int m, int n) { pre[i][j][r] = epi.load(m, n); });
    each([&](int i, int j, int r, int m, int n) {
        if constexpr (DUAL) epi(m, n, acc[0][i][j][r], acc[1][i][j][r], pre[i][j][r]);
        else epi(m, n, acc[0][i][j][r], pre[i][j][r]);
    });
}

// Two products in one launch, as gemm_pair_kernel
template <bool A_KM, bool B_KM, class Epi>
struct SplitPart {
    SplitArgs q;
    Epi epi;
    int gx, gy;  // tile grid: m tiles, n tiles (slices: q.g.ksplit)
};
template <int BNT, bool DUAL, bool A0, bool B0, class E0, bool A1, bool B1, class E1, class X>
__global__ __launch_bounds__(NT, 2) void split_pair_kernel(SplitPart<A0, B0, E0> p0, SplitPart<A1, B1, E1> p1, X x) {
    static_assert(smem_bytes<BNT, DUAL>() >= 4 * 1088, "the extra blocks' LDS");
    __shared__ __attribute__((aligned(16))) float smem[smem_bytes<BNT, DUAL>() / 4];
    const int n0 = p0.gx * p0.gy * p0.q.g.ksplit;
    int b = blockIdx.x;
    if (b < x.count) {
        x(b, smem);
        return;
    }
    b -= x.count;
    if (b < n0) {
        const int per = p0.gx * p0.gy, r = b % per;
        split_block<A0, B0, BNT, E0, DUAL>(p0.q, p0.epi, r % p0.gx, r / p0.gx, b / per, smem);
    } else {
        b -= n0;
        const int per = p1.gx * p1.gy, r = b % per;
        split_block<A1, B1, BNT, E1, DUAL>(p1.q, p1.epi, r % p1.gx, r / p1.gx, b / per, smem);
    }
}

// K split of an M x N x K product by 128 x bnt tiles on `cus` compute units, from a cost model
// in microseconds: the CU with the most blocks sets the time: blocks per CU x K steps per block
// x the time of one block step with two blocks resident (128 x 128 x 16: 0.75 us, 128 x 64 x 16:
// 0.48, a dual 128 x 64 x 16: 1.2, measured on MI355X at K = 784..3920), longer by a half when
// the CU has one block only (one wave per SIMD: the splitting and the MFMAs of a wave do not
// overlap).  A K split costs its atomic traffic (4 bytes per element and slice, overlapped with
// the other blocks' work: about 10 TB/s of issue).  Every K slice keeps at least 8 steps.
// nout = 2 plans a dual product (three products per step over shared loads, two outputs; its tile is
// the narrow one).  The two products of a pair take one tile width (bnt).
inline Plan plan_split(int M, int N, int Ktot, int cus, int nout, int bnt) {
    const long mt = (M + BM - 1) / BM;
    const long steps = (Ktot + KT - 1) / KT;
    const double step_us = nout == 2 ? 1.2 : bnt == 64 ? 0.48 : 0.75;
    const long tiles = mt * ((N + bnt - 1) / bnt);
    Plan best{bnt, 1, false, 0.0};
    for (int ks = 1; ks <= 16; ++ks) {
        if (ks > 1 && steps / ks < 8) break;
        const long per_cu = (tiles * ks + cus - 1) / cus;
        const long st = (steps + ks - 1) / ks;
        // a split is kept to two rounds of resident blocks (two per CU)
        if (ks > 1 && per_cu > 4) break;
        double cost = (double)per_cu * st * step_us * (per_cu < 2 ? 1.5 : 1.0);
        if (ks > 1) cost += 4.0 * ks * nout * (double)M * N / 1e7;
        if (cost < best.us || best.us == 0.0) best = Plan{bnt, ks, ks > 1, cost};
    }
    return best;
}

// the byte extents of q's operands: A spans K columns of lda (A_KM = false) or M columns, B spans N
// columns of ldb (B_KM = true) or K columns; the last column ends with its rows.  Whether they
// all fit 31 bits, as the buffer loads' offsets need
template <bool A_KM, bool B_KM, bool DUAL>
bool split_extents(SplitArgs& q) {
    bool fits = true;
    auto extent = [&](bool km, long ld, int rows, int K) -> uint32_t {
        const double e = K <= 0 ? 0.0 : 4.0 * (km ? (double)ld * (rows - 1) + K : (double)ld * (K - 1) + rows);
        fits = fits && e < 2147483648.0;
        return fits ? (uint32_t)e : 0u;
    };
    for (int s = 0; s < (DUAL ? 2 : 1); ++s) {
        q.abytes[s] = extent(A_KM, q.g.seg[s].lda, q.g.M, q.g.seg[s].K);
        q.bbytes[s] = extent(B_KM, q.g.seg[s].ldb, q.g.N, q.g.seg[s].K);
    }
    return fits;
}

// the share of g's tiles that the fp32 form loads without a test for each element
inline double whole_share(const Args& g, const Plan& f) {
    if (g.seg[0].K % KT != 0 || !operands_vec(g)) return 0.0;
    const long mt = (g.M + BM - 1) / BM, nt = (g.N + f.bnt - 1) / f.bnt;
    return (double)(g.M / BM) * (g.N / f.bnt) / ((double)mt * nt);
}

// Whether a pair of products runs by split bf16 rather than by fp32 MFMAs with the plans f0, f1.
// A split block carries more before its first and after its last step, and two of them share a CU
// where three fp32 ones do; the fp32 form loses most where it tests each element that it loads.
// So fp32 stays where its tiles are whole and the products are short, and for a few blocks that
// test nothing, where either form may be the faster.  Evaluations in fp32 / split, us:
//   adjoint, tiles whole       512 x 256 x 256 36.7 / 36.4, 2048 x 256 x 1024 75.7 / 80.2, 2048 x 640 x 640
//                              90.8 / 99.7, 2048 x 768 x 1024 131.7 / 137.7 (model: 67 us); 4096 x 512 x 1024
//                              157.6 / 152.0 (86 us), 4096 x 768 x 1024 219.3 / 204.8
//   adjoint, ragged            1000 x 500 x 700 76.4 / 72.6, 130 x 675 x 207 56.8 / 48.8, 4000 x 784 x 1000 282 / 218
//   adjoint, a few blocks of   384 x 144 x 192 42.3 / 43.8, 128 x 64 x 512 44.2 / 44.9, 32 x 16 x 32 25.6 / 24.4,
//   sizes in sixteens          192 x 176 x 64 48.2 / 45.0; with 45 blocks 1920 x 32 x 64 35.4 / 32.9
//   HVP (dual), tiles whole,   1024 x 512 x 512 119.7 / 124.8, 2048 x 512 x 512 171.4 / 174.6; 512 x 512 x 512
//   8 steps                    (128 blocks each) 101.7 / 97.3; everything else 1.01 to 1.3 times as fast split
inline bool split_pays(const Args& g0, const Plan& f0, const Args& g1, const Plan& f1, int cus, bool dual) {
    auto blocks = [](const Args& g, const Plan& f) {
        return (long)((g.M + BM - 1) / BM) * ((g.N + f.bnt - 1) / f.bnt) * f.ksplit;
    };
    auto steps = [](const Args& g, const Plan& f) { return ((g.seg[0].K + KT - 1) / KT + f.ksplit - 1) / f.ksplit; };
    const long b0 = blocks(g0, f0), b1 = blocks(g1, f1);
    const double w0 = whole_share(g0, f0), w1 = whole_share(g1, f1);
    if (dual) return !(w0 == 1.0 && w1 == 1.0 && steps(g0, f0) <= 8 && steps(g1, f1) <= 8 && b0 >= cus && b1 >= cus);
    if (w0 >= 0.75 && w1 >= 0.75) return f0.us + f1.us >= 80.0;
    auto sixteens = [](const Args& g) { return operands_vec(g) && (g.M | g.N | g.seg[0].K) % KT == 0; };
    return !(sixteens(g0) && sixteens(g1) && b0 + b1 <= 32);
}

// The pair of launch_pair by split bf16; false (and nothing launched) where the sizes or the
// operands are not for it (f0, f1: the fp32 form's plans).  Both epilogues accumulate by atomics
// where K is split.
template <bool A0, bool B0, class E0, bool A1, bool B1, class E1, bool DUAL, class X>
bool launch_split_pair(Args g0, E0 e0, const Plan& f0, Args g1, E1 e1, const Plan& f1, int cus, hipStream_t stream, X x,
                       hipError_t& err) {
    static_assert(has_atomic<E0>::value && has_atomic<E1>::value, "a split adds its slices by atomics");
    const int nout = DUAL ? 2 : 1;
    if (g0.M <= 0 || g0.N <= 0 || g1.M <= 0 || g1.N <= 0 || (DUAL && (g0.seg[0].K != g0.seg[1].K || g1.seg[0].K != g1.seg[1].K)))
        return false;
    if (!split_pays(g0, f0, g1, f1, cus, DUAL)) return false;
    SplitPart<A0, B0, E0> q0{SplitArgs{g0, {0, 0}, {0, 0}}, e0, 0, 0};
    SplitPart<A1, B1, E1> q1{SplitArgs{g1, {0, 0}, {0, 0}}, e1, 0, 0};
    if (!split_extents<A0, B0, DUAL>(q0.q) || !split_extents<A1, B1, DUAL>(q1.q)) return false;
    auto both = [&](int bnt) {
        return std::pair<Plan, Plan>(plan_split(g0.M, g0.N, g0.seg[0].K, cus, nout, bnt),
                                               plan_split(g1.M, g1.N, g1.seg[0].K, cus, nout, bnt));
    };
    const auto n64 = both(64), n128 = both(128);
    const auto& [p0, p1] = DUAL || n64.first.us + n64.second.us <= n128.first.us + n128.second.us ? n64 : n128;
    const int bnt = p0.bnt;
    q0.q.g.ksplit = p0.ksplit;
    q1.q.g.ksplit = p1.ksplit;
    q0.gx = (g0.M + BM - 1) / BM; q0.gy = (g0.N + bnt - 1) / bnt;
    q1.gx = (g1.M + BM - 1) / BM; q1.gy = (g1.N + bnt - 1) / bnt;
    const long nb = (long)x.count + (long)q0.gx * q0.gy * p0.ksplit + (long)q1.gx * q1.gy * p1.ksplit;
    if constexpr (DUAL) {
        split_pair_kernel<64, true, A0, B0, E0, A1, B1, E1, X><<<(unsigned)nb, NT, 0, stream>>>(q0, q1, x);
    } else {
        if (bnt == 128) split_pair_kernel<128, false, A0, B0, E0, A1, B1, E1, X><<<(unsigned)nb, NT, 0, stream>>>(q0, q1, x);
        else split_pair_kernel<64, false, A0, B0, E0, A1, B1, E1, X><<<(unsigned)nb, NT, 0, stream>>>(q0, q1, x);
    }
    err = hipGetLastError();
    return true;
}

}  // namespace gemm
}  // namespace stade
