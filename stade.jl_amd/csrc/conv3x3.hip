// Config 4: conv3x3 -- 3 x 3 convolution (stride 1, zero padding held in the input) and
// half the squared norm of the output, Float32.  Executes the generated adjoint, tangent and
// HVP of corpus/conv3x3.jl (corpus/conv3x3_{b,d,hv}.jl), the functions `stade_amdgpu_file`
// would port (/root/reference/src/STADE.jl:18604-18605).
//
// Layouts (Julia column-major, 0-based below):
//   xp  (i_w+2, i_h+2, i_c, i_nb): xp[n][c][yp][xq] at ((n*C + c)*Hp + yp)*Wp + xq
//   w   (3, 3, i_c, i_k):          w[co][c][ky][kx] at ((co*C + c)*3 + ky)*3 + kx
//   out (i_w, i_h, i_k, i_nb):     out[n][co][y][x] at ((n*K + co)*H + y)*W + x
//
// The generated loops are three products over one index space (pixel, tap, c, co):
//   forward  out[n][co][y][x]   = sum_{c,ky,kx} w[co][c][ky][kx] xp[n][c][y+ky][x+kx]
//   adjoint  g = outb + (0.5 (2 out)) lossb  (the accumulated outb, then reset to 0)
//            wb[co][c][ky][kx] += sum_{n,y,x} g[n][co][y][x] xp[n][c][y+ky][x+kx]
//            xpb[n][c][yp][xq] += sum_{co,ky,kx} w[co][c][ky][kx] g[n][co][yp-ky][xq-kx]
// All three run on the matrix cores as implicit GEMMs, with no im2col buffer: each block stages
// its operands in LDS, and the taps read them there at shifted offsets.  By split bf16, but for
// the forward of the tangent and the HVP (fp32 MFMAs).
//   tap_kernel    the adjoint's forward and the interior of xpb (and xpbd), which is the same
//                 shifted product on g with flipped, transposed weights
//   tap32_kernel  the forward of the tangent and the HVP: out and outd
//   border_kernel the one-cell frame of xpb (taps that land on the zero padding): four 1-D
//                 3-tap line correlations
//   wgrad_kernel  split over pixel tiles, partial 9 x 64 x 64 weight gradients per block
//   wreduce_kernel sums the partials in a fixed order into wb
#include "internal.hpp"
#include "gemm_f32.hpp"
#include "split_bf16.hpp"

#include <algorithm>

namespace stade {
namespace {

constexpr int NT = 256;
constexpr int kBufWord3 = 0x00020000;  // gfx9-family buffer resource word 3 (raw, 32-bit data)

__device__ __forceinline__ floatx16 mfma(float a, float b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// 16-channel chunks of the tap kernel's input channels
__host__ __device__ __forceinline__ int tap_chunks(int Cin) { return (Cin + 15) / 16; }

// ------------------------------------------------------------------------------------------
// weights for the tap kernel, split into their bf16 parts (split_bf16.hpp) in the order of the
// matrix-core fragments that read them: 16-byte cell
//   ((((rt * chunks + ch) * 9 + t) * 3 + part) * 2 + i) * 64 + lane
// holds rows r = 64 rt + 32 i + lane % 32, input channels 16 ch + 8 (lane / 32) + 0..7 of tap t
// (zero past the last row or channel).  Forward: cin = c, r = co, t = 3 ky + kx.  Interior of
// xpb: cin = co, r = c, and the tap flipped (t' = 8 - t), so both products read their source
// at (y + ky' - 1 + ...).  blockIdx.y runs over the forward's rtf row tiles and then those of xpb,
// blockIdx.z over the weights and their direction, and blockIdx.x over a row tile's cells.  Each
// block writes whether it met a weight that the split cannot hold:
//   flags[(blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x],
// so that a tap block asks for those of its own row tile.
// ------------------------------------------------------------------------------------------
struct PrepArgs {
    const float* w[2];
    u32x4* wf[2];
    u32x4* wg[2];
    int* flags;
    int C, K, rtf;
};
__global__ __launch_bounds__(NT) void prep_kernel(PrepArgs a) {
    const int set = blockIdx.z, C = a.C, K = a.K;
    const bool back = (int)blockIdx.y >= a.rtf;
    const int rt = back ? blockIdx.y - a.rtf : blockIdx.y;
    const int Cin = back ? K : C, R = back ? C : K, chunks = tap_chunks(Cin);
    const float* __restrict__ w = a.w[set];
    const long q = (long)blockIdx.x * NT + threadIdx.x;  // (ch, t, i, lane) of the row tile
    uint32_t lost = 0;
    if (q < (long)chunks * 9 * 128) {
        const int lane = (int)(q & 63), i = (int)(q >> 6) & 1;
        const int rest = (int)(q >> 7), t = rest % 9, ch = rest / 9;
        const int r = 64 * rt + 32 * i + (lane & 31), c0 = 16 * ch + 8 * (lane >> 5);
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int cin = c0 + k;
            v[k] = (r < R && cin < Cin) ? (back ? w[((long)cin * C + r) * 9 + (8 - t)] : w[((long)r * C + cin) * 9 + t]) : 0.f;
        }
        u32x4 c[3];
        split8(v, c, lost);
        u32x4* dst = (back ? a.wg : a.wf)[set] + ((((long)rt * chunks + ch) * 9 + t) * 3 * 2 + i) * 64 + lane;
#pragma unroll
        for (int part = 0; part < 3; ++part) dst[part * 128] = c[part];
    }
    const int any = __syncthreads_or(any_lost(lost));
    if (threadIdx.x == 0) a.flags[((long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = any;
}

// ------------------------------------------------------------------------------------------
// tap kernel: o[r][y][x] = sum_{cin, ty, tx} w(cin, 3 ty + tx, r) * src[cin][y + ty + ofs][x + tx + ofs]
//
// Block: TY waves, wave w owning pixel row y0 + w of a 64-row (r) x (TX x TY pixel) output tile
// as 2 x NJ MFMA 32 x 32 tiles (r halves x pixel halves; TX = 32 NJ).  Input channels advance 16
// at a time: the (TY+2) x (TX+2) patch of the chunk is split into bf16 parts in LDS
// (split_bf16.hpp), a 16-byte cell per pixel, part and eight channels, so that a tap's pixel
// fragment is one 128-bit read at a shifted pixel and each element is split once for its 9 taps
// and 64 rows.  The weight fragments come split from prep_kernel.  A tap is one k step of 16
// channels, six bf16 products per tile and source-weight pair; its successor's fragments are
// read while its MFMAs run, and the next chunk is loaded into registers meanwhile.
// One source (NP = 1; adjoint): NJ = 2, and the weights go through LDS with the patch.  Read
// from the cache beside the MFMAs instead, a tap's weights wait for every older load of the
// wave, the next chunk's pixels from HBM among them (loads return in order).  Eight rows give
// two waves a SIMD.
// Two sources (NP = 2; the HVP's xpb and xpbd: three products a tap into two outputs): NJ = 1, the
// weights (two sets, too many for LDS) from the cache.  The two outputs' sums are kept per chunk
// and then added to their totals, which more than halves their rounding.
// Measured, us with fp32 MFMAs -> split: 8 x 64 -> 64 x 256^2, forward 391 -> 287, xpb 385 -> 270;
// the matrix cores are busy for 38 and 39 % of it.  Without the MFMAs' operands being staged, the
// MFMAs and the epilogue alone take 186 and 157 us (672 and 406 MB of HBM traffic); weights
// from the cache with four rows a block: 306 and 290; the splitting interleaved with the MFMAs
// over a double-buffered patch: no faster.  Error against 64 bits 5.0e-7 -> 4.2e-7 (one source;
// two: xpb 3.8e-7 -> 2.3e-7, xpbd 6.4e-7 -> 4.4e-7 at 4 x 32 -> 48 x 112 x 100).
// FRESH: fewer roundings at the total's size, for few channels, where v_mfma_f32_32x32x2_f32
// would round less often than the six products of a tap and chunk do.  One source: a tap's
// products are summed from zero and then added to the total.  Two sources (one chunk then): the
// five small products of all taps first, then the h h of all taps, nine roundings in all.
// A block that meets an element which the split cannot hold, among its pixels or its row tile's
// weights, forms its tile again by v_mfma_f32_32x32x2_f32 with operands straight from memory.
// With one such weight in a single row tile every block does: adjoint at 8 x 64 -> 64 x 256^2 2114 us,
// 810 without (1200 with fp32 MFMAs throughout; 2336 with a tap's loads at a time); 256 -> 256
// channels at 32^2, a weight in one of four row tiles 791 us, 275 without (434; 1076).
// ------------------------------------------------------------------------------------------
constexpr int RT = 64, CC = 16;
constexpr int WCELLS = 9 * 6 * 64;   // weight cells of a chunk and row tile
enum { FWD_B, FWD_D, FWD_HV, DG_B, DG_HV };
constexpr int tap_sources(int mode) { return mode == FWD_B || mode == DG_B ? 1 : 2; }
constexpr bool tap_split(int mode) { return mode != FWD_D && mode != FWD_HV; }
constexpr int tap_width(int mode) { return mode == DG_HV ? 32 : 64; }

struct TapArgs {
    const float* src[2];   // sources (n, cin, SH, SW)
    const u32x4* wt[2];    // split weights (prep_kernel)
    const float* wt32[2];  // the tangent's forward: weights [cin][9][Rpad] (prep32_kernel)
    const float* w[2];     // the weights themselves: (r, cin, t) at w[r * wr + cin * wc + (flip ? 8 - t : t)]
    long wr, wc;
    bool flip;
    const int* flags;      // prep_kernel's: of row tile rt, nflags at rt * nflags, and those of the
    int nflags;            // direction fset further on
    long fset;
    int Cin, R, Rpad, N;
    int SH, SW, ofs;      // source plane and patch origin offset
    int H, W;             // output domain
    float* o0;            // out / xpb
    float* o1;            // outd / xpbd
    int OH, OW, oofs;     // o[((n*R + r)*OH + y + oofs)*OW + x + oofs]
    float* g0;            // forward adjoint: g = accumulated outb, and its tangent
    float* g1;
    float* ob;            // outb, outbd (read, then reset to zero)
    float* obd;
    const float* lossb;
    const float* lossbd;
    double* partials;     // loss sums per block
};

// The outputs of a wave's tile: pixel row y, columns x0..., rows of tile rt.
template <int MODE, int NJ>
__device__ __forceinline__ void tap_epilogue(const TapArgs& a, floatx16 (&acc)[tap_sources(MODE)][2][NJ], int n, int rt, int x0, int y,
                                             double* red) {
    constexpr bool FWD = MODE == FWD_B || MODE == FWD_D || MODE == FWD_HV;
    constexpr int NV = MODE == FWD_B ? 1 : 2;
    const int h = (threadIdx.x & 63) >> 5, l32 = threadIdx.x & 31;
    // accumulator (i, j, q) is row r = rt*64 + 32 i + 8 (q / 4) + 4 h + q % 4,
    // pixel x = x0 + 32 j + l32 of row y
    double ls[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) ls[k] = 0.0;
    float lb = 0.f, lbd = 0.f;
    if constexpr (MODE == FWD_B || MODE == FWD_HV) lb = a.lossb[0];
    if constexpr (MODE == FWD_HV) lbd = a.lossbd[0];
    // The read-modify-write inputs (outb, outbd of the forward adjoint; xpb, xpbd of the
    // interior) are all loaded before any store: the output arrays may alias as far as the
    // compiler knows, so interleaving would serialise one HBM round trip per element.
    constexpr bool RMW = MODE != FWD_D;
    constexpr int NR = (MODE == FWD_HV || MODE == DG_HV) ? 2 : 1;
    float pre[NR][2][NJ][16];
    auto index = [&](int i, int j, int q, long& oi) {
        const int x = x0 + 32 * j + l32;
        const int r = rt * RT + 32 * i + 8 * (q >> 2) + 4 * h + (q & 3);
        oi = ((long)(n * a.R + r) * a.OH + y + a.oofs) * a.OW + x + a.oofs;
        return y < a.H && x < a.W && r < a.R;
    };
    if constexpr (RMW) {
        const float* s0 = FWD ? a.ob : a.o0;
        const float* s1 = FWD ? a.obd : a.o1;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    long oi;
                    const bool ok = index(i, j, q, oi);
                    pre[0][i][j][q] = ok ? s0[oi] : 0.f;
                    if constexpr (NR == 2) pre[NR - 1][i][j][q] = ok ? s1[oi] : 0.f;
                }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                long oi;
                if (!index(i, j, q, oi)) continue;
                const float v = acc[0][i][j][q];
                if constexpr (FWD) {
                    a.o0[oi] = v;
                    ls[0] += 0.5 * (double)v * (double)v;
                    if constexpr (MODE == FWD_B) {
                        a.g0[oi] = pre[0][i][j][q] + (0.5f * (2.0f * v)) * lb;
                        a.ob[oi] = 0.f;
                    } else {
                        const float vd = acc[1][i][j][q];
                        a.o1[oi] = vd;
                        ls[1] += 0.5 * ((double)(2.0f * v) * (double)vd);
                        if constexpr (MODE == FWD_HV) {
                            const float c8 = 0.5f * (2.0f * v);
                            a.g1[oi] = pre[NR - 1][i][j][q] + (lb * (0.5f * (2.0f * vd)) + c8 * lbd);
                            a.g0[oi] = pre[0][i][j][q] + c8 * lb;
                            a.ob[oi] = 0.f;
                            a.obd[oi] = 0.f;
                        }
                    }
                } else {
                    a.o0[oi] = pre[0][i][j][q] + v;
                    if constexpr (MODE == DG_HV) a.o1[oi] = pre[NR - 1][i][j][q] + acc[1][i][j][q];
                }
            }
    if constexpr (FWD) block_partials<NV>(ls, red, a.partials);
}

template <int MODE, int TY, bool FRESH>
__global__ __launch_bounds__(64 * TY) void tap_kernel(TapArgs a) {
    constexpr int NP = tap_sources(MODE);  // sources = weight sets = outputs
    constexpr int TX = tap_width(MODE), NJ = TX / 32;
    constexpr int NTH = 64 * TY, PXW = TX + 2, PYH = TY + 2, PPL = PXW * PYH;  // patch row, rows, pixels
    constexpr int PLANE = PPL * 16;                                // bytes of one (part, octet) plane
    constexpr bool WLDS = NP == 1;                                 // weights staged in LDS
    constexpr int WPT = WLDS ? (WCELLS + NTH - 1) / NTH : 1;       // weight cells of a thread

    __shared__ __attribute__((aligned(16))) char lds[NP * 6 * PLANE];
    __shared__ u32x4 wlds[WLDS ? WCELLS : 1];
    __shared__ double red[16];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY;
    const int rtiles = a.Rpad / RT;
    const int n = blockIdx.z / rtiles, rt = blockIdx.z - n * rtiles;
    const int nchunks = tap_chunks(a.Cin);

    // Patch staging: a cell is one pixel's eight channels of an octet; a source's 2 x PYH x PXW
    // cells (octet, row, column) are shared out over the threads in order, so that consecutive
    // lanes load consecutive pixels.  The loads are buffer loads: a scalar resource per source
    // image n, the channel as a scalar offset, the rest as the lane's.  An element outside the
    // source reads an offset past the resource, which returns 0.  (The host keeps one image of
    // a source under 2^31 bytes.)
    constexpr int NCELL = (2 * PPL + NTH - 1) / NTH;
    float pr[NP][NCELL][8];
    u32x4 wr[WPT];
    const long plane = (long)a.SH * a.SW;
    const uint32_t sbytes = (uint32_t)((long)a.Cin * plane * 4);
    constexpr uint32_t kPast = 0x80000000u;
    __amdgpu_buffer_rsrc_t rs[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p)
        rs[p] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.src[p] + (long)n * a.Cin * plane), (short)0, sbytes,
                                                  kBufWord3);
    uint32_t voff[NCELL];  // the cell's byte offset at channel 8 octet
    int clim[NCELL];       // channels from there on
    int coff[NCELL];       // the cell's place in LDS (part 0)
#pragma unroll
    for (int k = 0; k < NCELL; ++k) {
        const int e = threadIdx.x + NTH * k, row = e / PXW, col = e - row * PXW;
        const int oct = row >= PYH, ty = row - oct * PYH;
        const int sy = y0 + ty + a.ofs, sx = x0 + col + a.ofs;
        const bool in = e < 2 * PPL && (unsigned)sy < (unsigned)a.SH && (unsigned)sx < (unsigned)a.SW;
        clim[k] = in ? a.Cin - 8 * oct : 0;
        voff[k] = in ? (uint32_t)((8 * oct * plane + (long)sy * a.SW + sx) * 4) : kPast;
        coff[k] = oct * PLANE + (ty * PXW + col) * 16;
    }
    auto load = [&](int ch) {
        if constexpr (WLDS) {
            const u32x4* w = a.wt[0] + ((long)rt * nchunks + ch) * WCELLS;
#pragma unroll
            for (int q = 0; q < WPT; ++q)
                if (WCELLS % NTH == 0 || threadIdx.x + NTH * q < WCELLS) wr[q] = w[threadIdx.x + NTH * q];
        }
#pragma unroll
        for (int k = 0; k < NCELL; ++k)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int c = CC * ch + e;
                const uint32_t soff = (uint32_t)(min(c, a.Cin) * plane * 4), v = c < clim[k] ? voff[k] : kPast;
#pragma unroll
                for (int p = 0; p < NP; ++p)
                    pr[p][k][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs[p], v, soff, 0));
            }
    };
    uint32_t lost = 0;
    auto store = [&]() {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int k = 0; k < NCELL; ++k) {
                u32x4 c[3];
                split8(pr[p][k], c, lost);
                if ((2 * PPL) % NTH == 0 || threadIdx.x + NTH * k < 2 * PPL)
#pragma unroll
                    for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(lds + (p * 6 + 2 * q) * PLANE + coff[k]) = c[q];
            }
        if constexpr (WLDS) {
#pragma unroll
            for (int q = 0; q < WPT; ++q)
                if (WCELLS % NTH == 0 || threadIdx.x + NTH * q < WCELLS) wlds[threadIdx.x + NTH * q] = wr[q];
        }
    };

    floatx16 acc[NP][2][NJ];
    auto clear = [&]() {
#pragma unroll
        for (int o = 0; o < NP; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int q = 0; q < 16; ++q) acc[o][i][j][q] = 0.f;
    };
    clear();

    // fragments, two sets: a tap's are read during the tap before
    bf16x8 wv[2][NP][2][3], pv[2][NP][NJ][3];
    auto read_weights = [&](int ch, int t, int buf) {
        if constexpr (WLDS) {
#pragma unroll
            for (int q = 2; q >= 0; --q)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    wv[buf][0][i][q] = __builtin_bit_cast(bf16x8, wlds[(t * 6 + q * 2 + i) * 64 + lane]);
            return;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<u32x4*>(a.wt[p] + ((long)rt * nchunks + ch) * (9 * 6 * 64)), (short)0, 9 * 6 * 1024, kBufWord3);
#pragma unroll
            for (int q = 2; q >= 0; --q)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    wv[buf][p][i][q] = __builtin_bit_cast(
                        bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, (uint32_t)lane * 16u, (uint32_t)(t * 6 + q * 2 + i) * 1024u, 0));
        }
    };
    auto read_pixels = [&](int t, int buf) {
        const int ky = t / 3, kx = t % 3;
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    pv[buf][p][j][q] = *reinterpret_cast<const bf16x8*>(lds + (p * 6 + 2 * q + h) * PLANE + ((wave + ky) * PXW + kx + 32 * j + l32) * 16);
    };
    // two sources: the chunks' sums (acc) are added up here; one source, FRESH: the taps'
    constexpr bool TOT = NP == 2 || FRESH;
    // two sources, FRESH: the taps' small products first, then those of the h parts
    constexpr int PASSES = NP == 2 && FRESH ? 2 : 1, STEPS = 9 * PASSES;
    floatx16 tot[TOT ? NP : 1][2][NJ];
    if constexpr (TOT) {
#pragma unroll
        for (int o = 0; o < NP; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) tot[o][i][j] = acc[o][i][j];
    }
    if (nchunks > 0) {
        load(0);
        if (!WLDS) read_weights(0, 0, 0);
    }
    for (int ch = 0; ch < nchunks; ++ch) {
        __syncthreads();
        store();
        __syncthreads();
        if (ch + 1 < nchunks) load(ch + 1);
        if (WLDS) read_weights(ch, 0, 0);
        read_pixels(0, 0);
        auto tap = [&](int t, int b) {
            if (t < STEPS - 1) {
                read_pixels((t + 1) % 9, b ^ 1);
                read_weights(ch, (t + 1) % 9, b ^ 1);
            } else if (!WLDS && ch + 1 < nchunks) {
                read_weights(ch + 1, 0, b ^ 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int x = t < 9 ? 0 : 5; x < (PASSES == 2 && t < 9 ? 5 : 6); ++x)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        acc[0][i][j] = mfma_bf16(wv[b][0][i][kSplitB[x]], pv[b][0][j][kSplitA[x]], acc[0][i][j]);
                        if constexpr (NP == 2) {
                            acc[1][i][j] = mfma_bf16(wv[b][1][i][kSplitB[x]], pv[b][0][j][kSplitA[x]], acc[1][i][j]);
                            acc[1][i][j] = mfma_bf16(wv[b][0][i][kSplitB[x]], pv[b][1][j][kSplitA[x]], acc[1][i][j]);
                        }
                    }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int t = 0; t < STEPS; ++t) {
            tap(t, t & 1);
            if constexpr (TOT) {
                if (!(NP == 1 && FRESH) && t != STEPS - 1) continue;
#pragma unroll
                for (int o = 0; o < NP; ++o)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < NJ; ++j)
#pragma unroll
                            for (int q = 0; q < 16; ++q) {
                                tot[o][i][j][q] += acc[o][i][j][q];
                                acc[o][i][j][q] = 0.f;
                            }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (!WLDS && STEPS % 2 == 1) {
            // (nine taps leave the next chunk's first weights in the other set: it is copied over)
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int q = 0; q < 3; ++q) wv[0][p][i][q] = wv[1][p][i][q];
        }
    }

    if constexpr (TOT) {
#pragma unroll
        for (int o = 0; o < NP; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[o][i][j] = tot[o][i][j];
    }
    // an element that the split cannot hold, or a sum that is not finite: the tile again in fp32
    {
        float z = 0.f;
#pragma unroll
        for (int o = 0; o < NP; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int q = 0; q < 16; ++q) z = __builtin_fmaf(acc[o][i][j][q], 0.f, z);
        bool redo = z != 0.f || any_lost(lost);
#pragma unroll
        for (int p = 0; p < NP; ++p)
            for (int k = threadIdx.x; k < a.nflags; k += NTH) redo = redo || a.flags[p * a.fset + (long)rt * a.nflags + k];
        if (__syncthreads_or(redo)) {
            clear();
            // (a channel pair's nine taps are in flight together: one memory latency a pair)
            for (int c0 = 0; c0 < a.Cin; c0 += 2) {
                const int c = c0 + h;
                float wf[9][NP][2], pf[9][NP][NJ];
#pragma unroll
                for (int t = 0; t < 9; ++t) {
                    const int sy = y0 + wave + t / 3 + a.ofs;
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            const int r = rt * RT + 32 * i + l32;
                            wf[t][p][i] = c < a.Cin && r < a.R ? a.w[p][r * a.wr + c * a.wc + (a.flip ? 8 - t : t)] : 0.f;
                        }
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            const int sx = x0 + 32 * j + l32 + t % 3 + a.ofs;
                            pf[t][p][j] = c < a.Cin && (unsigned)sy < (unsigned)a.SH && (unsigned)sx < (unsigned)a.SW
                                              ? a.src[p][((long)(n * a.Cin + c) * a.SH + sy) * a.SW + sx] : 0.f;
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < 9; ++t)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            acc[0][i][j] = mfma(wf[t][0][i], pf[t][0][j], acc[0][i][j]);
                            if constexpr (NP == 2) {
                                acc[1][i][j] = mfma(wf[t][1][i], pf[t][0][j], acc[1][i][j]);
                                acc[1][i][j] = mfma(wf[t][0][i], pf[t][1][j], acc[1][i][j]);
                            }
                        }
            }
        }
    }

    tap_epilogue<MODE, NJ>(a, acc, n, rt, x0, y0 + wave, red);
}

// ------------------------------------------------------------------------------------------
// the tangent's forward (tangent, HVP): out and outd by fp32 MFMAs (v_mfma_f32_32x32x2_f32).
// lossd is a sum of products of out and outd that cancel: its relative error is theirs times a
// condition number that is 10 for one set of inputs and 100 for another, so that two forms of
// rounding agree in lossd to 5e-6 or not by chance.  By split bf16 this kernel takes 0.66 of the
// time (8 x 64 -> 64 x 256^2: 1028 -> 678 us a tangent), with half the error in out and outd, but
// with a lossd that differs by up to 6e-6 (4 x 32 -> 48 x 112 x 100) from that of a sum rounded in
// channel order.
//
// Block: 256 threads, a 64-row (r) x (64 x 4 pixel) output tile.  Wave w owns pixel row
// y0 + w: 2 x 2 MFMA 32 x 32 tiles (r halves x pixel halves) of each output.  Input channels
// advance 8 at a time; each step stages the (4+2) x (64+2) patch of every channel and the 9 x 64
// weight rows in LDS.  The next step's global loads are issued into registers before the MFMAs
// of the current one.  The MFMA k pair (lane / 32) is a pair of channels at the same tap, so
// every LDS read has a lane base plus an immediate offset.  72 % of the fp32 matrix peak
// (8 x 64 -> 64 x 256^2).
// ------------------------------------------------------------------------------------------
// its weights and their directions: wt[cin][t][r], rows padded to a multiple of 64 with zeros
__global__ __launch_bounds__(NT) void prep32_kernel(const float* __restrict__ w, const float* __restrict__ wd, int C, int K,
                                                    float* __restrict__ wf, float* __restrict__ wfd, int Kpad) {
    const long q = (long)blockIdx.x * NT + threadIdx.x;
    if (q >= (long)C * 9 * Kpad) return;
    const int r = (int)(q % Kpad);
    const long ct = q / Kpad;
    const int t = (int)(ct % 9), c = (int)(ct / 9);
    const long i = ((long)r * C + c) * 9 + t;
    wf[q] = r < K ? w[i] : 0.f;
    wfd[q] = r < K ? wd[i] : 0.f;
}

template <int MODE>
__global__ __launch_bounds__(NT) void tap32_kernel(TapArgs a) {
    constexpr int NP = 2;  // sources = weight sets = outputs
    constexpr int TX = 64, TY = 4, CC = 8;
    constexpr int PXW = TX + 2, PYH = TY + 2, PPL = PXW * PYH;  // patch row, rows, plane (floats)
    constexpr int KW = 9 * RT;                                    // weight floats per channel
    constexpr int PSZ = CC * PPL, WSZ = CC * KW;
    constexpr int WLD = NP * WSZ / 4 / NT;
    static_assert(NP * WSZ % (4 * NT) == 0, "weight stage");

    __shared__ float lds[NP * (PSZ + WSZ)];
    __shared__ double red[32];
    float* Ps = lds;
    float* Ws = lds + NP * PSZ;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = lane >> 5, l32 = lane & 31;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY;
    const int rtiles = a.Rpad / RT;
    const int n = blockIdx.z / rtiles, rt = blockIdx.z - n * rtiles;

    // Patch staging by rows: the NP * CC * PYH = 96 patch rows of PXW = 66 floats; wave w
    // takes rows w, w + 4, ..., one column per lane (columns 0..63), so the channel, row and
    // row bounds are wave-uniform (scalar) and a lane's address is a row base plus its lane;
    // columns 64, 65 of every row go to threads 0..191, one element each.
    constexpr int PROWS = NP * CC * PYH, RPW = PROWS / 4;
    static_assert(PROWS % 4 == 0 && PXW == 66 && 2 * PROWS <= NT, "patch rows");
    float pr[RPW + 1];
    float4 wr[WLD];
    // Staging loads are buffer loads: a scalar resource per source image n (and per weight
    // set), the row part of a patch address as a scalar offset (patch rows are wave-uniform)
    // and the column as the lane's offset.  An element outside the source reads offset =
    // the resource's size, which returns 0.  Vector registers hold no 64-bit addresses, so the
    // staging fits two waves per SIMD without spilling.  (The host keeps one image of a
    // source and a weight set under 2^31 bytes.)
    const long plane = (long)a.SH * a.SW;
    const uint32_t sbytes = (uint32_t)((long)a.Cin * plane * 4);
    const uint32_t wbytes = (uint32_t)((long)a.Cin * 9 * a.Rpad * 4);
    __amdgpu_buffer_rsrc_t rs[NP], rw[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        rs[p] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.src[p] + (long)n * a.Cin * plane), (short)0, sbytes,
                                                  kBufWord3);
        rw[p] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.wt32[p] + rt * RT), (short)0, wbytes, kBufWord3);
    }
    const int sx_l = x0 + lane + a.ofs;
    const uint32_t lane_col = (unsigned)sx_l < (unsigned)a.SW ? (uint32_t)sx_l * 4u : sbytes;
    auto load = [&](int c0) {
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            const int rr = wave + 4 * i;  // wave-uniform patch row (p, cc, ty)
            const int p = rr / (CC * PYH);
            const int rem = rr - p * (CC * PYH);
            const int cc = rem / PYH, ty = rem - cc * PYH;
            const int c = c0 + cc, sy = y0 + ty + a.ofs;
            const bool ok = c < a.Cin && (unsigned)sy < (unsigned)a.SH;
            const uint32_t soff = ok ? (uint32_t)(((long)c * a.SH + sy) * a.SW * 4) : 0u;
            const uint32_t voff = ok ? lane_col : sbytes;
            pr[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(p ? rs[NP - 1] : rs[0], voff, soff, 0));
        }
        if (threadIdx.x < 2 * PROWS) {
            // columns 64, 65: the row varies across a wave, so the whole offset is the lane's
            const int rr = threadIdx.x >> 1, col = 64 + (threadIdx.x & 1);
            const int p = rr / (CC * PYH);
            const int rem = rr - p * (CC * PYH);
            const int cc = rem / PYH, ty = rem - cc * PYH;
            const int c = c0 + cc, sy = y0 + ty + a.ofs, sx = x0 + col + a.ofs;
            float v = 0.f;
            if (c < a.Cin && (unsigned)sy < (unsigned)a.SH && (unsigned)sx < (unsigned)a.SW)
                v = a.src[p][((long)(n * a.Cin + c) * a.SH + sy) * a.SW + sx];
            pr[RPW] = v;
        }
        const uint32_t wsoff = (uint32_t)((long)c0 * 9 * a.Rpad * 4);
#pragma unroll
        for (int q = 0; q < WLD; ++q) {
            const int f = threadIdx.x + q * NT;  // float4 slot of [w][cc][t][r]
            const int wi = __builtin_amdgcn_readfirstlane(f / (WSZ / 4));  // uniform per wave
            const int rem = f - wi * (WSZ / 4);
            const int row = rem / (RT / 4), r4 = (rem - row * (RT / 4)) * 4;
            const int cc = row / 9, t = row - cc * 9;
            const uint32_t voff = c0 + cc < a.Cin ? (uint32_t)(((cc * 9 + t) * a.Rpad + r4) * 4) : wbytes;
            const v4f x = __builtin_amdgcn_raw_buffer_load_b128(wi ? rw[NP - 1] : rw[0], voff, wsoff, 0);
            wr[q] = make_float4(x.x, x.y, x.z, x.w);
        }
    };
    auto store = [&]() {
        // patch row rr = (p, cc, ty) is at Ps + p * PSZ + cc * PPL + ty * PXW = Ps + rr * PXW
#pragma unroll
        for (int i = 0; i < RPW; ++i) Ps[(wave + 4 * i) * PXW + lane] = pr[i];
        if (threadIdx.x < 2 * PROWS) Ps[(threadIdx.x >> 1) * PXW + 64 + (threadIdx.x & 1)] = pr[RPW];
#pragma unroll
        for (int q = 0; q < WLD; ++q) {
            const int f = threadIdx.x + q * NT;
            *reinterpret_cast<float4*>(Ws + 4 * f) = wr[q];
        }
    };

    floatx16 acc[NP][2][2];
#pragma unroll
    for (int o = 0; o < NP; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[o][i][j][q] = 0.f;

    // lane bases: patch channel (2 qq + h), row (wave + ky), column (32 j + l32 + kx);
    // weight row (2 qq + h, t), column 32 i + l32
    const int pbase = h * PPL + wave * PXW + l32;
    const int wbase = h * KW + l32;
    const int nchunks = (a.Cin + CC - 1) / CC;
    if (nchunks > 0) load(0);
    for (int ch = 0; ch < nchunks; ++ch) {
        __syncthreads();
        store();
        __syncthreads();
        if (ch + 1 < nchunks) load((ch + 1) * CC);
        // k steps st = (channel pair qq, tap t); the fragments of step st+1 are read from LDS
        // while the MFMAs of step st run (two register sets; the scheduling barriers keep
        // the compiler from sinking each read to its use)
        constexpr int NSTEP = CC / 2 * 9;
        float pf[2][NP][2], wf[2][NP][2];
        auto frag = [&](int st, int buf) {
            const int qq = st / 9, t = st % 9, ky = t / 3, kx = t % 3;
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int j = 0; j < 2; ++j) pf[buf][p][j] = Ps[p * PSZ + pbase + 2 * qq * PPL + ky * PXW + kx + 32 * j];
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int i = 0; i < 2; ++i) wf[buf][p][i] = Ws[p * WSZ + wbase + (2 * qq * 9 + t) * RT + 32 * i];
        };
        frag(0, 0);
#pragma unroll
        for (int st = 0; st < NSTEP; ++st) {
            const int b = st & 1;
            if (st + 1 < NSTEP) frag(st + 1, b ^ 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    acc[0][i][j] = mfma(wf[b][0][i], pf[b][0][j], acc[0][i][j]);
                    acc[1][i][j] = mfma(wf[b][1][i], pf[b][0][j], acc[1][i][j]);
                    acc[1][i][j] = mfma(wf[b][0][i], pf[b][1][j], acc[1][i][j]);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    tap_epilogue<MODE, 2>(a, acc, n, rt, x0, y0 + wave, red);
}

// loss (and lossd) += the sum of the tap kernel's block partials, rounded once to Float32
template <int NV>
__global__ __launch_bounds__(NT) void loss_kernel(const double* __restrict__ partials, int nparts, float* l0, float* l1) {
    __shared__ double red[16 * NV];
    double acc[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = 0.0;
    // unrolled so that several partials' loads are in flight (the sums keep their order)
#pragma unroll 8
    for (int b = threadIdx.x; b < nparts; b += NT)
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[k] += partials[(long)b * NV + k];
    block_sum<NV>(acc, red);
    if (threadIdx.x == 0) {
        // both destinations read before either is written (they may alias as far as the
        // compiler knows)
        const float o0 = l0[0], o1 = NV == 2 ? l1[0] : 0.f;
        l0[0] = (float)((double)o0 + acc[0]);
        if (NV == 2) l1[0] = (float)((double)o1 + acc[NV - 1]);
    }
}

// ------------------------------------------------------------------------------------------
// frame of xpb: padded cells with yp in {0, Hp-1} or xq in {0, Wp-1}.  On each edge only one
// tap row (or column) lands inside the image, so an edge is a 1-D 3-tap full correlation
// along one line of g:
//   top    (yp = 0,    p = xq in 0..W+1):  sum_co sum_d w[co][c][0][d]  g[co][0][p - d]
//   bottom (yp = Hp-1, p = xq):            sum_co sum_d w[co][c][2][d]  g[co][H-1][p - d]
//   left   (xq = 0,    p = yp-1 in 0..H-1): sum_co sum_d w[co][c][d][0] g[co][p + 1 - d][0]
//   right  (xq = Wp-1, p = yp-1):          sum_co sum_d w[co][c][d][2]  g[co][p + 1 - d][W-1]
// (g zero outside the image).  Block: 64 cells of one edge x 16 channels c; output
// channels advance 16 at a time through LDS (the g line segment and the weight slice).
// ------------------------------------------------------------------------------------------
constexpr int BSEG = 64, BKC = 64, BCG = 16;  // cells, output channels per staging round, input channels

struct BorderArgs {
    const float* w;
    const float* wd;
    const float* g;
    const float* gd;
    float* xpb;
    float* xpbd;
    int N, C, K, H, W;
};

template <bool HV>
__global__ __launch_bounds__(NT) void border_kernel(BorderArgs a) {
    constexpr int NG = HV ? 2 : 1;
    __shared__ float gl[NG][BKC][BSEG + 2];
    __shared__ float4 wv[NG][BKC][3][BCG / 4];  // [kk][d][c]: a thread's 4 channels in one read
    const int e = blockIdx.y;
    const int L = e < 2 ? a.W + 2 : a.H;
    const int p0 = blockIdx.x * BSEG;
    if (p0 >= L) return;  // whole block
    const int ncg = (a.C + BCG - 1) / BCG;
    const int n = blockIdx.z / ncg, c0 = (blockIdx.z % ncg) * BCG;
    const int off = e < 2 ? 0 : 1;
    const int fixed = (e == 0 || e == 2) ? 0 : 2;
    const int lim = e < 2 ? a.W : a.H;
    const int cell = threadIdx.x & 63, cg = threadIdx.x >> 6;
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, accd[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < a.K; k0 += BKC) {
        __syncthreads();
        // every staging load of the round issued before any LDS store (one memory round trip)
        constexpr int NGL = (BKC * (BSEG + 2) + NT - 1) / NT, NWL = BKC * BCG * 3 / NT;
        static_assert(BKC * BCG * 3 % NT == 0, "weight staging");
        float gv_[NGL], gvd_[NGL], wv_[NWL], wvd_[NWL];
#pragma unroll
        for (int u = 0; u < NGL; ++u) {
            const int f = threadIdx.x + u * NT;
            const int kk = f / (BSEG + 2), i = f - kk * (BSEG + 2);
            const int co = k0 + kk, q = p0 + off - 2 + i;
            float v = 0.f, vd = 0.f;
            if (f < BKC * (BSEG + 2) && co < a.K && q >= 0 && q < lim) {
                const long plane = (long)(n * a.K + co) * a.H;
                const long gi = e < 2 ? (plane + (e == 0 ? 0 : a.H - 1)) * a.W + q : (plane + q) * a.W + (e == 2 ? 0 : a.W - 1);
                v = a.g[gi];
                if (HV) vd = a.gd[gi];
            }
            gv_[u] = v;
            gvd_[u] = vd;
        }
#pragma unroll
        for (int u = 0; u < NWL; ++u) {
            const int f = threadIdx.x + u * NT;
            const int kk = f / (BCG * 3), r = f - kk * (BCG * 3);
            const int cc = r / 3, d = r - cc * 3;
            const int co = k0 + kk, c = c0 + cc;
            float v = 0.f, vd = 0.f;
            if (co < a.K && c < a.C) {
                const int ky = e < 2 ? fixed : d, kx = e < 2 ? d : fixed;
                const long wi = ((long)co * a.C + c) * 9 + 3 * ky + kx;
                v = a.w[wi];
                if (HV) vd = a.wd[wi];
            }
            wv_[u] = v;
            wvd_[u] = vd;
        }
#pragma unroll
        for (int u = 0; u < NGL; ++u) {
            const int f = threadIdx.x + u * NT;
            if (f < BKC * (BSEG + 2)) {
                const int kk = f / (BSEG + 2), i = f - kk * (BSEG + 2);
                gl[0][kk][i] = gv_[u];
                if (HV) gl[NG - 1][kk][i] = gvd_[u];
            }
        }
#pragma unroll
        for (int u = 0; u < NWL; ++u) {
            const int f = threadIdx.x + u * NT;
            const int kk = f / (BCG * 3), r = f - kk * (BCG * 3);
            const int cc = r / 3, d = r - cc * 3;
            reinterpret_cast<float*>(&wv[0][kk][d][0])[cc] = wv_[u];
            if (HV) reinterpret_cast<float*>(&wv[NG - 1][kk][d][0])[cc] = wvd_[u];
        }
        __syncthreads();
#pragma unroll 4
        for (int kk = 0; kk < BKC; ++kk)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const float gv = gl[0][kk][cell + 2 - d];
                const float gvd = HV ? gl[NG - 1][kk][cell + 2 - d] : 0.f;
                const float4 w4 = wv[0][kk][d][cg];
                const float4 wd4 = HV ? wv[NG - 1][kk][d][cg] : make_float4(0.f, 0.f, 0.f, 0.f);
                const float wc_[4] = {w4.x, w4.y, w4.z, w4.w}, wdc_[4] = {wd4.x, wd4.y, wd4.z, wd4.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc[i] += wc_[i] * gv;
                    if (HV) accd[i] += wdc_[i] * gv + wc_[i] * gvd;
                }
            }
    }
    const int p = p0 + cell;
    if (p >= L) return;
    const int Hp = a.H + 2, Wp = a.W + 2;
    const int yp = e == 0 ? 0 : e == 1 ? Hp - 1 : p + 1;
    const int xq = e < 2 ? p : (e == 2 ? 0 : Wp - 1);
    // every xpb (xpbd) value read before any is written (the arrays may alias as far as the
    // compiler knows)
    float old[4], oldd[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = c0 + 4 * cg + i;
        const long oi = ((long)(n * a.C + c) * Hp + yp) * Wp + xq;
        old[i] = c < a.C ? a.xpb[oi] : 0.f;
        oldd[i] = (HV && c < a.C) ? a.xpbd[oi] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = c0 + 4 * cg + i;
        if (c >= a.C) continue;
        const long oi = ((long)(n * a.C + c) * Hp + yp) * Wp + xq;
        a.xpb[oi] = old[i] + acc[i];
        if (HV) a.xpbd[oi] = oldd[i] + accd[i];
    }
}

// ------------------------------------------------------------------------------------------
// weight gradient: part[split][ct][kt][t][ci][co] = sum over the split's pixel rows of
//   sum_p sum_{pixel} x_p[n][c][y+ky][x+kx] * g_p[n][co][y][x]
// Block: 256 threads, a 64 (c) x 64 (co) slab of all 9 taps; wave (wa, wb) owns the 32 x 32
// quarter (c half wa, co half wb) of every tap: 9 accumulator tiles.  The pixels are the
// product's k: strips of 8 S columns, walked down row by row.  Each row's x (64 channels) and g
// (64 channels) are split into bf16 parts (split_bf16.hpp) once and kept in LDS, x in a ring of
// four rows, so that a row is read from memory once for its three ky.
// Cell s of a row holds the eight pixels s, s + S, .., s + 7 S of one channel: a tap's shift by
// kx is then another cell and not a misaligned read (S + 2 cells hold all three shifts, a quarter
// of the row twice), and cells 2 ks, 2 ks + 1 are one k step of 16 pixels.  A cell plane is 65
// channels wide so that the staging threads, consecutive in s, write to different banks.
// A row's products (24 a tap) are summed from zero and then added to the total, which rounds
// once a row there where v_mfma_f32_32x32x2_f32 rounds every two pixels.  The next row is
// loaded, split and stored between the MFMAs.  A block that meets an element which the split
// cannot hold forms its sums again in fp32 with operands straight from memory (with one such
// pixel the adjoint at 8 x 64 -> 64 x 256^2 takes 1649 us, 810 without; through LDS, without the
// loads of the next pixels in flight, 1678).
// Measured, us with fp32 MFMAs (tiles of 32 x 2 pixels, each row staged twice) -> split:
// 8 x 64 -> 64 x 256^2 390 -> 235 (165 TFLOP/s; the MFMAs alone 93 at the bf16 peak).  One wave
// a SIMD (453 registers): what the MFMAs do not hide is the LDS reads (120 of 16 bytes a wave and
// row beside 216 MFMAs) and the two barriers a row.
// ------------------------------------------------------------------------------------------
constexpr int WGP = 65;  // channels of a cell plane, padded

struct WgArgs {
    const float* x[2];  // xp-shaped
    const float* g[2];  // out-shaped
    int N, C, K, H, W;
    int ntx;            // strips
    long nrows;         // pixel rows of all strips, images and (x, g) pairs
    float* part;
};

// a block's pixel rows: [lo, hi) of the nrows, in the order pair, image, strip, y
struct WgRow {
    int pr, n, x0, y;
    __device__ __forceinline__ WgRow(const WgArgs& a, long r, int width) {
        const long q = r / a.H;
        y = (int)(r - q * a.H);
        const long i = q / a.ntx;
        x0 = (int)(q - i * a.ntx) * width;
        pr = i >= a.N;
        n = (int)(i - (long)pr * a.N);
    }
};

template <int S>
__global__ __launch_bounds__(NT) void wgrad_kernel(WgArgs a) {
    constexpr int XC = 64 * (S + 2), GC = 64 * S;                    // cells of a row
    constexpr int NX = (XC + NT - 1) / NT, NG = (GC + NT - 1) / NT;  // ... of a thread
    constexpr int XPART = (S + 2) * WGP, GPART = S * WGP;            // ... of a part, padded
    __shared__ u32x4 xs[4][3 * XPART];
    __shared__ u32x4 gs[3 * GPART];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const int ktn = (a.K + 63) / 64;
    const int ct = blockIdx.x / ktn, kt = blockIdx.x - ct * ktn;
    const int c0 = ct * 64, k0 = kt * 64;
    const int wa = wave & 1, wb = wave >> 1;
    const int Hp = a.H + 2, Wp = a.W + 2;
    const int xplane = Hp * Wp, gplane = a.H * a.W;
    const long lo = a.nrows * blockIdx.y / gridDim.y, hi = a.nrows * (blockIdx.y + 1) / gridDim.y;

    // Buffer loads: a scalar resource per image, the row as a scalar offset, channel and pixel
    // as the lane's; an element outside reads an offset past the resource, which returns 0.
    // (The host keeps one image under 2^31 bytes.)
    constexpr uint32_t kPast = 0x80000000u;
    __amdgpu_buffer_rsrc_t rx, rg;
    auto image = [&](const WgRow& w) {
        rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x[w.pr] + (long)w.n * a.C * xplane), (short)0,
                                               (uint32_t)((long)a.C * xplane * 4), kBufWord3);
        rg = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.g[w.pr] + (long)w.n * a.K * gplane), (short)0,
                                               (uint32_t)((long)a.K * gplane * 4), kBufWord3);
    };
    auto fetch = [&](__amdgpu_buffer_rsrc_t rs, uint32_t v, uint32_t soff) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, v, soff, 0));
    };

    floatx16 acc[9];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[t][q] = 0.f;
    };
    clear();

    float xr[NX][8], gr[NG][8];
    uint32_t xoff[NX], goff[NG];  // byte offset of a cell's first pixel in row 0
    int xlim[NX], glim[NG];       // its pixels inside the row
    auto strip = [&](int x0) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int e = threadIdx.x + NT * i, ci = e / (S + 2), s = e - ci * (S + 2);
            const bool in = e < XC && c0 + ci < a.C;
            xoff[i] = in ? (uint32_t)((c0 + ci) * xplane + x0 + s) * 4u : kPast;
            xlim[i] = in ? (Wp - x0 - s + S - 1) / S : 0;
        }
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int e = threadIdx.x + NT * i, co = e / S, s = e - co * S;
            const bool in = e < GC && k0 + co < a.K;
            goff[i] = in ? (uint32_t)((k0 + co) * gplane + x0 + s) * 4u : kPast;
            glim[i] = in ? (a.W - x0 - s + S - 1) / S : 0;
        }
    };
    auto load_x = [&](int i, int yy) {  // row yy of the padded image
        const uint32_t soff = (uint32_t)(min(yy, Hp - 1) * Wp) * 4u;
#pragma unroll
        for (int j = 0; j < 8; ++j) xr[i][j] = fetch(rx, j < xlim[i] ? xoff[i] + (uint32_t)(S * j * 4) : kPast, soff);
    };
    auto load_g = [&](int i, int y) {
        const uint32_t soff = (uint32_t)(min(y, a.H - 1) * a.W) * 4u;
#pragma unroll
        for (int j = 0; j < 8; ++j) gr[i][j] = fetch(rg, j < glim[i] ? goff[i] + (uint32_t)(S * j * 4) : kPast, soff);
    };
    uint32_t lost = 0;
    auto store_x = [&](int i, int yy) {
        const int e = threadIdx.x + NT * i, ci = e / (S + 2), s = e - ci * (S + 2);
        u32x4 c[3];
        split8(xr[i], c, lost);
        if (XC % NT == 0 || e < XC)
#pragma unroll
            for (int q = 0; q < 3; ++q) xs[yy & 3][q * XPART + s * WGP + ci] = c[q];
    };
    auto store_g = [&](int i) {
        const int e = threadIdx.x + NT * i, co = e / S, s = e - co * S;
        u32x4 c[3];
        split8(gr[i], c, lost);
        if (GC % NT == 0 || e < GC)
#pragma unroll
            for (int q = 0; q < 3; ++q) gs[q * GPART + s * WGP + co] = c[q];
    };

    for (long r = lo; r < hi;) {
        const WgRow w(a, r, 8 * S);
        const long end = min(hi, r + (a.H - w.y));
        image(w);
        strip(w.x0);
        // the strip's first rows; the row after them stays in registers
#pragma unroll
        for (int k = 0; k < 3; ++k) {
#pragma unroll
            for (int i = 0; i < NX; ++i) load_x(i, w.y + k);
#pragma unroll
            for (int i = 0; i < NX; ++i) store_x(i, w.y + k);
        }
#pragma unroll
        for (int i = 0; i < NG; ++i) load_g(i, w.y);
#pragma unroll
        for (int i = 0; i < NG; ++i) store_g(i);
#pragma unroll
        for (int i = 0; i < NX; ++i) load_x(i, w.y + 3);
#pragma unroll
        for (int i = 0; i < NG; ++i) load_g(i, w.y + 1);
        __syncthreads();
        for (int y = w.y; r < end; ++r, ++y) {
            bf16x8 gf[S / 2][3], xf[2][3][3];
#pragma unroll
            for (int ks = 0; ks < S / 2; ++ks)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    gf[ks][q] = __builtin_bit_cast(bf16x8, gs[q * GPART + (2 * ks + h) * WGP + 32 * wb + l32]);
            auto frag = [&](int u, int buf) {  // u: ky S / 2 + ks
                const int ky = u / (S / 2), ks = u % (S / 2);
                const u32x4* row = xs[(y + ky) & 3];
#pragma unroll
                for (int kx = 0; kx < 3; ++kx)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        xf[buf][kx][q] = __builtin_bit_cast(bf16x8, row[q * XPART + (2 * ks + kx + h) * WGP + 32 * wa + l32]);
            };
            frag(0, 0);
            __syncthreads();  // g's fragments are read: its next row may be stored
            floatx16 sum[3];
#pragma unroll
            for (int u = 0; u < 3 * (S / 2); ++u) {
                const int ky = u / (S / 2), ks = u % (S / 2), b = u & 1;
                if (u + 1 < 3 * (S / 2)) frag(u + 1, b ^ 1);
                if (ks == 0)
#pragma unroll
                    for (int kx = 0; kx < 3; ++kx)
#pragma unroll
                        for (int q = 0; q < 16; ++q) sum[kx][q] = 0.f;
                __builtin_amdgcn_sched_barrier(0);
                // a cell of the next row a group (the last stored row is never read)
                if (u < NX) {
                    store_x(u, y + 3);
                    load_x(u, y + 4);
                } else if (u - NX < NG) {
                    store_g(u - NX);
                    load_g(u - NX, y + 2);
                }
#pragma unroll
                for (int x = 0; x < 6; ++x)
#pragma unroll
                    for (int kx = 0; kx < 3; ++kx) sum[kx] = mfma_bf16(xf[b][kx][kSplitA[x]], gf[ks][kSplitB[x]], sum[kx]);
                if (ks == S / 2 - 1)
#pragma unroll
                    for (int kx = 0; kx < 3; ++kx)
#pragma unroll
                        for (int q = 0; q < 16; ++q) acc[3 * ky + kx][q] += sum[kx][q];
                __builtin_amdgcn_sched_barrier(0);
            }
            static_assert(NX + NG <= 3 * (S / 2), "staging groups");
            __syncthreads();
        }
    }

    float z = 0.f;  // NaN where a sum is not finite
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int q = 0; q < 16; ++q) z = __builtin_fmaf(acc[t][q], 0.f, z);
    if (__syncthreads_or(z != 0.f || any_lost(lost))) {
        clear();
        const int c = c0 + 32 * wa + l32, k = k0 + 32 * wb + l32;
        for (long r = lo; r < hi; ++r) {
            const WgRow w(a, r, 8 * S);
            image(w);
            // (four pixel pairs are in flight together)
            for (int px = 0; px < 8 * S; px += 8) {
                float gv[4], xv[4][9];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int x = w.x0 + px + 2 * u + h;
                    gv[u] = fetch(rg, k < a.K && x < a.W ? (uint32_t)(k * gplane + x) * 4u : kPast, (uint32_t)(w.y * a.W) * 4u);
#pragma unroll
                    for (int t = 0; t < 9; ++t)
                        xv[u][t] = fetch(rx, c < a.C && x + t % 3 < Wp ? (uint32_t)(c * xplane + x + t % 3) * 4u : kPast,
                                         (uint32_t)((w.y + t / 3) * Wp) * 4u);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int t = 0; t < 9; ++t) acc[t] = mfma(xv[u][t], gv[u], acc[t]);
            }
        }
    }
    // accumulator (t, q): c = 32 wa + 8 (q / 4) + 4 h + q % 4, co = 32 wb + l32 (slab-local)
    float* dst = a.part + (long)(blockIdx.y * gridDim.x + blockIdx.x) * 9 * 4096;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int ci = 32 * wa + 8 * (q >> 2) + 4 * h + (q & 3), co = 32 * wb + l32;
            dst[t * 4096 + ci * 64 + co] = acc[t][q];
        }
}

// wb[co][c][t] += the sum of the partials over splits.  Block: 64 consecutive partial
// elements x 4 split lanes; lane l sums splits l, l+4, ... in order, then the 4 lane sums
// are added in lane order (a fixed order: the result does not depend on scheduling).
__global__ __launch_bounds__(NT) void wreduce_kernel(const float* __restrict__ part, int nsplit, int nslab, int ktn, int C,
                                                     int K, float* __restrict__ wb) {
    __shared__ double red[4][64];
    const long total = (long)nslab * 9 * 4096;
    const int el = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const long q = (long)blockIdx.x * 64 + el;
    double s = 0.0;
    // unrolled so that several splits' loads are in flight (the sum keeps its order)
    if (q < total) {
#pragma unroll 8
        for (int sp = sl; sp < nsplit; sp += 4) s += part[(long)sp * total + q];
    }
    red[sl][el] = s;
    __syncthreads();
    if (sl != 0 || q >= total) return;
    s = ((red[0][el] + red[1][el]) + red[2][el]) + red[3][el];
    const int co_l = (int)(q & 63), ci_l = (int)((q >> 6) & 63);
    const long rest = q >> 12;
    const int t = (int)(rest % 9), slab = (int)(rest / 9);
    const int ct = slab / ktn, kt = slab - ct * ktn;
    const int c = ct * 64 + ci_l, k = kt * 64 + co_l;
    if (c >= C || k >= K) return;
    const long wi = ((long)k * C + c) * 9 + t;
    wb[wi] = (float)((double)wb[wi] + s);
}

// ------------------------------------------------------------------------------------------
// host
// ------------------------------------------------------------------------------------------
enum { ADJ, TAN, HVP };

struct Ptrs {
    float *loss, *lossb, *xp, *xpb, *w, *wb, *out, *outb;
    float *lossd, *lossbd, *xpd, *xpbd, *wd, *wbd, *outd, *outbd;
};

struct Dims {
    int N, C, K, H, W, Hp, Wp, Kpad, Cpad;
};

int32_t check(int64_t N, int64_t C, int64_t K, int64_t H, int64_t W, const char* fn, Dims& d) {
    if (N < 0 || C < 0 || K < 0 || H < 0 || W < 0) return set_error(STADE_HIP_EINVAL, "%s: negative size", fn);
    const double lim = 2147483647.0;
    // one image of a source and one weight set are read through buffer resources: < 2^31 bytes
    const double blim = 536870911.0;
    if ((double)C * (H + 2) * (W + 2) > blim || (double)K * H * W > blim || 9.0 * (C + 64) * (K + 64) > blim)
        return set_error(STADE_HIP_ERANGE, "%s: one image or the weights exceed 2^29 elements", fn);
    if ((double)N * C * (H + 2) * (W + 2) > lim || (double)N * K * H * W > lim || 9.0 * C * K > lim ||
        (double)N * ((K + 63) / 64) > 65535 || (double)N * ((C + 15) / 16) > 65535 || H > 200000 || W > 200000)
        return set_error(STADE_HIP_ERANGE, "%s: sizes out of range", fn);
    d.N = (int)N; d.C = (int)C; d.K = (int)K; d.H = (int)H; d.W = (int)W;
    d.Hp = d.H + 2; d.Wp = d.W + 2;
    d.Kpad = (d.K + 63) / 64 * 64;
    d.Cpad = (d.C + 63) / 64 * 64;
    const long tapblocks = (long)((d.W + 63) / 64) * ((d.H + 3) / 4) * d.N * (d.Kpad / 64);
    if (tapblocks * 2 > kPartialSlots) return set_error(STADE_HIP_ERANGE, "%s: sizes out of range", fn);
    return STADE_HIP_OK;
}

inline size_t up64(size_t n) { return (n + 63) / 64 * 64; }

template <int MODE>
hipError_t launch_tap(const TapArgs& a, const char* name, hipStream_t stream, unsigned& nblocks) {
    constexpr int TX = tap_width(MODE), NP = tap_sources(MODE);
    // one source: eight pixel rows a block where that still gives every CU one (two waves a
    // SIMD; the halo rows are a quarter of the patch instead of a half), otherwise four
    const long tiles = (long)((a.W + TX - 1) / TX) * a.N * (a.Rpad / RT);
    // (two sources: a chunk's sum is added to the total once)
    const bool fresh = (a.Cin + 1) / 2 < 6 * (NP == 1 ? tap_chunks(a.Cin) : 1);
    const bool tall = NP == 1 && !fresh && tiles * ((a.H + 7) / 8) >= gemm::device_cus();
    const int ty = tall ? 8 : 4;
    const dim3 grid((a.W + TX - 1) / TX, (a.H + ty - 1) / ty, a.N * (a.Rpad / RT));
    nblocks = grid.x * grid.y * grid.z;
    if constexpr (!tap_split(MODE)) {
        STADE_TIMED(name, stream, (tap32_kernel<MODE><<<grid, NT, 0, stream>>>(a)));
    } else if (fresh) {
        STADE_TIMED(name, stream, (tap_kernel<MODE, 4, true><<<grid, 256, 0, stream>>>(a)));
    } else if (!tall) {
        STADE_TIMED(name, stream, (tap_kernel<MODE, 4, false><<<grid, 256, 0, stream>>>(a)));
    } else if constexpr (NP == 1) {
        STADE_TIMED(name, stream, (tap_kernel<MODE, 8, false><<<grid, 512, 0, stream>>>(a)));
    }
    return hipGetLastError();
}

// cells a k group of the weight gradient's strips (8 S columns): 64 columns, or 32 where that
// leaves at least a sixth less of the columns empty.  Adjoint, 32 / 64 columns, us: W = 256
// 848 / 819, 224 717 / 711, 160 495 / 501, 96 220 / 228, 28 87 / 91
inline int wgrad_cells(int W) {
    const int s = (W + 31) / 32;
    return s % 2 && s <= 5 ? 4 : 8;
}
inline long wgrad_rows(const Dims& d) {
    const int width = 8 * wgrad_cells(d.W);
    return (long)((d.W + width - 1) / width) * d.H * d.N;
}

// wb += sum x0 g0 (+ sum x1 g1)
int32_t weight_grad(const Dims& d, const float* x0, const float* g0, const float* x1, const float* g1, float* part,
                    int nsplit, float* wb, const char* name, hipStream_t stream) {
    WgArgs a{};
    a.x[0] = x0; a.g[0] = g0; a.x[1] = x1; a.g[1] = g1;
    a.N = d.N; a.C = d.C; a.K = d.K; a.H = d.H; a.W = d.W;
    const int cells = wgrad_cells(d.W);
    a.ntx = (d.W + 8 * cells - 1) / (8 * cells);
    a.nrows = wgrad_rows(d) * (x1 ? 2 : 1);
    a.part = part;
    const int ctn = d.Cpad / 64, ktn = d.Kpad / 64;
    dim3 grid(ctn * ktn, nsplit);
    if (cells == 8) {
        STADE_TIMED(name, stream, (wgrad_kernel<8><<<grid, NT, 0, stream>>>(a)));
    } else {
        STADE_TIMED(name, stream, (wgrad_kernel<4><<<grid, NT, 0, stream>>>(a)));
    }
    STADE_LAUNCHED("conv3x3 wgrad_kernel");
    const long nr = (long)ctn * ktn * 9 * 4096;
    STADE_TIMED("conv_wreduce", stream,
                (wreduce_kernel<<<(unsigned)((nr + 63) / 64), NT, 0, stream>>>(part, nsplit, ctn * ktn, ktn, d.C, d.K, wb)));
    STADE_LAUNCHED("conv3x3 wreduce_kernel");
    return STADE_HIP_OK;
}

template <int MODE>
int32_t run(const Ptrs& p, const Dims& d, hipStream_t stream) {
    if (d.N == 0 || d.K == 0 || d.H == 0 || d.W == 0) return STADE_HIP_OK;
    WsCall call_(stream);
    Workspace* ws = call_.ws;
    if (!ws) return STADE_HIP_ENOMEM;
    // split weights (the adjoint's forward; xpb): 16-byte cells, 3 parts of 128 a tap, chunk and
    // row tile (in floats below).  The tangent's forward: both weight sets in fp32
    const size_t cf = MODE == ADJ ? (size_t)tap_chunks(d.C) * 9 * 128 * (d.Kpad / 64) : 0;
    const size_t cg = MODE == TAN ? 0 : (size_t)tap_chunks(d.K) * 9 * 128 * (d.Cpad / 64);
    const size_t n32 = MODE == ADJ ? 0 : up64((size_t)d.C * 9 * d.Kpad);
    const size_t nwf = cf * 12 + 2 * n32, nwg = cg * 12;
    // prep_kernel's grid: blocks of a row tile, row tiles
    const int rtf = cf ? d.Kpad / 64 : 0, rtg = cg ? d.Cpad / 64 : 0;
    const int bpt = (std::max(rtf ? tap_chunks(d.C) : 0, rtg ? tap_chunks(d.K) : 0) * 9 * 128 + NT - 1) / NT;
    const int two = MODE == ADJ ? 1 : 2;
    const size_t nflag = up64((size_t)two * (rtf + rtg) * bpt);
    const size_t nout = up64((size_t)d.N * d.K * d.H * d.W);
    const int ctn = d.Cpad / 64, ktn = d.Kpad / 64;
    // ctn is 0 when C = 0 (no weight gradient to form)
    const int nsplit = ctn == 0 ? 0 : (int)std::max(1L, std::min(wgrad_rows(d), (long)std::max(1, 256 / (ctn * ktn))));
    const size_t npart = (MODE == TAN || d.C == 0) ? 0 : (size_t)nsplit * ctn * ktn * 9 * 4096;
    const size_t total = nwf + (MODE == TAN ? 0 : two * nwg + two * nout) + nflag + npart;
    float* base = (float*)scratch(sizeof(float) * total + 256);
    if (!base) return scratch_error();
    float* wf = base;
    float* wg0 = wf + nwf;
    float* wg1 = wg0 + nwg;
    float* G = wg0 + (MODE == TAN ? 0 : two * nwg);
    float* GD = G + nout;
    int* flags = (int*)(G + (MODE == TAN ? 0 : two * nout));
    float* part = (float*)(flags + nflag);

    // weights in the tap kernels' forms
    if (n32 > 0) {
        STADE_TIMED("conv_prep", stream, (prep32_kernel<<<(unsigned)((n32 + NT - 1) / NT), NT, 0, stream>>>(p.w, p.wd, d.C, d.K, wf, wf + n32, d.Kpad)));
        STADE_LAUNCHED("conv3x3 prep32_kernel");
    }
    if (rtf + rtg > 0) {
        const PrepArgs a{{p.w, p.wd}, {(u32x4*)wf, nullptr}, {(u32x4*)wg0, (u32x4*)wg1}, flags, d.C, d.K, rtf};
        STADE_TIMED("conv_prep", stream, (prep_kernel<<<dim3(bpt, rtf + rtg, two), NT, 0, stream>>>(a)));
        STADE_LAUNCHED("conv3x3 prep_kernel");
    }
    // forward: out (and outd), loss (and lossd); adjoint seeds g (and gd), outb (and outbd) reset
    {
        TapArgs a{};
        a.src[0] = p.xp; a.src[1] = p.xpd;
        a.wt[0] = (u32x4*)wf; a.wt32[0] = wf; a.wt32[1] = wf + n32;
        a.w[0] = p.w; a.w[1] = p.wd; a.wr = 9L * d.C; a.wc = 9; a.flip = false;
        a.flags = flags; a.nflags = bpt;
        a.Cin = d.C; a.R = d.K; a.Rpad = d.Kpad; a.N = d.N;
        a.SH = d.Hp; a.SW = d.Wp; a.ofs = 0;
        a.H = d.H; a.W = d.W;
        a.o0 = p.out; a.o1 = p.outd;
        a.OH = d.H; a.OW = d.W; a.oofs = 0;
        a.g0 = G; a.g1 = GD; a.ob = p.outb; a.obd = p.outbd;
        a.lossb = p.lossb; a.lossbd = p.lossbd;
        a.partials = ws->partials;
        unsigned nblocks = 0;
        hipError_t e;
        if (MODE == ADJ) e = launch_tap<FWD_B>(a, "conv_fwd", stream, nblocks);
        else if (MODE == TAN) e = launch_tap<FWD_D>(a, "conv_fwd_d", stream, nblocks);
        else e = launch_tap<FWD_HV>(a, "conv_fwd_hv", stream, nblocks);
        if (e != hipSuccess) return check_hip(e, "conv3x3 tap_kernel (forward)");
        if (MODE == ADJ) {
            STADE_TIMED("conv_loss", stream, (loss_kernel<1><<<1, NT, 0, stream>>>(ws->partials, (int)nblocks, p.loss, nullptr)));
        } else {
            STADE_TIMED("conv_loss", stream, (loss_kernel<2><<<1, NT, 0, stream>>>(ws->partials, (int)nblocks, p.loss, p.lossd)));
        }
        STADE_LAUNCHED("conv3x3 loss_kernel");
    }
    if (MODE == TAN || d.C == 0) return STADE_HIP_OK;
    // wb += sum xp g;  HVP: wbd += sum (xpd g + xp gd)
    int32_t rc = weight_grad(d, p.xp, G, nullptr, nullptr, part, nsplit, p.wb, "conv_wgrad", stream);
    if (rc) return rc;
    if (MODE == HVP) {
        // both products of wbd in one launch over twice the rows
        rc = weight_grad(d, p.xpd, G, p.xp, GD, part, nsplit, p.wbd, "conv_wgrad2", stream);
        if (rc) return rc;
    }
    // xpb interior += flipped taps over g;  HVP: xpbd += wd g + w gd
    {
        TapArgs a{};
        a.src[0] = G; a.src[1] = GD;
        a.wt[0] = (u32x4*)wg0; a.wt[1] = (u32x4*)wg1;
        a.w[0] = p.w; a.w[1] = p.wd; a.wr = 9; a.wc = 9L * d.C; a.flip = true;
        a.flags = flags + (size_t)rtf * bpt; a.nflags = bpt; a.fset = (long)(rtf + rtg) * bpt;
        a.Cin = d.K; a.R = d.C; a.Rpad = d.Cpad; a.N = d.N;
        a.SH = d.H; a.SW = d.W; a.ofs = -1;
        a.H = d.H; a.W = d.W;
        a.o0 = p.xpb; a.o1 = p.xpbd;
        a.OH = d.Hp; a.OW = d.Wp; a.oofs = 1;
        unsigned nblocks = 0;
        hipError_t e = MODE == ADJ ? launch_tap<DG_B>(a, "conv_dgrad", stream, nblocks)
                                   : launch_tap<DG_HV>(a, "conv_dgrad_hv", stream, nblocks);
        if (e != hipSuccess) return check_hip(e, "conv3x3 tap_kernel (xpb)");
    }
    // xpb frame
    {
        BorderArgs b{p.w, p.wd, G, GD, p.xpb, p.xpbd, d.N, d.C, d.K, d.H, d.W};
        const dim3 grid((std::max(d.W + 2, d.H) + BSEG - 1) / BSEG, 4, d.N * ((d.C + BCG - 1) / BCG));
        if (MODE == ADJ) {
            STADE_TIMED("conv_border", stream, (border_kernel<false><<<grid, NT, 0, stream>>>(b)));
        } else {
            STADE_TIMED("conv_border", stream, (border_kernel<true><<<grid, NT, 0, stream>>>(b)));
        }
        STADE_LAUNCHED("conv3x3 border_kernel");
    }
    return STADE_HIP_OK;
}

}  // namespace
}  // namespace stade

using namespace stade;

extern "C" {

int32_t stade_hip_conv3x3_b(float* loss, const float* lossb, const float* xp, float* xpb, const float* w, float* wb,
                            float* out, float* outb, int64_t i_nb, int64_t i_c, int64_t i_k, int64_t i_h, int64_t i_w,
                            hipStream_t stream) {
    Dims d;
    if (int32_t rc = check(i_nb, i_c, i_k, i_h, i_w, "stade_hip_conv3x3_b", d)) return rc;
    Ptrs p{};
    p.loss = loss; p.lossb = (float*)lossb; p.xp = (float*)xp; p.xpb = xpb; p.w = (float*)w; p.wb = wb; p.out = out; p.outb = outb;
    return run<ADJ>(p, d, stream);
}

int32_t stade_hip_conv3x3_d(float* loss, float* lossd, const float* xp, const float* xpd, const float* w, const float* wd,
                            float* out, float* outd, int64_t i_nb, int64_t i_c, int64_t i_k, int64_t i_h, int64_t i_w,
                            hipStream_t stream) {
    Dims d;
    if (int32_t rc = check(i_nb, i_c, i_k, i_h, i_w, "stade_hip_conv3x3_d", d)) return rc;
    Ptrs p{};
    p.loss = loss; p.lossd = lossd; p.xp = (float*)xp; p.xpd = (float*)xpd; p.w = (float*)w; p.wd = (float*)wd;
    p.out = out; p.outd = outd;
    return run<TAN>(p, d, stream);
}

int32_t stade_hip_conv3x3_hv(float* loss, const float* lossb, const float* xp, float* xpb, const float* w, float* wb,
                             float* out, float* outb, int64_t i_nb, int64_t i_c, int64_t i_k, int64_t i_h, int64_t i_w,
                             float* lossd, const float* lossbd, const float* xpd, float* xpbd, const float* wd, float* wbd,
                             float* outd, float* outbd, hipStream_t stream) {
    Dims d;
    if (int32_t rc = check(i_nb, i_c, i_k, i_h, i_w, "stade_hip_conv3x3_hv", d)) return rc;
    Ptrs p{};
    p.loss = loss; p.lossb = (float*)lossb; p.xp = (float*)xp; p.xpb = xpb; p.w = (float*)w; p.wb = wb; p.out = out; p.outb = outb;
    p.lossd = lossd; p.lossbd = (float*)lossbd; p.xpd = (float*)xpd; p.xpbd = xpbd; p.wd = (float*)wd; p.wbd = wbd;
    p.outd = outd; p.outbd = outbd;
    return run<HVP>(p, d, stream);
}

}  // extern "C"
