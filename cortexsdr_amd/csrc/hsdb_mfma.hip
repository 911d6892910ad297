// hsdb_mfma.hip — batched (M >= 2) block-coded product Y = W.X on gfx950 matrix cores.
//
// Path (cortexSDR tree): HierarchicalSDRStrategy::matmulRowMajor with batch > 1
// (strategies/HierarchicalSDRStrategy.cpp:1257-1338), block-coded as in research
// exp_c_kernel/benchmark.py:106-130. W is never stored: 64-column tiles of a row strip are
// decoded to fp16, in LDS or in registers, and multiplied against the matching 64 x M slice of X.
//
// Decode: W[r][k] = g0 * sum_j (c_j * g_j / g0) * D[idx_j][k] over the row's slots (g0 the
// largest stage gain), with the dictionary held in LDS as fp16 (K <= 1024 atoms: 128 KiB):
// packed fp16 fused multiply-adds (v_pk_fma_f16, two weights per lane instruction) over the
// slots in order, fp32 accumulation on the matrix cores (v_mfma_f32_16x16x32_f16; gfx950 runs it
// at full rate), and g0 scales the fp32 result. X is fp16 as given, or split into fp16 hi + lo
// parts for fp32 input (two MFMAs). The fp16 dictionary and the fp16 accumulation over the slots
// keep the product within ~5e-4 relative L2 of the fp32 decode (the path's bar is 1e-3).
//
// Layout. Every 64-long k range (one block column) is stored permuted (kperm64), in both the
// LDS dictionary and the transposed X, so that lane l (q = l/16) reads 16 consecutive
// positions 16q .. 16q + 15 as one contiguous 32-byte run; the block's two 32-deep MFMA steps
// take positions 16q + 8c .. + 7 (c = 0, 1) as lane group q's 8 k values in both operands
// (any common bijection of k leaves the product unchanged). The result: lane l holds rows
// 4(l/16) + i (i = 0..3) of column l % 16.
//
// Launches: an init kernel (Y = bias (+ Y when accumulating) + the fp32 edge strip times X,
// and X transposed to fp16 operand granules with the permutation, in the workspace), then one
// persistent kernel: the (row strip, block column) units of all matrices are split in
// contiguous ranges over one workgroup per CU, and each strip's partial sums are added into Y
// with device-scope float atomics. Two or more 16-column tiles: mfma_dec_kernel. One (M <= 16):
// with fp16 X and 4 or 8 slots the dictionary route (qroute_kernel: no weight is decoded, each
// unit's Q_b = D . X_b is formed on the matrix cores and every row gathers its slots' rows of Q_b
// from LDS), else mfma_kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "hsdb_impl.hpp"

namespace {

using csdr::set_error;

constexpr int kThreads = 256;  // 4 waves
constexpr int kMaxAtoms = 1024;
constexpr int kMaxMTile = 256;
constexpr int kGroup = 8;
constexpr int kMfmaMinM = 2;  // smallest batch routed to this path (M = 1: the P-path GEMV)

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct MDesc {
    const uint32_t* codes;
    const _Float16* dict16p;  // K x 64 fp16, rows in kperm64 order
    const float* edge;
    const void* x;
    float* y;
    const float* bias;
    _Float16* xt;  // Mpad x C_full fp16 (hi), then Mpad x C_full (lo) for fp32 X
    int R, K, NB, NBc, slots, Ce, C_full;
    int u_base, u_count;  // units (row strip x block column) [u_base, u_base + u_count)
    float g0;             // the largest stage gain: scales the accumulated products
    uint32_t grel[16];    // slot j's gain relative to g0 as an fp16 pair (g_j / g0, same)
};

struct MParams {
    MDesc m[kGroup];
    int G, M, Mpad, x_f16, accumulate, total_units;
    int tm;  // token-major X (M x C) and Y (M x R)
    int m0;  // first column of this launch (the launch covers 16 * NT columns)
};

// Transposed X: 16-byte granule g (8 permuted k positions) of block column b and column m, in the
// order in which a wave loads a 16-column operand: [b][m / 16][g % 2][g / 2][m % 16], so that
// one load instruction reads 1 KiB in a row. In halves from xt (the lo part xt_part on).
__device__ __forceinline__ size_t xt_granule(const MParams& p, int b, int m, int g) {
    return ((((size_t)b * (p.Mpad >> 4) + (m >> 4)) * 2 + (g & 1)) * 64 + (g >> 1) * 16 + (m & 15)) * 8;
}
__device__ __forceinline__ size_t xt_part(const MParams& p, const MDesc& d) {
    return (size_t)p.Mpad * d.C_full;
}

// ---- init: Y start values, and X transposed into operand granules. blockIdx.x below xwgs: one
// block column and MW columns of X through LDS (read along X's rows, written granule by
// granule; straight from X to the granules each lane's 8 values were 8 separate 2-byte loads
// and its 16-byte store a line of its own). The others: Y. Bound by round trips where the matrix
// is small, so all of a thread's X values are loaded before the first is used (896 x 896, 65
// columns: 8.6 us with four rounds of four loads, 4.0 here), and by the edge strip's operands
// where there is one, so a thread takes four outputs that share the coalesced operand once there
// are more than kEdgeWide of them (14336 x 300, 256 columns: 94 us an output a thread and at most
// 1024 workgroups, 34 here; with fewer, one: 9 columns 18.0 us a call, 24.3 with four).
constexpr size_t kEdgeWide = 1 << 20;

template <typename XT, int MW>
__device__ __forceinline__ void init_x(const MParams& p, const MDesc& d, int wg, float (*tile)[65]) {
    constexpr int kPer = 64 * MW / kThreads;  // values per thread
    const int tid = threadIdx.x, M = p.M;
    const int nmt = p.Mpad / MW;
    const int b = wg / nmt, m0 = (wg - b * nmt) * MW;
    if (b >= d.NB) return;
    const XT* x = static_cast<const XT*>(d.x);
    // feature-major: threads along a feature's columns; token-major: along a column's features
    // (at clamped columns)
    const size_t C = d.C_full + d.Ce;
    float v[kPer];
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int i = tid + e * kThreads;
        const int k = p.tm ? (i & 63) : i / MW, c = p.tm ? (i >> 6) : i & (MW - 1);
        const int m = min(m0 + c, M - 1);
        v[e] = (float)x[p.tm ? (size_t)m * C + b * 64 + k : (size_t)(b * 64 + k) * M + m];
    }
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int i = tid + e * kThreads;
        const int k = p.tm ? (i & 63) : i / MW, c = p.tm ? (i >> 6) : i & (MW - 1);
        tile[k][c] = m0 + c < M ? v[e] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int i0 = 0; i0 < MW * 8; i0 += kThreads) {
        const int i = i0 + tid;
        if (MW * 8 < kThreads && i >= MW * 8) break;
        const int c = i & (MW - 1), g = i / MW;
        _Float16 hi[8], lo[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float xv = tile[csdr::kperm64(g * 8 + j)][c];
            hi[j] = (_Float16)xv;
            lo[j] = (_Float16)(xv - (float)hi[j]);
        }
        const size_t o = xt_granule(p, b, m0 + c, g);
        *reinterpret_cast<u32x4*>(d.xt + o) = __builtin_bit_cast(u32x4, hi);
        if (sizeof(XT) == 4)
            *reinterpret_cast<u32x4*>(d.xt + xt_part(p, d) + o) = __builtin_bit_cast(u32x4, lo);
    }
}

// Y = (Y +) bias + edge . X: OUT rows of a column (row-major Y: threads along the columns) or
// columns of a row (token-major: along the rows), each sum in feature order.
template <typename XT, int OUT>
__device__ __forceinline__ void init_edge(const MParams& p, const MDesc& d, size_t t0,
                                          size_t stride) {
    const int M = p.M, R = d.R, Ce = d.Ce;
    const XT* x = static_cast<const XT*>(d.x);
    const size_t C = d.C_full + Ce;
    const int fast = p.tm ? R : M, slow = p.tm ? M : R;
    const size_t n = (size_t)((slow + OUT - 1) / OUT) * fast;
    for (size_t t = t0; t < n; t += stride) {
        const int f = (int)(t % fast), s0 = (int)(t / fast) * OUT;
        const float* e[OUT];
        const XT* xv[OUT];
        float s[OUT];
#pragma unroll
        for (int q = 0; q < OUT; ++q) {  // past the end the last one (not stored)
            const int sq = min(s0 + q, slow - 1), r = p.tm ? f : sq, m = p.tm ? sq : f;
            e[q] = d.edge + (size_t)r * Ce;
            xv[q] = x + (p.tm ? (size_t)m * C + d.C_full : (size_t)d.C_full * M + m);
            s[q] = 0.0f;
        }
        const size_t xs = p.tm ? 1 : M;
#pragma unroll 8
        for (int cc = 0; cc < Ce; ++cc)
            if (p.tm) {
                const float ev = e[0][cc];
#pragma unroll
                for (int q = 0; q < OUT; ++q) s[q] = fmaf(ev, (float)xv[q][cc], s[q]);
            } else {
                const float x0 = (float)xv[0][cc * xs];
#pragma unroll
                for (int q = 0; q < OUT; ++q) s[q] = fmaf(e[q][cc], x0, s[q]);
            }
#pragma unroll
        for (int q = 0; q < OUT; ++q) {
            if (s0 + q >= slow) break;
            float& y = d.y[(size_t)(s0 + q) * fast + f];
            float v = p.accumulate ? y : 0.0f;
            if (d.bias) v += d.bias[p.tm ? f : s0 + q];
            y = v + s[q];
        }
    }
}

template <typename XT, int MW>
__global__ __launch_bounds__(kThreads) void mfma_init_kernel(MParams p, int xwgs) {
    __shared__ float tile[64][65];
    const MDesc& d = p.m[blockIdx.y];
    if ((int)blockIdx.x < xwgs) {
        init_x<XT, MW>(p, d, blockIdx.x, tile);
        return;
    }
    if (p.accumulate && !d.bias && d.Ce == 0) return;  // Y stays as it is
    const size_t ny = (size_t)d.R * p.M;
    const size_t stride = (size_t)(gridDim.x - xwgs) * kThreads;
    const size_t t0 = (size_t)(blockIdx.x - xwgs) * kThreads + threadIdx.x;
    if (d.Ce > 0) {
        if (ny > kEdgeWide) init_edge<XT, 4>(p, d, t0, stride);
        else init_edge<XT, 1>(p, d, t0, stride);
        return;
    }
    for (size_t t = t0; t < ny; t += stride) {
        float v = p.accumulate ? d.y[t] : 0.0f;
        if (d.bias) v += d.bias[p.tm ? t % d.R : t / p.M];
        d.y[t] = v;
    }
}

__device__ __forceinline__ int find_matrix(const MParams& p, int u, int g) {
    if (g >= 0 && u >= p.m[g].u_base && u < p.m[g].u_base + p.m[g].u_count) return g;
    g = 0;
    while (g + 1 < p.G && u >= p.m[g + 1].u_base) ++g;
    return g;
}

// ---- main, one 16-column tile (M <= 16) where the dictionary route below does not run (fp32 X,
// 16 slots): 16 waves, each decoding its own 16-row strips' tiles into the A operands of the
// matrix-core steps. XS: fp32-X split. The codes and X operands of unit u + 1 are loaded into
// registers while unit u is decoded and multiplied (X straight from the transposed X: global
// memory, L1 / L2 hits, as the waves all take the same unit sequence), so the units need no
// barriers. The slots' dictionary reads are issued four at a time before their multiply-adds.
template <bool XS, int SLOTS>
__global__ __launch_bounds__(1024) void mfma_kernel(MParams p) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    constexpr int W = 16;
    constexpr int CW = SLOTS / 4;  // 16-byte code pieces per tile
    constexpr int kThreads = W * 64;
    constexpr int kStripRows = W * 16;
    extern __shared__ __attribute__((aligned(16))) _Float16 smem16[];
    constexpr int NP = XS ? 2 : 1;           // X parts (fp32 X: hi, lo)
    constexpr int LB = 4;
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int q = lane >> 4, rl = lane & 15;
    const int U = p.total_units;
    const int u0 = (int)((long long)U * blockIdx.x / gridDim.x);
    const int u1 = (int)((long long)U * (blockIdx.x + 1) / gridDim.x);
    if (u0 >= u1) return;
    // K x 64; 16-byte granule g of atom a at g ^ ((a >> 1) & 7): rows are 128 bytes, so
    // without it the 16 lanes of one k segment would meet in two bank groups
    _Float16* Ds = smem16;
    const int M = p.M;

    floatx4 acc;
    u32x4 xb[NP][2];  // prefetched X operands of the next unit
    u32x4 cr[CW];     // prefetched code words of the next unit
    int ng = -1, nstrip = 0, nb = 0;  // the prefetched unit

    auto prefetch = [&](int u) {
        ng = find_matrix(p, u, ng);
        const MDesc& d = p.m[ng];
        const int lu = u - d.u_base;
        nstrip = lu / d.NB;
        nb = lu - nstrip * d.NB;
        // lane (column rl, group q): granules 2q and 2q + 1 of the block
#pragma unroll
        for (int part = 0; part < NP; ++part)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                xb[part][c] = *reinterpret_cast<const u32x4*>(
                    d.xt + part * xt_part(p, d) + xt_granule(p, nb, p.m0 + rl, 2 * q + c));
        const int r = min(nstrip * kStripRows + wave * 16 + rl, d.R - 1);
        const uint32_t* cw = d.codes + csdr::tile_word_offset(r, nb, d.R, d.NB, d.NBc, d.slots);
#pragma unroll
        for (int j4 = 0; j4 < CW; ++j4) cr[j4] = *reinterpret_cast<const u32x4*>(cw + j4 * 4);
    };

    auto flush = [&](int g, int strip) {
        const MDesc& d = p.m[g];
        const int rbase = strip * kStripRows + wave * 16 + q * 4;
        const int m = p.m0 + rl;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = rbase + i;
            if (r < d.R && m < M)
                __hip_atomic_fetch_add(d.y + (p.tm ? (size_t)m * d.R + r : (size_t)r * M + m),
                                       acc[i] * d.g0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };

    int cur_g = -1, cur_strip = -1;
    prefetch(u0);
    for (int u = u0; u < u1; ++u) {
        const int g = ng, strip = nstrip;
        const MDesc& d = p.m[g];
        if (g != cur_g || strip != cur_strip) {
            if (cur_strip >= 0) flush(cur_g, cur_strip);
            acc = floatx4{0.f, 0.f, 0.f, 0.f};
            if (g != cur_g) {
                // the matrix's fp16 dictionary -> LDS (16-byte granules, 8 loads in flight)
                __syncthreads();
                const int n = d.K * 8;
                for (int i0 = 0; i0 < n; i0 += kThreads * 8) {
                    u32x4 v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        v[j] = *reinterpret_cast<const u32x4*>(
                            d.dict16p + (size_t)min(i0 + j * kThreads + tid, n - 1) * 8);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int i = i0 + j * kThreads + tid;
                        const int a = i >> 3, gr = i & 7;
                        if (i < n)
                            *reinterpret_cast<u32x4*>(Ds + (size_t)a * 64 +
                                                      ((gr ^ ((a >> 1) & 7)) * 8)) = v[j];
                    }
                }
                __syncthreads();
            }
            cur_g = g;
            cur_strip = strip;
        }
        u32x4 xc[NP][2];
#pragma unroll
        for (int part = 0; part < NP; ++part)
#pragma unroll
            for (int c = 0; c < 2; ++c) xc[part][c] = xb[part][c];
        u32x4 cc[CW];
#pragma unroll
        for (int j4 = 0; j4 < CW; ++j4) cc[j4] = cr[j4];
        if (u + 1 < u1) prefetch(u + 1);
        // decode this lane's 16 k values of its row: per slot the coefficient as an fp16 pair
        // (times the slot's gain relative to the largest) and 8 packed fp16 FMAs over the atom's
        // two 16-byte granules, accumulated in place as the two 8-value A operands
        h2 w[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) w[t] = h2{(_Float16)0.0f, (_Float16)0.0f};
#pragma unroll
        for (int j0 = 0; j0 < SLOTS; j0 += LB) {
            // the batch's LB atoms: both 16-byte granules of each read before any is used
            u32x4 lo[LB], hi[LB];
#pragma unroll
            for (int jj = 0; jj < LB; ++jj) {
                const uint32_t word = cc[(j0 + jj) >> 2][(j0 + jj) & 3];
                const uint32_t at = word & 0x7FFFu;
                const uint32_t sw = (at >> 1) & 7;
                const _Float16* drow = Ds + at * 64;
                lo[jj] = *reinterpret_cast<const u32x4*>(drow + (((2 * q) ^ sw) * 8));
                hi[jj] = *reinterpret_cast<const u32x4*>(drow + (((2 * q + 1) ^ sw) * 8));
            }
#pragma unroll
            for (int jj = 0; jj < LB; ++jj) {
                const int j = j0 + jj;
                const uint32_t word = cc[j >> 2][j & 3];
                // (c, c): the word's high half in both halves
                const h2 c2 =
                    __builtin_bit_cast(h2, __builtin_amdgcn_perm(word, word, 0x07060706u)) *
                    __builtin_bit_cast(h2, d.grel[j]);
                // (vector elements go through a scalar: bit-casting a subscripted vector
                // element directly reads element 0 whatever the subscript)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint32_t el = lo[jj][t], eh = hi[jj][t];
                    w[t] = __builtin_elementwise_fma(c2, __builtin_bit_cast(h2, el), w[t]);
                    w[4 + t] = __builtin_elementwise_fma(c2, __builtin_bit_cast(h2, eh), w[4 + t]);
                }
            }
        }
        // two 32-deep steps over the block column: lane group q holds positions 16 q + 8 c ..
        // + 7 of the permuted k order in step c, in both operands
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const u32x4 v = {__builtin_bit_cast(uint32_t, w[4 * c]),
                             __builtin_bit_cast(uint32_t, w[4 * c + 1]),
                             __builtin_bit_cast(uint32_t, w[4 * c + 2]),
                             __builtin_bit_cast(uint32_t, w[4 * c + 3])};
#pragma unroll
            for (int part = 0; part < NP; ++part)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(half8, v), __builtin_bit_cast(half8, xc[part][c]), acc, 0,
                    0, 0);
        }
    }
    if (cur_strip >= 0) flush(cur_g, cur_strip);
}

// ---- main, one 16-column tile (M <= 16): the dictionary route. Per unit (256-row strip,
// block column b) the workgroup forms Q_b = D . X_b (K atoms x 16 columns) on the matrix
// cores and each row then gathers its slots' rows of Q_b from LDS:
//   y[r][m] += g0 * sum_j (c_j * g_j / g0) * Q_b[idx_j][m],
// 32 bytes of LDS per (row, slot) where decoding the weights reads the atom's 128.
// - The dictionary lives in registers for the whole launch: 16 waves x 64 atoms, each wave's
//   atoms as the B operands of v_mfma_f32_16x16x32_f16 (8 x 16 bytes per lane), so LDS holds
//   only Q (two 32 KiB buffers: Q_{u+1} is formed while unit u is gathered, one barrier per
//   unit).
// - Q^T = X_b^T . D^T: lane (n = l % 16, q = l / 16) of a 16-atom tile ends with atom n's
//   columns 4q .. 4q + 3, one 8-byte LDS store. Q rows are 32 bytes of four 8-byte pieces,
//   piece q at q ^ 2 on atoms with bit 2 set, so that the gather's 16-byte halves stay whole
//   and its reads of random rows spread over all bank groups. Q is stored in fp16 (fp32
//   accumulation; |Q| <= ||x_b|| for unit-norm atoms).
// - Gather: lane (row l % 16 of the wave's 16, slot group q) takes slots q S/4 .. of its row
//   (S/4 code words, no lane loads another's) and all 16 columns (two 16-byte reads per slot,
//   fp16 x fp16 -> fp32 multiply-adds). When the strip ends the four slot groups of a row are
//   reduce-scattered by shuffles and the wave's 16 x 16 tile goes through LDS, so that each
//   device-scope atomic instruction into Y covers four whole rows.
// - Loads: each unit's code words and the X operands of the unit after it form one bundle,
//   issued two units ahead into a register ring (the wait for a bundle's X also covers every
//   earlier load, so both streams share one depth). Every load is unconditional (see below).
// A unit's position: strip, block column b, and the chunk holding b (first column b0,
// width nbc), advanced one unit at a time within one matrix whose geometry the caller keeps
// in registers (reading it from the kernel arguments inside the loop puts a scalar load and
// its wait, which also drains every LDS operation in flight, into every unit).
struct UnitCursor {
    int strip, b, b0, nbc;
};

struct SegGeom {
    int NB, NBc, R, nstrips, nfull;  // nfull: columns in full chunks
};

__device__ __forceinline__ void cursor_chunk(const SegGeom& s, UnitCursor& c) {
    if (c.b < s.nfull) {
        c.b0 = c.b & ~(s.NBc - 1);
        c.nbc = s.NBc;
        return;
    }
    uint32_t cc, b0, nbc;
    csdr::chunk_of((uint32_t)c.b, (uint32_t)s.NB, (uint32_t)s.NBc, cc, b0, nbc);
    c.b0 = (int)b0;
    c.nbc = (int)nbc;
}

// Next unit of the same matrix (wrapping past its last unit, so a cursor always names valid
// codes and X: the pipeline's loads past a range's end stay unconditional and in bounds).
__device__ __forceinline__ void cursor_next(const SegGeom& s, UnitCursor& c) {
    if (++c.b == s.NB) {
        c.b = 0;
        if (++c.strip == s.nstrips) c.strip = 0;
    }
    if (c.b == 0 || c.b >= c.b0 + c.nbc) cursor_chunk(s, c);
}

template <int SLOTS, bool XS>
__global__ __launch_bounds__(1024) void qroute_kernel(MParams p) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    constexpr int SPL = SLOTS / 4;   // slots per lane
    constexpr int NP = XS ? 2 : 1;   // X parts (fp32 X: hi, lo)
    constexpr int QB = kMaxAtoms * 16;  // fp16 per Q buffer
    typedef typename std::conditional<SPL == 4, u32x4,
            typename std::conditional<SPL == 2, uint2, uint32_t>::type>::type cword_t;
    extern __shared__ __attribute__((aligned(16))) _Float16 smem16[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int q = lane >> 4, rl = lane & 15;
    const int U = p.total_units;
    const int u0 = (int)((long long)U * blockIdx.x / gridDim.x);
    const int u1 = (int)((long long)U * (blockIdx.x + 1) / gridDim.x);
    if (u0 >= u1) return;
    const int M = p.M;

    // the units of one matrix at a time: its atoms in registers, then a pipeline over its units
    // in which every load is unconditional (a load under a branch makes the compiler's wait
    // counts assume the worst at the join, which drained the pipeline every unit)
    for (int s0 = u0; s0 < u1;) {
        const int g = find_matrix(p, s0, -1);
        const MDesc& d = p.m[g];
        const int s1 = min(u1, d.u_base + d.u_count);
        half8 dreg[4][2];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int a = min(wave * 64 + t * 16 + rl, d.K - 1);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                dreg[t][c] = __builtin_bit_cast(
                    half8, *reinterpret_cast<const u32x4*>(d.dict16p + (size_t)a * 64 + (2 * q + c) * 8));
        }
        // this lane's slots' gains relative to g0 (fp16), chosen from uniform loads
        _Float16 gl[SPL];
#pragma unroll
        for (int j = 0; j < SPL; ++j) {
            const uint32_t a0 = d.grel[j], a1 = d.grel[SPL + j], a2 = d.grel[2 * SPL + j],
                           a3 = d.grel[3 * SPL + j];
            const uint32_t w = q == 0 ? a0 : (q == 1 ? a1 : (q == 2 ? a2 : a3));
            gl[j] = __builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu));
        }
        const _Float16* xt0 = d.xt + xt_granule(p, 0, rl, 2 * q);
        const size_t nxt = xt_part(p, d);
        const int K = d.K;
        SegGeom sg;
        sg.NB = d.NB;
        sg.NBc = d.NBc;
        sg.R = d.R;
        sg.nstrips = (d.R + 255) >> 8;
        sg.nfull = d.NB & ~(d.NBc - 1);
        const uint32_t* codes = d.codes;
        float* y = d.y;
        const float g0 = d.g0;

        u32x4 xr[2][NP][2];
        cword_t cr[2];
        float ya[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) ya[e] = 0.0f;

        auto load_x = [&](const UnitCursor& c, u32x4 (&dst)[NP][2]) {
            const _Float16* src = xt0 + (size_t)c.b * 1024;  // Mpad = 16: 2 KiB a block
#pragma unroll
            for (int part = 0; part < NP; ++part)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc)
                    dst[part][cc] = *reinterpret_cast<const u32x4*>(src + part * nxt + cc * 512);
        };
        auto load_codes = [&](const UnitCursor& c, cword_t& dst) {
            const int r = min(c.strip * 256 + wave * 16 + rl, sg.R - 1);
            const size_t w =
                ((size_t)c.b0 * sg.R + (size_t)r * c.nbc + (c.b - c.b0)) * SLOTS + q * SPL;
            dst = *reinterpret_cast<const cword_t*>(codes + w);
        };
        // Q of a unit from its X operands xo, two atom tiles (t0, t0 + 1) at a time, each pair
        // then stored into buffer buf
        auto q_mfma = [&](const u32x4 (&xo)[NP][2], floatx4 (&acc)[2], int t0) {
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                for (int part = 0; part < NP; ++part)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(half8, xo[part][cc]), dreg[t0 + t][cc], acc[t], 0, 0, 0);
        };
        auto q_store = [&](const floatx4 (&acc)[2], int buf, int t0) {
            _Float16* Qb = smem16 + (size_t)buf * QB;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int a = wave * 64 + (t0 + t) * 16 + rl;
                if (wave * 64 + (t0 + t) * 16 < K) {  // (uniform per wave)
                    const h2 lo = h2{(_Float16)acc[t][0], (_Float16)acc[t][1]};
                    const h2 hi = h2{(_Float16)acc[t][2], (_Float16)acc[t][3]};
                    const uint2 v = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
                    // 8-byte piece q of the 32-byte row at q ^ 2 (a bit 2): the two halves read
                    // by the gather stay 16-byte granules, spread over all bank groups
                    *reinterpret_cast<uint2*>(Qb + (size_t)a * 16 + ((q ^ ((a >> 1) & 2)) * 4)) = v;
                }
            }
        };
        auto words_of = [&](const cword_t& cw, uint32_t (&words)[SPL]) {
            if constexpr (SPL == 1) {
                words[0] = cw;
            } else if constexpr (SPL == 2) {
                words[0] = cw.x;
                words[1] = cw.y;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) words[j] = cw[j];
            }
        };
        auto g_read = [&](const uint32_t (&words)[SPL], int buf, u32x4 (&h)[SPL][2]) {
            const _Float16* Qb = smem16 + (size_t)buf * QB;
#pragma unroll
            for (int j = 0; j < SPL; ++j) {
                const uint32_t at = words[j] & 0x7FFFu;
                const uint32_t sw = (at >> 2) & 1;
                const _Float16* row = Qb + at * 16;
                h[j][0] = *reinterpret_cast<const u32x4*>(row + sw * 8);
                h[j][1] = *reinterpret_cast<const u32x4*>(row + (sw ^ 1) * 8);
            }
        };
        // the gather's multiply-adds of slot j
        auto g_acc = [&](const uint32_t (&words)[SPL], const u32x4 (&h)[SPL][2], int j) {
            const _Float16 cf = __builtin_bit_cast(_Float16, (uint16_t)(words[j] >> 16)) * gl[j];
            const float cfl = (float)cf;
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t dw = h[j][half][k];
                    const h2 pr = __builtin_bit_cast(h2, dw);
                    ya[half * 8 + 2 * k] = fmaf(cfl, (float)pr[0], ya[half * 8 + 2 * k]);
                    ya[half * 8 + 2 * k + 1] = fmaf(cfl, (float)pr[1], ya[half * 8 + 2 * k + 1]);
                }
        };
        // the strip's row sums: the four slot groups of a row summed by shuffles, then the
        // wave's 16 x 16 tile through LDS so that each atomic instruction covers four whole rows
        // of Y (token-major: four whole columns) instead of 16 scattered 16-byte pieces
        auto flush = [&](int strip) {
            float* T = reinterpret_cast<float*>(smem16 + 2 * (size_t)QB) + wave * 256;
            // reduce-scatter over the four slot groups (lanes l, l ^ 16, l ^ 32, l ^ 48): lane q
            // ends with columns 8 (q & 1) + 4 (q >> 1) .. + 3 of its row
            const bool b = q & 1, c = q >> 1;
            float t[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float keep = b ? ya[8 + k] : ya[k];
                const float send = b ? ya[k] : ya[8 + k];
                t[k] = keep + __shfl_xor(send, 16, 64);
            }
            float4 w;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float keep = c ? t[4 + k] : t[k];
                const float send = c ? t[k] : t[4 + k];
                w[k] = keep + __shfl_xor(send, 32, 64);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) ya[e] = 0.0f;
            *reinterpret_cast<float4*>(T + rl * 16 + 8 * (q & 1) + 4 * (q >> 1)) = w;
            const int r0 = strip * 256 + wave * 16;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // row-major: rows 4i + lane / 16, column lane % 16; token-major: rows lane % 16,
                // column 4i + lane / 16
                const int rr = p.tm ? rl : 4 * i + q;
                const int m = p.tm ? 4 * i + q : rl;
                const float v = T[rr * 16 + m];
                const int r = r0 + rr;
                if (r < sg.R && m < M)
                    __hip_atomic_fetch_add(y + (p.tm ? (size_t)m * sg.R + r : (size_t)r * M + m),
                                           v * g0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };

        // cursors: gathered unit v, its successor (Q formed), the next bundle's codes (v + 2)
        // and X (v + 3); bundle w = (codes of w, X of w + 1), two in flight
        UnitCursor cg;
        {
            const int lu = s0 - d.u_base;
            cg.strip = lu / sg.NB;
            cg.b = lu - cg.strip * sg.NB;
            cursor_chunk(sg, cg);
        }
        UnitCursor cm = cg;
        cursor_next(sg, cm);
        UnitCursor cc = cg, cx = cm;
        {
            u32x4 x0[NP][2];
            load_x(cg, x0);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                load_x(cx, xr[i]);
                load_codes(cc, cr[i]);
                cursor_next(sg, cx);
                cursor_next(sg, cc);
            }
#pragma unroll
            for (int t0 = 0; t0 < 4; t0 += 2) {
                floatx4 acc[2];
                q_mfma(x0, acc, t0);
                q_store(acc, 0, t0);
            }
        }
        __syncthreads();
        // per unit: the gather's LDS reads of Q_v, the matrix-core steps of Q_{v+1} while they
        // are in flight, the gather's multiply-adds, then Q_{v+1} into the other buffer
        auto step = [&](int v, auto S) {
            constexpr int sl = decltype(S)::value;
            const bool more = v + 1 < s1;
            uint32_t words[SPL];
            words_of(cr[sl], words);
            u32x4 h[SPL][2];
            g_read(words, (v - s0) & 1, h);
            // tile pairs interleaved with the slots' multiply-adds
            constexpr int JP = SPL >= 2 ? SPL / 2 : 1;  // slots per tile pair
#pragma unroll
            for (int t0 = 0; t0 < 4; t0 += 2) {
                floatx4 acc[2];
                if (more) q_mfma(xr[sl], acc, t0);
#pragma unroll
                for (int jj = 0; jj < JP; ++jj) {
                    const int j = (t0 / 2) * JP + jj;
                    if (j < SPL) g_acc(words, h, j);
                }
                if (more) q_store(acc, (v + 1 - s0) & 1, t0);
            }
            load_x(cx, xr[sl]);
            load_codes(cc, cr[sl]);
            if (!more || cm.strip != cg.strip) flush(cg.strip);
            cg = cm;
            cursor_next(sg, cm);
            cursor_next(sg, cc);
            cursor_next(sg, cx);
            __syncthreads();
        };
        int v = s0;
        for (; v + 1 < s1; v += 2) {
            step(v, std::integral_constant<int, 0>{});
            step(v + 1, std::integral_constant<int, 1>{});
        }
        if (v < s1) step(v, std::integral_constant<int, 0>{});
        s0 = s1;
    }
}

// ---- main, two or more 16-column tiles: weights decoded once per workgroup into LDS.
// A workgroup (8 waves) owns strips of ROWS rows. Per unit (strip, block column) the waves decode
// the ROWS x 64 tile of W into one of two LDS buffers while the previous unit's tile is multiplied
// from the other with every column of the launch: one barrier a unit.
// - Decode: a wave takes rows eight at a time, eight lanes a row, lane g of them the 16-byte
//   granule g of every slot's atom (8 weights): a read covers eight whole 128-byte atom rows,
//   which no bank conflict can slow (a row per lane and granules apart, as the A operands would
//   have it, measured 13.7 LDS cycles a read against 9.6), and the slots' packed fp16 FMAs run
//   in the same order as mfma_kernel's. The tile's granules lie at g ^ (row % 8), so the A
//   operand reads (16 rows, one granule) spread over all banks.
// - Product: waves RG x CG, each ROWS / RG rows by CT 16-column tiles; A from the LDS tile, B
//   straight from the transposed X (1 KiB a load, issued before the unit's decode, used after
//   it), so that X takes no LDS: where each wave decoded its own rows and read all of X from LDS
//   for them, the X reads were twice the decode's at 256 columns.
// - Code words two units ahead in a register ring; every load unconditional (clamped rows, units
//   past the range's end wrap), as in qroute_kernel.
// Bound by the LDS at many columns (per 64-row unit of 8 slots and 256 columns 136 KiB read or
// written, about 1,350 of its 2,000 cycles; matrix cores 512, vector ALU 560), and by the chain of
// a unit's reads, multiply-adds and writes at few; beside the units a 256-column call of 63 us
// spends 4 in the init launch, 8 before the first unit and 9 in the atomics into Y.
// 4096 x 11008, K = 1024, 8 slots, us per call before (each wave decoding its own rows, X through
// LDS) and after: fp16 X M = 32 40.2 -> 31.4, 64 48.2 -> 35, 128 63.7 -> 49.7, 256 90.7 ->
// 62.6; fp32 X M = 32 41.6 -> 33.8, 64 53 -> 45.6, 128 78 -> 64.7, 256 156 -> 83.
constexpr int kDecWaves = 8;

template <int ROWS, int RG, int CG, int CT, bool XS, int SLOTS>
__global__ __launch_bounds__(kDecWaves * 64) void mfma_dec_kernel(MParams p) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    static_assert(RG * CG == kDecWaves, "waves");
    constexpr int RT = ROWS / 16 / RG;  // 16-row tiles of a wave's product
    constexpr int NP = XS ? 2 : 1;          // X parts (fp32 X: hi, lo)
    constexpr int CW = SLOTS / 4;           // 16-byte code pieces per tile
    constexpr int DG = ROWS / kDecWaves / 8;  // groups of 8 rows that a wave decodes
    constexpr int TB = ROWS * 64;             // halves of a tile buffer
    // A unit's atoms read during the unit before, so that they and the A operands' reads keep the
    // LDS busy through the arithmetic (256 columns 70.8 -> 68.2 us a call, 128 56.0 -> 54.5);
    // waves without a barrier between their units drift apart and gain nothing by it.
    constexpr bool AHEAD = CG > 1 && DG * SLOTS <= 16;
    extern __shared__ __attribute__((aligned(16))) _Float16 smem16[];
    _Float16* Wt = smem16;           // two tile buffers
    _Float16* Ds = smem16 + 2 * TB;  // K x 64
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int q = lane >> 4, rl = lane & 15;
    const int dr = lane >> 3, dg = lane & 7;  // decode: row of the group, granule
    const int wr = wave / CG, wc = wave % CG;
    const int U = p.total_units;
    const int u0 = (int)((long long)U * blockIdx.x / gridDim.x);
    const int u1 = (int)((long long)U * (blockIdx.x + 1) / gridDim.x);
    if (u0 >= u1) return;

    for (int s0 = u0; s0 < u1;) {  // the units of one matrix at a time
        const int g = find_matrix(p, s0, -1);
        const MDesc& d = p.m[g];
        const int s1 = min(u1, d.u_base + d.u_count);
        SegGeom sg;
        sg.NB = d.NB;
        sg.NBc = d.NBc;
        sg.R = d.R;
        sg.nstrips = (d.R + ROWS - 1) / ROWS;
        sg.nfull = d.NB & ~(d.NBc - 1);
        const uint32_t* codes = d.codes;
        float* y = d.y;
        const float g0 = d.g0;
        uint32_t grel[SLOTS];
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) grel[j] = d.grel[j];
        const size_t nxt = xt_part(p, d), xblk = (size_t)p.Mpad * 64;
        const _Float16* xt0 = d.xt + xt_granule(p, 0, p.m0 + wc * CT * 16 + rl, 2 * q);

        u32x4 cr[2][DG][CW];
        auto load_codes = [&](const UnitCursor& c, u32x4 (&dst)[DG][CW]) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < DG; ++e) {
                const int r = min(c.strip * ROWS + (wave * DG + e) * 8 + dr, sg.R - 1);
                const uint32_t* w =
                    codes + ((size_t)c.b0 * sg.R + (size_t)r * c.nbc + (c.b - c.b0)) * SLOTS;
#pragma unroll
                for (int j = 0; j < CW; ++j) dst[e][j] = *reinterpret_cast<const u32x4*>(w + 4 * j);
            }
        };
        // the slots' granules of rows group e, all issued before the first is used (left to itself
        // the compiler keeps three or four in flight)
        auto atoms = [&](const u32x4 (&cw)[CW], u32x4 (&at)[SLOTS]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < SLOTS; ++j) {
                const uint32_t word = cw[j >> 2][j & 3];
                at[j] = *reinterpret_cast<const u32x4*>(Ds + (word & 0x7FFFu) * 64 + dg * 8);
            }
        };
        auto weights = [&](const u32x4 (&cw)[CW], const u32x4 (&at)[SLOTS], int e,
                           int buf) __attribute__((always_inline)) {
            h2 w[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) w[t] = h2{(_Float16)0.0f, (_Float16)0.0f};
#pragma unroll
            for (int j = 0; j < SLOTS; ++j) {
                const uint32_t word = cw[j >> 2][j & 3];
                const h2 c2 =
                    __builtin_bit_cast(h2, __builtin_amdgcn_perm(word, word, 0x07060706u)) *
                    __builtin_bit_cast(h2, grel[j]);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint32_t v = at[j][t];
                    w[t] = __builtin_elementwise_fma(c2, __builtin_bit_cast(h2, v), w[t]);
                }
            }
            const int row = (wave * DG + e) * 8 + dr;
            const u32x4 v = {__builtin_bit_cast(uint32_t, w[0]), __builtin_bit_cast(uint32_t, w[1]),
                             __builtin_bit_cast(uint32_t, w[2]), __builtin_bit_cast(uint32_t, w[3])};
            *reinterpret_cast<u32x4*>(Wt + buf * TB + row * 64 + ((dg ^ (row & 7)) * 8)) = v;
        };
        floatx4 acc[RT][CT];
        auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < RT; ++x)
#pragma unroll
                for (int c = 0; c < CT; ++c) acc[x][c] = floatx4{0.f, 0.f, 0.f, 0.f};
        };
        auto flush = [&](int strip) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < RT; ++x) {
                const int rbase = strip * ROWS + (wr * RT + x) * 16 + q * 4;
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const int m = p.m0 + (wc * CT + c) * 16 + rl;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = rbase + i;
                        if (r < sg.R && m < p.M)
                            __hip_atomic_fetch_add(
                                y + (p.tm ? (size_t)m * sg.R + r : (size_t)r * p.M + m),
                                acc[x][c][i] * g0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            }
        };
        // cursors: the unit multiplied, its successor, and the unit whose codes are loaded next
        UnitCursor cg;
        {
            const int lu = s0 - d.u_base;
            cg.strip = lu / sg.NB;
            cg.b = lu - cg.strip * sg.NB;
            cursor_chunk(sg, cg);
        }
        UnitCursor cc = cg;
        load_codes(cc, cr[1]);  // unit s0: ring slot of unit s0 + i is (i + 1) % 2
        cursor_next(sg, cc);
        load_codes(cc, cr[0]);
        cursor_next(sg, cc);
        {
            // the matrix's fp16 dictionary -> LDS (16-byte granules, 8 loads in flight)
            __syncthreads();
            const int n = d.K * 8;
            for (int i0 = 0; i0 < n; i0 += kDecWaves * 64 * 8) {
                u32x4 v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    v[j] = *reinterpret_cast<const u32x4*>(
                        d.dict16p + (size_t)min(i0 + j * kDecWaves * 64 + tid, n - 1) * 8);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    *reinterpret_cast<u32x4*>(
                        Ds + (size_t)min(i0 + j * kDecWaves * 64 + tid, n - 1) * 8) = v[j];
            }
            __syncthreads();
        }
        clear();
#pragma unroll
        for (int e = 0; e < DG; ++e) {
            u32x4 at[SLOTS];
            atoms(cr[1][e], at);
            weights(cr[1][e], at, e, 0);
        }
        load_codes(cc, cr[1]);
        cursor_next(sg, cc);
        u32x4 cw[DG][CW], at[AHEAD ? DG : 1][SLOTS];  // unit v + 1's words, and its atoms' granules
        if constexpr (AHEAD) {
#pragma unroll
            for (int e = 0; e < DG; ++e) {
                atoms(cr[0][e], at[e]);
#pragma unroll
                for (int j = 0; j < CW; ++j) cw[e][j] = cr[0][e][j];
            }
            load_codes(cc, cr[0]);
            cursor_next(sg, cc);
        }
        auto step = [&](int v, auto S) __attribute__((always_inline)) {
            constexpr int sl = decltype(S)::value;  // ring slot and target buffer of unit v + 1
            // unit v's tile is whole, unit v - 1's has been read (with one column group a wave
            // multiplies the rows that it decoded: its own LDS order does, which the fence, no
            // instruction, keeps the compiler to)
            if constexpr (CG > 1) {
                __syncthreads();
            } else {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            u32x4 xb[CT][NP][2];
            const _Float16* xs = xt0 + (size_t)cg.b * xblk;
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int part = 0; part < NP; ++part)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        xb[c][part][h] = *reinterpret_cast<const u32x4*>(
                            xs + part * nxt + (size_t)c * 1024 + h * 512);
            const _Float16* wb = Wt + sl * TB + (wr * RT * 16 + rl) * 64;
            half8 a[2][RT];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int x = 0; x < RT; ++x)
                    a[h][x] = __builtin_bit_cast(
                        half8, *reinterpret_cast<const u32x4*>(
                                   wb + x * 16 * 64 + (((2 * q + h) ^ (rl & 7)) * 8)));
            __builtin_amdgcn_sched_barrier(0);  // the loads above go first
            if constexpr (AHEAD) {
                // unit v + 1 from the granules read during the last unit's products, then unit
                // v + 2's reads, in flight during this unit's
#pragma unroll
                for (int e = 0; e < DG; ++e) weights(cw[e], at[e], e, 1 - sl);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < DG; ++e) {
                    atoms(cr[1 - sl][e], at[e]);
#pragma unroll
                    for (int j = 0; j < CW; ++j) cw[e][j] = cr[1 - sl][e][j];
                }
                load_codes(cc, cr[1 - sl]);
                __builtin_amdgcn_sched_barrier(0);
            } else if constexpr (DG * SLOTS <= 16) {
                u32x4 ag[DG][SLOTS];
#pragma unroll
                for (int e = 0; e < DG; ++e) atoms(cr[sl][e], ag[e]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < DG; ++e) weights(cr[sl][e], ag[e], e, 1 - sl);
                load_codes(cc, cr[sl]);
            } else {  // a group at a time: two groups of 16 slots' reads would spill
#pragma unroll
                for (int e = 0; e < DG; ++e) {
                    u32x4 ag[SLOTS];
                    atoms(cr[sl][e], ag);
                    weights(cr[sl][e], ag, e, 1 - sl);
                }
                load_codes(cc, cr[sl]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int part = 0; part < NP; ++part)
#pragma unroll
                        for (int x = 0; x < RT; ++x)
                            acc[x][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                a[h][x], __builtin_bit_cast(half8, xb[c][part][h]), acc[x][c], 0, 0,
                                0);
            const int strip = cg.strip;
            cursor_next(sg, cg);
            cursor_next(sg, cc);
            if (v + 1 == s1 || cg.strip != strip) {
                flush(strip);
                clear();
            }
        };
        int v = s0;
        for (; v + 1 < s1; v += 2) {
            step(v, std::integral_constant<int, 0>{});
            step(v + 1, std::integral_constant<int, 1>{});
        }
        if (v < s1) step(v, std::integral_constant<int, 0>{});
        s0 = s1;
    }
}

// Columns of X the kernels see: M rounded up to a power of two >= 16 (<= 256), beyond 256 to
// a multiple of 256, so every launch covers a power-of-two tile of 16 NT columns.
int padded_m(int M) {
    if (M > kMaxMTile) return (M + kMaxMTile - 1) / kMaxMTile * kMaxMTile;
    int p = 16;
    while (p < M) p *= 2;
    return p;
}

size_t xt_bytes(const csdr_hsdb* s, int M) {
    const size_t mpad = (size_t)padded_m(M);
    return csdr::align_up(2 * mpad * s->C_full * sizeof(_Float16), 256);
}

// The dictionary route for one 16-column tile (M <= 16); CSDR_HSDB_QROUTE=0 keeps the
// weight-decoding kernel there.
bool qroute_enabled() {
    const char* e = std::getenv("CSDR_HSDB_QROUTE");
    return !(e && *e && std::atoi(e) == 0);
}

template <typename F>
int launch_lds(F kern, const MParams& p, int grid, int threads, size_t lds, hipStream_t st) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    kern<<<grid, threads, lds, st>>>(p);
    CSDR_LAUNCH_CHECK("hsdb mfma");
    return CSDR_OK;
}

// Rows of a strip by column tiles of the launch: each strip's partial sums are added into Y once
// per workgroup that has units of it, as float atomics in memory, so R x M times the strips'
// share of 256 workgroups: at 128 rows and 256 columns those were 19 us of a 61 us launch (13 of
// 48 at 128 columns), half of that at 64 rows, where the X loads (per unit) count double. With
// fewer columns the decode counts more, and 128 rows give each wave its own 16.
constexpr int dec_rows(int nt) { return nt >= 8 ? 64 : 128; }

template <bool XS, int SLOTS>
int launch_main(const MParams& p, int nt, int grid, size_t lds, hipStream_t st) {
    constexpr int kT = kDecWaves * 64;
    switch (nt) {
        case 16: return launch_lds(&mfma_dec_kernel<64, 1, 8, 2, XS, SLOTS>, p, grid, kT, lds, st);
        case 8: return launch_lds(&mfma_dec_kernel<64, 2, 4, 2, XS, SLOTS>, p, grid, kT, lds, st);
        case 4: return launch_lds(&mfma_dec_kernel<128, 8, 1, 4, XS, SLOTS>, p, grid, kT, lds, st);
        case 2: return launch_lds(&mfma_dec_kernel<128, 8, 1, 2, XS, SLOTS>, p, grid, kT, lds, st);
        default: return launch_lds(&mfma_kernel<XS, SLOTS>, p, grid, 1024, lds, st);
    }
}

template <bool XS>
int launch_slots(const MParams& p, int nt, int slots, int grid, size_t lds, hipStream_t st) {
    switch (slots) {
        case 4: return launch_main<XS, 4>(p, nt, grid, lds, st);
        case 8: return launch_main<XS, 8>(p, nt, grid, lds, st);
        default: return launch_main<XS, 16>(p, nt, grid, lds, st);
    }
}

}  // namespace

namespace csdr {

bool mfma_eligible(int n, const csdr_hsdb* const* segs, int M) {
    const char* e = std::getenv("CSDR_HSDB_MFMA");
    if (e && *e && std::atoi(e) == 0) return false;
    if (M < kMfmaMinM) return false;
    for (int i = 0; i < n; ++i) {
        const csdr_hsdb* s = segs[i];
        if (!s || s->tile_rows != 1 || s->tile_cols != 64 || s->K > (uint32_t)kMaxAtoms ||
            !s->d_dict16p ||
            s->NB == 0 || !(s->slots == 4 || s->slots == 8 || s->slots == 16) ||
            s->slots != segs[0]->slots)
            return false;
    }
    return true;
}

size_t mfma_workspace_bytes(int n, const csdr_hsdb* const* segs, int M) {
    size_t t = csdr::kWsHead;
    for (int i = 0; i < n; ++i) t += xt_bytes(segs[i], M);
    return t;
}

int mfma_matmul(int n, const csdr_hsdb* const* segs, const void* const* xs, int x_dtype, int M,
                float* const* ys, const float* const* bias, int accumulate, int token_major,
                void* workspace, size_t workspace_bytes, hipStream_t st) {
    const size_t need = mfma_workspace_bytes(n, segs, M);
    if (!workspace || workspace_bytes < need)
        return set_error(CSDR_E_WORKSPACE,
                         "hsdb_matmul: workspace needs " + std::to_string(need) + " bytes");
    MParams p{};
    p.G = n;
    p.M = M;
    p.Mpad = padded_m(M);
    p.x_f16 = (x_dtype == CSDR_F16);
    p.accumulate = accumulate;
    p.tm = token_major;
    char* ws = static_cast<char*>(workspace);
    size_t off = csdr::kWsHead;
    size_t max_y = 0;
    int max_nb = 0;
    bool any_edge = false;
    for (int i = 0; i < n; ++i) {
        const csdr_hsdb* s = segs[i];
        MDesc& d = p.m[i];
        d.codes = s->d_codes;
        d.dict16p = s->d_dict16p;
        d.edge = s->d_edge;
        d.x = xs[i];
        d.y = ys[i];
        d.bias = bias ? bias[i] : nullptr;
        d.xt = reinterpret_cast<_Float16*>(ws + off);
        off += xt_bytes(s, M);
        d.R = (int)s->R;
        d.K = (int)s->K;
        d.NB = (int)s->NB;
        d.NBc = (int)s->NBc;
        d.slots = (int)s->slots;
        d.Ce = (int)s->Ce;
        d.C_full = (int)s->C_full;
        // the slots' gains relative to the largest: 1 for the usual single stage and powers of
        // two for gamma_l = 0.5^l (exact in fp16), never above 1 (no fp16 overflow)
        float gmax = 0.0f;
        for (uint32_t j = 0; j < s->slots && j < 16; ++j)
            gmax = std::max(gmax, std::fabs(s->h_slot_gamma[j]));
        d.g0 = gmax > 0.0f ? gmax : 1.0f;
        for (uint32_t j = 0; j < 16; ++j) {
            const float rel = j < s->slots ? s->h_slot_gamma[j] / d.g0 : 0.0f;
            const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)rel);
            d.grel[j] = h << 16 | h;
        }
        max_y = std::max(max_y, (size_t)d.R * M);
        max_nb = std::max(max_nb, d.NB);
        any_edge = any_edge || d.Ce > 0;
    }
    int dev = 0, ncu = 256, lds_max = 65536;
    if (hipGetDevice(&dev) == hipSuccess) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            v > 0)
            ncu = v;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) ==
                hipSuccess &&
            v > 0)
            lds_max = v;
    }
    {
        // a workgroup per block column and MW columns of X, and some for Y
        const int mw = std::min(64, p.Mpad);
        const size_t yper = any_edge && max_y <= kEdgeWide ? kThreads : 4 * kThreads;
        const int xwgs = max_nb * (p.Mpad / mw);
        const int ywgs = (int)std::min<size_t>(any_edge ? 4096 : 1024, (max_y + yper - 1) / yper);
        const dim3 grid(xwgs + std::max(ywgs, 1), n);
        auto go = [&](auto kern) { kern<<<grid, kThreads, 0, st>>>(p, xwgs); };
        auto pick = [&](auto xt) {
            using XT = decltype(xt);
            if (mw == 64) go(&mfma_init_kernel<XT, 64>);
            else if (mw == 32) go(&mfma_init_kernel<XT, 32>);
            else go(&mfma_init_kernel<XT, 16>);
        };
        if (p.x_f16) pick(_Float16{});
        else pick(float{});
        CSDR_LAUNCH_CHECK("hsdb mfma init");
    }
    const bool xsplit = !p.x_f16;
    const int mt = std::min(p.Mpad, kMaxMTile), nt = mt / 16;  // columns of a launch
    uint32_t kmax = 0;
    for (int i = 0; i < n; ++i) kmax = std::max(kmax, segs[i]->K);
    const size_t lds = (size_t)kmax * 64 * sizeof(_Float16) +
                       (nt > 1 ? (size_t)2 * dec_rows(nt) * 64 * sizeof(_Float16) : 0);
    if (lds > (size_t)lds_max)
        return set_error(CSDR_E_UNSUPPORTED, "hsdb_matmul: LDS too small for the MFMA path");
    const int strip_rows = nt > 1 ? dec_rows(nt) : 256;
    int units = 0;
    for (int i = 0; i < n; ++i) {
        MDesc& d = p.m[i];
        d.u_base = units;
        d.u_count = (d.R + strip_rows - 1) / strip_rows * d.NB;
        units += d.u_count;
    }
    p.total_units = units;
    const int grid = std::max(1, std::min(units, ncu));
    const int slots0 = (int)segs[0]->slots;
    if (nt == 1 && !xsplit && (slots0 == 4 || slots0 == 8) && qroute_enabled()) {
        // one 16-column tile of fp16 X: Q_b formed per unit on the matrix cores, rows gathered
        // from LDS (fp32 X and 16 slots keep the decoding kernel: their operand rings spill)
        // two Q buffers, then a 16 x 16 fp32 tile per wave for the strip flushes
        const size_t qlds = (size_t)2 * kMaxAtoms * 16 * sizeof(_Float16) + 16 * 256 * sizeof(float);
        auto go = [&](auto kern) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)qlds);
            kern<<<grid, 1024, qlds, st>>>(p);
        };
        if (slots0 == 4) go(qroute_kernel<4, false>);
        else go(qroute_kernel<8, false>);
        CSDR_LAUNCH_CHECK("hsdb qroute");
        return CSDR_OK;
    }
    for (int m0 = 0; m0 < p.Mpad; m0 += mt) {
        p.m0 = m0;
        const int rc = xsplit ? launch_slots<true>(p, nt, slots0, grid, lds, st)
                              : launch_slots<false>(p, nt, slots0, grid, lds, st);
        if (rc != CSDR_OK) return rc;
    }
    return CSDR_OK;
}

}  // namespace csdr
