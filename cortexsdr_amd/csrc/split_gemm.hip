// split_gemm.hip — Y = X . W^T of fp32 values on the fp16 matrix cores (gfx950), for the
// decoder's batched prefill: W decoded from its codes once per pass, X the prompt's rows.
//
// The fp32 matrix-core rate (157 TFLOP/s dense) bounds the fp32 product (gemm_f32.hip), a
// sixteenth of the fp16 one. Here each value is hi + 2^-12 lo, two fp16 numbers after scaling its
// row by a power of two that puts the row's largest magnitude in [2^14, 2^15): hi has 11 bits, lo
// the next 11. lo is stored 2^12 times its size, as large as hi can be, so that it keeps its bits
// where the value is small: the pair is the value to 2^-23 of it down to 2^-27 of the row's
// largest, and to 2^-51 of that below (stored at its size lo ran out at 2^-39, and a row with one
// value 2^24 times the rest lost 2^-16 of the rest). Then
//   x . w = hi hi + 2^-12 (hi lo + lo hi) + 2^-24 lo lo
// with the last term (at most 2^-22 of a product) left out: three 16x16x32 products, exact in fp32
// and summed in fp32, the cross terms in accumulators of their own. Against 64 bits the product
// is 1.4e-7 to 6.9e-7 off (relative L2, 896 to 16384 columns), the fp32 matrix cores' 5.0e-7 to
// 2.3e-6 (their longer chains of rounded sums).
// A 511-token pass of such a block: 410 -> 245 us (products 245 -> 110, decodes 134 -> 50).
// Rows with a NaN or an infinity are marked (inv < 0) and their outputs recomputed from the
// planes' values in plain fp32, so that they come out as an fp32 product's.
//
// Reference: Kernels::linear_forward (kernels/blas_kernels.cpp:264-293) over the decoded weight,
// as gemm_f32.hip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "split_gemm.hpp"

namespace {

using csdr::set_error;
using csdr::SplitPlanes;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float block_max(float v) {
    __shared__ float red[kWaves];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v = fmaxf(v, red[w]);
    __syncthreads();
    return v;
}

__device__ __forceinline__ float block_sum(float v) {
    __shared__ float red[kWaves];
    v = csdr::wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v += red[w];
    __syncthreads();
    return v;
}

// The power of two that takes a finite magnitude mx into [2^14, 2^15) (1 for a zero row; at
// most 2^126, so that it and its inverse are normal numbers), and its inverse.
__device__ __forceinline__ void row_scale(float mx, float& up, float& down) {
    int e = 0;
    if (mx > 0.f) e = min(14 - ilogbf(mx), 126);
    up = ldexpf(1.0f, e);
    down = ldexpf(1.0f, -e);
}

constexpr float kLoUp = 4096.f, kLoDown = 1.f / 4096.f;  // |s - hi| <= 2^3: lo to 2^15

__device__ __forceinline__ void split1(float v, float up, _Float16& hi, _Float16& lo) {
    const float s = v * up;
    hi = (_Float16)s;
    lo = fabsf(s) < INFINITY ? (_Float16)((s - (float)hi) * kLoUp) : (_Float16)0.f;
}

// v times the row scales a and b (powers of two, signs aside): by their exponents' sum, since
// one of the two alone may take v out of range on the way to a result that is in it.
__device__ __forceinline__ float unscale(float v, float a, float b) {
    const auto ex = [](float f) { return (int)(__builtin_bit_cast(uint32_t, f) >> 23 & 0xFF) - 127; };
    return __builtin_amdgcn_ldexpf(v, ex(a) + ex(b));
}

// A magnitude for the row's largest: 0 for a value that is not finite (noted in `odd`).
__device__ __forceinline__ float finite_abs(float v, bool& odd) {
    const float a = fabsf(v);
    if (a < INFINITY) return a;
    odd = true;
    return 0.f;
}

// ---------------------------------------------------------------- W: codes -> planes

struct DecodeMat {
    const uint32_t* codes;
    const float* dict;
    const float* gamma;  // per slot
    const float* edge;
    _Float16* hi;
    _Float16* lo;
    float* inv;
    uint32_t R, C, C_full, Ce, NB, NBc, slots, ld;
};
struct DecodeArgs {
    DecodeMat m[csdr::kSplitMats];
    uint32_t first[csdr::kSplitMats + 1];  // first workgroup of each matrix
};

// One workgroup per row of W: 16 lanes per 64-long tile take 4 elements each (an atom row is a
// 256-byte L2 read per slot), a thread's tiles b = group, group + 16, ... (NI of them) stay in
// registers until the row's largest magnitude is known. Slots in order from 0, as
// decode_dense_kernel. Bound by the atom reads out of L2. (4864 x 896, 8 slots: 33 us as
// decode_dense_kernel, a thread per element; 12 us for two such matrices here with both planes written.)
template <int SLOTS, int NI>
__global__ __launch_bounds__(kThreads) void split_decode_kernel(DecodeArgs a) {
    int i = 0;
#pragma unroll
    for (int q = 1; q < csdr::kSplitMats; ++q)
        if (blockIdx.x >= a.first[q]) i = q;
    const DecodeMat& m = a.m[i];
    const uint32_t r = blockIdx.x - a.first[i];
    const uint32_t slots = SLOTS ? SLOTS : m.slots;
    const int l16 = threadIdx.x & 15, grp = threadIdx.x >> 4;
    floatx4 v[NI];
    float mx = 0.f;
    bool odd = false;
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        v[q] = floatx4{0.f, 0.f, 0.f, 0.f};
        const uint32_t b = grp + 16 * q;
        if (b >= m.NB) continue;
        const uint32_t* w = m.codes + csdr::tile_word_offset(r, b, m.R, m.NB, m.NBc, slots);
        auto add = [&](uint32_t j, uint32_t wd) {
            const float cf = m.gamma[j] * csdr::h2f(wd >> 16);
            const floatx4 d =
                *reinterpret_cast<const floatx4*>(m.dict + (wd & 0x7FFFu) * 64 + 4 * l16);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[q][e] = fmaf(cf, d[e], v[q][e]);
        };
        if constexpr (SLOTS != 0) {  // a multiple of 4: 16-byte aligned tiles
            uint4 ws[SLOTS / 4];
#pragma unroll
            for (int j = 0; j < SLOTS / 4; ++j) ws[j] = reinterpret_cast<const uint4*>(w)[j];
#pragma unroll
            for (int j = 0; j < SLOTS / 4; ++j) {
                add(4 * j, ws[j].x);
                add(4 * j + 1, ws[j].y);
                add(4 * j + 2, ws[j].z);
                add(4 * j + 3, ws[j].w);
            }
        } else {
            for (uint32_t j = 0; j < slots; ++j) add(j, w[j]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, finite_abs(v[q][e], odd));
    }
    float ev = 0.f;  // one edge value per thread (fewer than 64 of them)
    if (threadIdx.x < m.Ce) {
        ev = m.edge[(size_t)r * m.Ce + threadIdx.x];
        mx = fmaxf(mx, finite_abs(ev, odd));
    }
    const bool any_odd = __syncthreads_or(odd);
    float up, down;
    row_scale(block_max(mx), up, down);
    _Float16* hi = m.hi + (size_t)r * m.ld;
    _Float16* lo = m.lo + (size_t)r * m.ld;
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const uint32_t b = grp + 16 * q;
        if (b >= m.NB) continue;
        h4 h, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            _Float16 x, y;
            split1(v[q][e], up, x, y);
            h[e] = x;
            l[e] = y;
        }
        *reinterpret_cast<h4*>(hi + b * 64 + 4 * l16) = h;
        *reinterpret_cast<h4*>(lo + b * 64 + 4 * l16) = l;
    }
    const uint32_t c = m.C_full + threadIdx.x;
    if (c < m.ld) {  // the edge, then zeros to the end of the plane's row
        _Float16 x, y;
        split1(ev, up, x, y);
        hi[c] = x;
        lo[c] = y;
    }
    if (threadIdx.x == 0) m.inv[r] = any_odd ? -down : down;
}

// ---------------------------------------------------------------- X: rows -> planes

// One workgroup per token row; the row's values wait in LDS for its largest magnitude. The
// norm and the gate are rms_norm_kernel's and silu_mul_kernel's expressions.
template <csdr::SplitOp OP>
__global__ __launch_bounds__(kThreads) void split_rows_kernel(float* __restrict__ x,
                                                              const float* __restrict__ x2,
                                                              const float* __restrict__ parts,
                                                              int n_parts, int M, int n, float eps,
                                                              SplitPlanes o) {
    extern __shared__ float row[];
    const size_t at = (size_t)blockIdx.x * n;
    float ss = 0.f, mx = 0.f;
    bool odd = false;
    for (int i = threadIdx.x; i < n; i += kThreads) {
        float v = x[at + i];
        if (n_parts) {
            float p = parts[at + i];
            for (int z = 1; z < n_parts; ++z) p += parts[(size_t)z * M * n + at + i];
            v += p;
            x[at + i] = v;
        }
        if constexpr (OP == csdr::SplitOp::rms_norm) ss = fmaf(v, v, ss);
        if constexpr (OP == csdr::SplitOp::silu_mul) {
            const float sig = 1.0f / (1.0f + expf(-v));
            v = (v * sig) * x2[at + i];
        }
        if constexpr (OP != csdr::SplitOp::rms_norm) mx = fmaxf(mx, finite_abs(v, odd));
        row[i] = v;
    }
    if constexpr (OP == csdr::SplitOp::rms_norm) {
        ss = block_sum(ss);
        const float inv = 1.0f / sqrtf(ss / (float)n + eps);
        for (int i = threadIdx.x; i < n; i += kThreads) {
            const float v = row[i] * inv * x2[i];
            row[i] = v;  // this thread's own values
            mx = fmaxf(mx, finite_abs(v, odd));
        }
    }
    const bool any_odd = __syncthreads_or(odd);
    float up, down;
    row_scale(block_max(mx), up, down);
    _Float16* hi = o.hi + (size_t)blockIdx.x * o.ld;
    _Float16* lo = o.lo + (size_t)blockIdx.x * o.ld;
    for (int i = 4 * threadIdx.x; i < o.ld; i += 4 * kThreads) {
        h4 h, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            _Float16 a, b;
            split1(i + e < n ? row[i + e] : 0.f, up, a, b);
            h[e] = a;
            l[e] = b;
        }
        *reinterpret_cast<h4*>(hi + i) = h;
        *reinterpret_cast<h4*>(lo + i) = l;
    }
    if (threadIdx.x == 0) o.inv[blockIdx.x] = any_odd ? -down : down;
}

// ---------------------------------------------------------------- the product

struct GemmMat {
    SplitPlanes w;
    float* y;
    const float* bias;
    int R;
};
struct GemmArgs {
    GemmMat m[csdr::kSplitMats];
    uint32_t first[csdr::kSplitMats + 1];  // first row tile of each matrix
    SplitPlanes x;
    int M, stages, per_split;  // 32-deep stages in all and per part
    int parts;
};

constexpr int kBK = 32;

// A (32 WR rows of W) x (32 WM token rows) tile per 2 x 2 waves, each wave 16 WR x 16 WM. Per
// 32-deep stage the four planes' slices (64 bytes a row) go through registers into one of two
// LDS buffers while the other is multiplied: one barrier a stage, the next stage's loads in
// flight during the products. A row's four 16-byte pieces are placed at piece ^ (row / 2 % 4),
// which spreads the operand reads (16 rows, one piece) over all banks. Per stage and wave
// 3 WR WM products of 16 cycles against 2 (WR + WM) 1-KiB LDS reads: at 4 x 2 the LDS reads
// (4 waves, 128 bytes a cycle) and the matrix cores take about as long as each other.
// MFMA operands: A = W (row l % 16, k = 8 (l / 16) + j), B = X; lane l holds
// D[row 4 (l / 16) + v][token l % 16].
template <int WR, int WM>
__global__ __launch_bounds__(kThreads) void split_gemm_kernel(GemmArgs a) {
    constexpr int TR = 32 * WR, TM = 32 * WM;
    constexpr int NP = (TR + TM) * 2 / 16;  // 16-row pieces of a stage (1 KiB each)
    constexpr int NI = NP / kWaves;         // per wave
    static_assert(NP % kWaves == 0, "pieces per wave");
    __shared__ __attribute__((aligned(16))) _Float16 lds[2][(TR + TM) * 2 * kBK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    int i = 0;
#pragma unroll
    for (int q = 1; q < csdr::kSplitMats; ++q)
        if (blockIdx.x >= a.first[q]) i = q;
    const GemmMat& mat = a.m[i];
    const int r0 = (int)(blockIdx.x - a.first[i]) * TR, m0 = blockIdx.y * TM;
    const int wr0 = (wave >> 1) * 16 * WR, wm0 = (wave & 1) * 16 * WM;
    const int s0 = blockIdx.z * a.per_split, s1 = min(s0 + a.per_split, a.stages);

    // piece p of a stage: TR / 16 of W's hi plane, as many of lo, then X's
    const _Float16* src[NI];
    int dst[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int p = wave + kWaves * q;
        const int row16 = lane >> 2, slot = lane & 3;
        const int g = slot ^ ((row16 >> 1) & 3);
        const bool isw = p < 2 * TR / 16;
        const int pp = isw ? p : p - 2 * TR / 16, half = (isw ? TR : TM) / 16;
        const SplitPlanes& pl = isw ? mat.w : a.x;
        const int row = (pp % half) * 16 + row16;
        const int gr = isw ? min(r0 + row, mat.R - 1) : min(m0 + row, a.M - 1);
        src[q] = (pp < half ? pl.hi : pl.lo) + (size_t)gr * pl.ld + (size_t)s0 * kBK + g * 8;
        dst[q] = p * 16 * kBK + lane * 8;
    }
    h8 pre[NI];
    auto load = [&] {
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            pre[q] = *reinterpret_cast<const h8*>(src[q]);
            src[q] += kBK;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NI; ++q) *reinterpret_cast<h8*>(&lds[buf][dst[q]]) = pre[q];
    };
    floatx4 acc[WR][WM], cross[WR][WM];
#pragma unroll
    for (int x = 0; x < WR; ++x)
#pragma unroll
        for (int y = 0; y < WM; ++y) acc[x][y] = cross[x][y] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int piece = (lg ^ ((li >> 1) & 3)) * 8;
    load();
    store(0);
    __syncthreads();
    for (int s = s0; s < s1; ++s) {
        const int buf = (s - s0) & 1;
        if (s + 1 < s1) load();
        const _Float16* L = lds[buf];
        h8 wh[WR], wl[WR], xh[WM], xl[WM];
#pragma unroll
        for (int x = 0; x < WR; ++x) {
            wh[x] = *reinterpret_cast<const h8*>(L + (wr0 + x * 16 + li) * kBK + piece);
            wl[x] = *reinterpret_cast<const h8*>(L + (TR + wr0 + x * 16 + li) * kBK + piece);
        }
#pragma unroll
        for (int y = 0; y < WM; ++y) {
            xh[y] = *reinterpret_cast<const h8*>(L + (2 * TR + wm0 + y * 16 + li) * kBK + piece);
            xl[y] =
                *reinterpret_cast<const h8*>(L + (2 * TR + TM + wm0 + y * 16 + li) * kBK + piece);
        }
#pragma unroll
        for (int x = 0; x < WR; ++x)
#pragma unroll
            for (int y = 0; y < WM; ++y) {
                acc[x][y] =
                    __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[x], xh[y], acc[x][y], 0, 0, 0);
                cross[x][y] =
                    __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[x], xl[y], cross[x][y], 0, 0, 0);
                cross[x][y] =
                    __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[x], xh[y], cross[x][y], 0, 0, 0);
            }
        if (s + 1 < s1) store(buf ^ 1);
        __syncthreads();
    }

    float* yb = mat.y + (size_t)blockIdx.z * a.M * mat.R;
#pragma unroll
    for (int y = 0; y < WM; ++y) {
        const int m = m0 + wm0 + y * 16 + li;
        if (m >= a.M) continue;
        const float xi = a.x.inv[m];
        float* yr = yb + (size_t)m * mat.R;
#pragma unroll
        for (int x = 0; x < WR; ++x) {
            const int r = r0 + wr0 + x * 16 + 4 * lg;
            float out[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (r + v >= mat.R) continue;
                const float wi = mat.w.inv[r + v];
                out[v] = unscale(fmaf(cross[x][y][v], kLoDown, acc[x][y][v]), wi, xi);
                if (wi < 0.f || xi < 0.f) {  // a NaN or an infinity in the row: plain fp32
                    const _Float16 *wh2 = mat.w.hi + (size_t)(r + v) * mat.w.ld,
                                   *wl2 = mat.w.lo + (size_t)(r + v) * mat.w.ld;
                    const _Float16 *xh2 = a.x.hi + (size_t)m * a.x.ld,
                                   *xl2 = a.x.lo + (size_t)m * a.x.ld;
                    float sum = 0.f;
                    for (int k = s0 * kBK; k < s1 * kBK; ++k)
                        sum = fmaf(fmaf((float)wl2[k], kLoDown, (float)wh2[k]),
                                   fmaf((float)xl2[k], kLoDown, (float)xh2[k]), sum);
                    out[v] = unscale(sum, wi, xi);
                }
                if (mat.bias && a.parts == 1) out[v] += mat.bias[r + v];
            }
            if (r + 3 < mat.R && mat.R % 4 == 0) {
                *reinterpret_cast<floatx4*>(yr + r) = floatx4{out[0], out[1], out[2], out[3]};
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (r + v < mat.R) yr[r + v] = out[v];
            }
        }
    }
}

template <int WR, int WM>
void launch_gemm(GemmArgs& a, int n, hipStream_t st) {
    uint32_t tiles = 0;
    for (int i = 0; i < csdr::kSplitMats; ++i) {
        a.first[i] = i < n ? tiles : 0xFFFFFFFFu;
        if (i < n) tiles += (uint32_t)((a.m[i].R + 32 * WR - 1) / (32 * WR));
    }
    const dim3 grid(tiles, (unsigned)((a.M + 32 * WM - 1) / (32 * WM)), (unsigned)a.parts);
    split_gemm_kernel<WR, WM><<<grid, kThreads, 0, st>>>(a);
}

}  // namespace

namespace csdr {

bool split_eligible(const csdr_hsdb* s) {
    return s->tile_rows == 1 && s->tile_cols == 64 && s->C <= (uint32_t)kSplitMaxCols &&
           s->NB > 0;
}

int split_decode(int n, const csdr_hsdb* const* segs, const SplitPlanes* out, hipStream_t st) {
    DecodeArgs a{};
    uint32_t rows = 0, nb = 0;
    uint32_t slots = segs[0]->slots;
    for (int i = 0; i < kSplitMats; ++i) {
        a.first[i] = i < n ? rows : 0xFFFFFFFFu;
        if (i >= n) continue;
        const csdr_hsdb* s = segs[i];
        if (!codes_on_device(s))
            return set_error(CSDR_E_UNSUPPORTED, "prefill: the segment's codes are in host memory");
        a.m[i] = DecodeMat{s->d_codes, s->d_dict, s->d_slot_gamma, s->d_edge,  out[i].hi,
                           out[i].lo,  out[i].inv, s->R,           s->C,       s->C_full,
                           s->Ce,      s->NB,      s->NBc,         s->slots,   (uint32_t)out[i].ld};
        rows += s->R;
        nb = std::max(nb, s->NB);
        if (s->slots != slots) slots = 0;
    }
    auto go = [&](auto kern) { kern<<<rows, kThreads, 0, st>>>(a); };
    // tiles per thread: 1, 2, 5 (4864 columns), 11 (11008) or 16
#define CSDR_SPLIT_NI(SL)                                   \
    do {                                                    \
        if (nb <= 16) go(&split_decode_kernel<SL, 1>);      \
        else if (nb <= 32) go(&split_decode_kernel<SL, 2>); \
        else if (nb <= 80) go(&split_decode_kernel<SL, 5>); \
        else if (nb <= 176) go(&split_decode_kernel<SL, 11>); \
        else go(&split_decode_kernel<SL, 16>);              \
    } while (0)
    if (slots == 4) CSDR_SPLIT_NI(4);
    else if (slots == 8) CSDR_SPLIT_NI(8);
    else if (slots == 16) CSDR_SPLIT_NI(16);
    else CSDR_SPLIT_NI(0);
#undef CSDR_SPLIT_NI
    CSDR_LAUNCH_CHECK("prefill decode");
    return CSDR_OK;
}

int split_rows(SplitOp op, float* x, const float* x2_or_w, const float* parts, int n_parts, int M,
               int n, float eps, const SplitPlanes& out, hipStream_t st) {
    auto go = [&](auto kern) {
        const size_t lds = (size_t)n * 4;
        if (lds > 60 * 1024)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        kern<<<M, kThreads, lds, st>>>(x, x2_or_w, parts, n_parts, M, n, eps, out);
    };
    if (op == SplitOp::plain) go(&split_rows_kernel<SplitOp::plain>);
    else if (op == SplitOp::rms_norm) go(&split_rows_kernel<SplitOp::rms_norm>);
    else go(&split_rows_kernel<SplitOp::silu_mul>);
    CSDR_LAUNCH_CHECK("prefill rows");
    return CSDR_OK;
}

// 64 x 64 tiles: enough parts for 384 workgroups, each of at least 8 stages.
int split_count(int R, int K, int M) {
    const long long tiles = (long long)((R + 63) / 64) * ((M + 63) / 64);
    const int stages = split_ld(K) / kBK;
    int s = 1;
    while (s < 8 && tiles * s < 384 && stages / (2 * s) >= 8) s *= 2;
    return s;
}

int split_gemm(int n, const SplitPlanes* w, const int* R, const SplitPlanes& x, int M,
               float* const* ys, const float* const* bias, int splits, hipStream_t st) {
    GemmArgs a{};
    a.x = x;
    a.M = M;
    a.stages = x.ld / kBK;
    a.parts = splits;
    a.per_split = (a.stages + splits - 1) / splits;
    long long t128 = 0, t64 = 0;
    for (int i = 0; i < n; ++i) {
        a.m[i] = GemmMat{w[i], ys[i], bias ? bias[i] : nullptr, R[i]};
        t128 += (R[i] + 127) / 128;
        t64 += (R[i] + 63) / 64;
    }
    const long long c64 = (M + 63) / 64;
    // the largest tile that still gives every CU a workgroup
    if (t128 * c64 * splits >= 256) launch_gemm<4, 2>(a, n, st);
    else if (t64 * c64 * splits >= 256) launch_gemm<2, 2>(a, n, st);
    else launch_gemm<2, 1>(a, n, st);
    CSDR_LAUNCH_CHECK("prefill product");
    return CSDR_OK;
}

}  // namespace csdr
