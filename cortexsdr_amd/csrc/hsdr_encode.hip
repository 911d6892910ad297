// hsdr_encode.hip — the HSDR encoder on the GPU (gfx950): hierarchical binary matching pursuit
// over many tiles at once, and the strategy's compress around it.
//
// Reference (cortexSDR tree, src/ai_compression/strategies/HierarchicalSDRStrategy.cpp):
// hierarchicalBinaryCode :219-262 (per tile, per stage l with scale gamma_l, k greedy picks of
// argmax |<D_j, r>| with a strict '>' scan from (0, 0.0f), atoms picked earlier in the stage
// scoring 0, sign = +1 when the projection is >= 0, then r -= gamma_l * sign * D_best),
// dot_product_simd :157-190 and axpy_subtract_simd :193-216 (its AVX2 arithmetic),
// fitHierarchicalKSVD :495-602 (dictionary initialisation, hsdr_init.cpp), compress
// :1064-1237 (tiling, edge strips, serialisation), packIndexSign :76-80.
//
// mp_kernel: a workgroup of 256 threads encodes up to 8 tiles together, their residuals in
// LDS. Per pick: every 16-lane group takes atoms g, g + 16, ...; lane l accumulates the
// elements l, l + 16, ... of the dot product with one FMA chain per tile (the 16 lanes of the
// reference's two 8-wide accumulators), lanes 0..7 add the 8-element chunk, and xor-shuffles
// over 8, 4, 1, 2 lanes combine them in the reference's order (acc0 + acc1, low + high half,
// two horizontal adds): the projections are the reference's to the bit, so are the picks.
// Each D element loaded is used for every tile of the workgroup. Then one wave per tile scans
// the scores (first maximum), and the residuals are updated with one fused multiply-add per
// element.
//
// mp_gram_kernel makes the same picks without a projection per pick: scores start as tile . D^T
// and follow the residual through D . D^T, an error bound says which atoms can be the
// reference's pick, and only where that leaves more than one are the exact projections taken
// (see the comment there). launch_mp chooses between the two.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <type_traits>
#include <unordered_map>
#include <vector>

#include "common.hpp"

namespace csdr {
// fitHierarchicalKSVD's dictionary initialisation, in the reference build's arithmetic: the
// tiles picked, the factors of the atoms made from them (returns the common one), the whole of
// it on the host; and atomUpdateStep's re-seed of an atom (hsdr_init.cpp).
void hsdr_init_picks(uint32_t n, uint16_t K, std::mt19937& rng, uint32_t* src);
float hsdr_init_scales(const float* sq, uint16_t K, uint32_t slots, double mean_norm, float* unit);
void hsdr_init_dictionary(const float* tiles, uint32_t n, uint32_t C, uint16_t K, uint32_t slots,
                          float* D);
void hsdr_reseed_atom(const float* tiles, uint32_t n, uint32_t C, uint64_t base_seed, uint32_t j,
                      uint32_t mul, double target_norm, float* atom);
}  // namespace csdr

namespace {

using csdr::set_error;

constexpr int kEThreads = 256;
constexpr int kEGroups = kEThreads / 16;
constexpr int kMaxTT = 8;        // tiles per workgroup, at most
constexpr int kMaxStages = 32;
constexpr size_t kLdsSoft = 64 * 1024;    // several workgroups per CU below this
constexpr size_t kLdsHard = 160 * 1024;

struct MpArgs {
    const float* tiles;  // n x C
    const float* D;      // K x C
    uint16_t* codes;     // n x S*k, packIndexSign
    long long n;
    int C, K, S, k, tt;
    const int* list;   // mp_list_kernel: *count tiles by number
    const int* count;
    float gamma[kMaxStages];
};

// The TT tiles' residual values of one element (TT * 4 bytes, aligned to that size) in one
// or two wide LDS reads.
template <int TT>
__device__ __forceinline__ void load_tiles(const float* rc, float* rv) {
    if constexpr (TT % 4 == 0) {
#pragma unroll
        for (int t4 = 0; t4 < TT / 4; ++t4) {
            const float4 v = reinterpret_cast<const float4*>(rc)[t4];
            rv[4 * t4] = v.x;
            rv[4 * t4 + 1] = v.y;
            rv[4 * t4 + 2] = v.z;
            rv[4 * t4 + 3] = v.w;
        }
    } else if constexpr (TT == 2) {
        const float2 v = *reinterpret_cast<const float2*>(rc);
        rv[0] = v.x;
        rv[1] = v.y;
    } else {
        rv[0] = rc[0];
    }
}

// The nt tiles first, first + 1, ... or (LIST) list[first], list[first + 1], ...; kNA atoms per
// 16-lane group at a time.
template <int TT, bool LIST, int kNA = TT <= 2 ? 8 : 2>
__device__ __forceinline__ void mp_tiles(const MpArgs& a, long long first, int nt) {
    extern __shared__ __attribute__((aligned(16))) float smem[];  // (wide reads, load_tiles)
    const int tt = TT, C = a.C, K = a.K;
    float* r = smem;                                                    // C x TT residuals
    float* proj = r + (size_t)tt * C;                                   // nt x K scores
    uint8_t* used = reinterpret_cast<uint8_t*>(proj + (size_t)tt * K);  // nt x K
    __shared__ int best_s[TT];
    __shared__ float scale_s[TT];
    const auto number = [&](int t) {
        return LIST ? (long long)a.list[first + min(t, nt - 1)] : first + t;
    };
    const int tid = threadIdx.x, l16 = tid & 15, grp = tid >> 4;
    const int lane = tid & 63, wave = tid >> 6;
    // residuals tile-minor, r[c * TT + t] (one 16-byte LDS read gives four tiles' values of an
    // element); slots past nt hold zeros
    for (int i = tid; i < TT * C; i += kEThreads) {
        const int c = i / TT, t = i - c * TT;
        r[i] = t < nt ? a.tiles[number(t) * C + c] : 0.f;
    }
    // kNA: 8 with up to 2 tiles (D blocks of 4 chunks), 2 with
    // more (registers; measured 896 x 896 at 2 tiles: 0.60 ms with 2, 0.51 with 4, 0.45 with 8;
    // 4864 x 896 at 4 tiles: 3.48 ms with 2, 4.01 with 4)
    constexpr int kDB = kNA >= 4 ? 4 : 8;  // chunks of an atom loaded per block
    const int C16 = C & ~15, C8 = C & ~7;  // end of the 16-element chunks, of the 8-element one
    const int nch = C16 / 16;  // full 16-element chunks (block loads clamp into them)
    const int slots = a.S * a.k;
    for (int l = 0; l < a.S; ++l) {
        for (int i = tid; i < nt * K; i += kEThreads) used[i] = 0;
        __syncthreads();
        for (int st = 0; st < a.k; ++st) {
            // 1. projections of every tile onto every atom: the atom's values 16 chunks at
            // a time, the next block in flight while this one is used (loads clamp into the
            // row's full chunks: in bounds, uniform, so the waits stay per block); tile slots
            // past nt hold zeros and are computed too (no per-tile branches)
            // kNA atoms per group at a time (j, j + 16, ...): each residual read feeds all
            for (int j = grp; j < K; j += kNA * kEGroups) {
                const float* dj[kNA];
#pragma unroll
                for (int u = 0; u < kNA; ++u) {
                    const int ju = j + u * kEGroups;
                    dj[u] = a.D + (size_t)(ju < K ? ju : j) * C + l16;
                }
                float p[kNA][TT];
#pragma unroll
                for (int u = 0; u < kNA; ++u)
#pragma unroll
                    for (int t = 0; t < TT; ++t) p[u][t] = 0.f;
                float cv[kNA][kDB], nv[kNA][kDB];
#pragma unroll
                for (int u = 0; u < kNA; ++u)
#pragma unroll
                    for (int q = 0; q < kDB; ++q) cv[u][q] = nch ? dj[u][min(q, nch - 1) * 16] : 0.f;
                for (int b0 = 0; b0 < nch; b0 += kDB) {
#pragma unroll
                    for (int u = 0; u < kNA; ++u)
#pragma unroll
                        for (int q = 0; q < kDB; ++q)
                            nv[u][q] = dj[u][min(b0 + kDB + q, nch - 1) * 16];
#pragma unroll
                    for (int q = 0; q < kDB; ++q) {
                        if (b0 + q >= nch) break;
                        float rv[TT];
                        load_tiles<TT>(r + ((b0 + q) * 16 + l16) * TT, rv);
#pragma unroll
                        for (int u = 0; u < kNA; ++u)
#pragma unroll
                            for (int t = 0; t < TT; ++t) p[u][t] = fmaf(cv[u][q], rv[t], p[u][t]);
                    }
#pragma unroll
                    for (int u = 0; u < kNA; ++u)
#pragma unroll
                        for (int q = 0; q < kDB; ++q) cv[u][q] = nv[u][q];
                }
                if (C8 > C16 && l16 < 8) {
                    const float* rc = r + (C16 + l16) * TT;
#pragma unroll
                    for (int u = 0; u < kNA; ++u) {
                        const float dv = dj[u][C16];
#pragma unroll
                        for (int t = 0; t < TT; ++t) p[u][t] = fmaf(dv, rc[t], p[u][t]);
                    }
                }
#pragma unroll
                for (int u = 0; u < kNA; ++u) {
                    const int ju = j + u * kEGroups;
                    const float* dt = dj[u] - l16;  // the atom's row
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        float v = p[u][t];
                        v += __shfl_xor(v, 8, 16);  // acc0 + acc1
                        v += __shfl_xor(v, 4, 16);  // low + high 128 bits
                        v += __shfl_xor(v, 1, 16);  // horizontal add
                        v += __shfl_xor(v, 2, 16);  // horizontal add
                        // the last C % 8 elements: the scalar tail, in element order
                        for (int c = C8; c < C; ++c) v = fmaf(dt[c], r[c * TT + t], v);
                        if (l16 == 0 && t < nt && ju < K)
                            proj[t * K + ju] = used[t * K + ju] ? 0.0f : v;
                    }
                }
            }
            __syncthreads();
            // 2. the pick per tile: first maximum of |score|, as the reference's scan
            for (int t = wave; t < nt; t += kEThreads / 64) {
                float bv = 0.f;
                int bi = 0;
                for (int j = lane; j < K; j += 64) {
                    const float av = fabsf(proj[t * K + j]);
                    if (av > bv) {
                        bv = av;
                        bi = j;
                    }
                }
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) {
                    const float ov = __shfl_xor(bv, off, 64);
                    const int oi = __shfl_xor(bi, off, 64);
                    if (ov > bv || (ov == bv && oi < bi)) {
                        bv = ov;
                        bi = oi;
                    }
                }
                if (lane == 0) {
                    const int sg = proj[t * K + bi] >= 0.0f ? 1 : -1;
                    a.codes[(size_t)number(t) * slots + l * a.k + st] =
                        (uint16_t)((bi & 0x7FFF) | (sg < 0 ? 0x8000 : 0));
                    used[t * K + bi] = 1;
                    best_s[t] = bi;
                    scale_s[t] = a.gamma[l] * (float)sg;
                }
            }
            __syncthreads();
            // 3. r -= scale * D[best], fused
            for (int i = tid; i < nt * C; i += kEThreads) {
                const int t = i / C, c = i - t * C;
                float& rv = r[c * TT + t];
                rv = fmaf(-a.D[(size_t)best_s[t] * C + c], scale_s[t], rv);
            }
            __syncthreads();
        }
    }
}

template <int TT>
__global__ __launch_bounds__(kEThreads) void mp_kernel(MpArgs a) {
    const long long t0 = (long long)blockIdx.x * TT;
    mp_tiles<TT, false>(a, t0, (int)min((long long)TT, a.n - t0));
}

// The tiles that mp_gram_kernel leaves (list, count): one a workgroup up to kListFew of them,
// where a pick is a chain of round trips; past that (equal or parallel rows, whose atoms are all
// alike) TT at a time as mp_kernel takes them, since every workgroup reads all of D per pick and
// L2's rate bounds it (4864 x 896, K = 512, 24 picks, rows of one value each: 9.3 ms with one tile a
// workgroup throughout, 3.7 here, 3.4 with mp_kernel alone). With TT = 2, what mp_kernel takes
// below 4096 tiles, one at a time stays the faster (600 x 128, K = 512, 4 picks 103 us, 124).
// Beside the other form single tiles take 4 atoms at a time, and that form has a workgroup for
// every TT tiles that may be left: with 8, or with a loop, the registers leave it fewer waves (5.3
// ms).
constexpr int kListFew = 256;

template <int TT>
__global__ __launch_bounds__(kEThreads) void mp_list_kernel(MpArgs a) {
    const int n = *a.count;
    if constexpr (TT == 1) {
        for (int b = blockIdx.x; b < n; b += gridDim.x) mp_tiles<1, true>(a, b, 1);
    } else {
        const int b = blockIdx.x;
        if (n <= kListFew) {
            if (b < n) mp_tiles<1, true, 4>(a, b, 1);
        } else if (b * TT < n) {
            mp_tiles<TT, true>(a, b * TT, min(TT, n - b * TT));
        }
    }
}

size_t mp_lds_bytes(int tt, int C, int K) {
    return (size_t)tt * ((size_t)C + K) * 4 + csdr::align_up((size_t)tt * K, 16);
}

// Tiles per workgroup: about n / 1024, at least 2 (measured on the Qwen2-0.5B shapes, 1-row
// tiles: 896 x 896 best at 2 (0.93 ms vs 1.00 at 4, 1.31 at 8), 4864 x 896 at 4 (4.5 ms vs 5.0
// at 8, 7.3 at 2): enough workgroups per CU to hide latency, and every workgroup reads all of
// D once per pick, so more tiles each is less D traffic), a power of two, at most 8 and what
// fits under the soft LDS size; else one tile under the hard size; else 0 (too large).
int mp_tiles_per_wg(long long n, int C, int K) {
    const char* ev = std::getenv("CSDR_HSDR_TILES_PER_WG");  // tuning override: 1, 2, 4 or 8
    long long want = std::min<long long>(kMaxTT, std::max<long long>(2, n / 1024));
    if (ev && std::atoi(ev) >= 1) want = std::min(kMaxTT, std::atoi(ev));
    for (int tt = kMaxTT; tt >= 1; tt >>= 1)  // a power of two (the kernel's template)
        if (tt <= want && mp_lds_bytes(tt, C, K) <= kLdsSoft) return tt;
    return mp_lds_bytes(1, C, K) <= kLdsHard ? 1 : 0;
}

// ---------------------------------------------------------------- picks through the Gram matrix

// mp_kernel's K x C projections per tile and pick bound it (36% of the fp32 vector rate). The
// scores of the next residual are the last ones minus gamma sign (D . D^T)[best], K operations
// instead of K x C, so here a pick is one row of D . D^T per tile. The picks stay the
// reference's because its rounding is bounded. With u = 2^-24, N_t the residual's norm, dmax
// the longest atom's:
//   * the reference's projection: at most c1 = C / 16 + 16 roundings on any element's way, so
//     within c1 u dmax N_t of the true dot product with its residual;
//   * its residual: one rounding per element and pick, t u max N off the true one;
//   * the scores here: sums in double rounded to float once (u dmax N_0 and, through the Gram
//     entries, u dmax sum gamma |D_b|), one rounding per pick (t u dmax max N).
// Their sum is eps. An atom whose score is more than 2 eps below the largest cannot be the
// pick; a single one left is, with the sign of its score once that exceeds eps. Otherwise
// (about one pick in 500 on Gaussian tiles, more where D holds an atom twice) the wave brings
// the residual up to date in LDS with the reference's own fused updates and takes the left
// atoms' projections in its order, as mp_kernel does. A tile whose norm or atoms are outside
// [1e-12, 1e12], NaN or infinite, or with more than kGramMaxCand atoms left, goes to a list
// that mp_list_kernel encodes.
// One wave per tile: the scores (KPL per lane) stay in registers, a Gram row is KPL coalesced
// loads from L2, and a pick is bound by that one round trip and the wave's maximum.
// 4864 x 896, K = 512, 24 picks, with both products: 3.9 ms -> 0.30 ms (picks 119 us, scores
// about 115, D . D^T about 40); 896 x 896, K = 256, 15 picks: 807 -> 155 us; 3000 x 4096,
// K = 1024, 8 picks: 12.2 -> 1.0 ms; 300 x 39, K = 48: 74 -> 44 us.
constexpr int kGramMaxK = 2048;      // 32 scores per lane
constexpr int kGramMaxC = 8192;      // residual in LDS: 32 KiB per wave
constexpr int kGramMaxCand = 64;
constexpr size_t kGramScoreBytes = 64u << 20;  // scores of one chunk of tiles

struct GramArgs {
    const float* tiles;   // n x C
    const float* D;       // K x C
    const float* scores;  // n x K: tile . D^T
    const float* gram;    // K x K: D . D^T
    const float* sq;      // K: its diagonal
    uint16_t* codes;      // n x S*k
    int* list;            // tiles left to mp_list_kernel, and their count
    int* count;
    int C, K, S, k;
    float gamma[kMaxStages];
};

// out (M x R) = X (M x C) . W^T (W R x C) with the sums in double (v_mfma_f64_16x16x4_f64),
// rounded to float. A 64 x 64 tile per 2 x 2 waves, 32-deep stages through LDS with the next
// stage's loads in flight; the k order within a stage is permuted (step s of lane group g takes
// k = 8 g + s) so that a lane reads its eight values as one 32-byte run.
constexpr int kPLd = 36;
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

template <bool VEC>
__device__ __forceinline__ floatx4 load4(const float* p, int k, int C) {
    if constexpr (VEC)
        return k < C ? *reinterpret_cast<const floatx4*>(p + k) : floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = k + i < C ? p[k + i] : 0.f;
    return v;
}

template <bool VEC>
__global__ __launch_bounds__(kEThreads) void dots_f64_kernel(const float* __restrict__ X,
                                                             long long M,
                                                             const float* __restrict__ W, int R,
                                                             int C, float* __restrict__ out,
                                                             float* diag, int* zero) {
    __shared__ __attribute__((aligned(16))) float xs[64 * kPLd];
    __shared__ __attribute__((aligned(16))) float ws[64 * kPLd];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (zero && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) *zero = 0;
    const int li = lane & 15, lg = lane >> 4;
    const long long m0 = (long long)blockIdx.x * 64;
    const int r0 = blockIdx.y * 64;
    const int wm = (wave >> 1) * 32, wr = (wave & 1) * 32;
    const int row = tid >> 3, kq = (tid & 7) * 4;  // and row + 32
    const float* xp[2];
    const float* wp[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // rows past the end repeat the last one (not stored)
        xp[j] = X + (size_t)min(m0 + row + 32 * j, M - 1) * C;
        wp[j] = W + (size_t)min(r0 + row + 32 * j, R - 1) * C;
    }
    floatx4 px[2], pw[2];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            px[j] = load4<VEC>(xp[j], k0 + kq, C);
            pw[j] = load4<VEC>(wp[j], k0 + kq, C);
        }
    };
    doublex4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = doublex4{0., 0., 0., 0.};
    const int nst = (C + 31) / 32;
    load(0);
    for (int s = 0; s < nst; ++s) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            *reinterpret_cast<floatx4*>(xs + (row + 32 * j) * kPLd + kq) = px[j];
            *reinterpret_cast<floatx4*>(ws + (row + 32 * j) * kPLd + kq) = pw[j];
        }
        __syncthreads();
        if (s + 1 < nst) load((s + 1) * 32);
        floatx4 xf[2][2], wf[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                xf[a][h] = *reinterpret_cast<const floatx4*>(xs + (wm + a * 16 + li) * kPLd +
                                                             lg * 8 + 4 * h);
                wf[a][h] = *reinterpret_cast<const floatx4*>(ws + (wr + a * 16 + li) * kPLd +
                                                             lg * 8 + 4 * h);
            }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const double x0 = xf[0][q >> 2][q & 3], x1 = xf[1][q >> 2][q & 3];
            const double w0 = wf[0][q >> 2][q & 3], w1 = wf[1][q >> 2][q & 3];
            acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x0, w0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x0, w1, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1, w0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1, w1, acc[1][1], 0, 0, 0);
        }
    }
    // the f64 form: lane holds D[4 v + l / 16][l % 16], X rows along the MFMA's rows
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int r = r0 + wr + b * 16 + li;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const long long m = m0 + wm + a * 16 + 4 * v + lg;
                if (m < M && r < R) {
                    out[(size_t)m * R + r] = (float)acc[a][b][v];
                    if (diag && m == r) diag[r] = (float)acc[a][b][v];
                }
            }
        }
}

// max over the wave of values >= 0 (NaN dropped), in every lane: DPP rows, then broadcasts
__device__ __forceinline__ float wave_max(float v) {
    const auto step = [&](auto ctrl, auto rows) {
        const int o = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                  decltype(ctrl)::value, decltype(rows)::value,
                                                  0xf, false);
        v = fmaxf(v, __builtin_bit_cast(float, o));
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});  // row_shr 1, 2, 4, 8
    step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});  // row 0 / 2 into 1 / 3
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});  // row 1 into 2, 3
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

template <int KPL>
__global__ __launch_bounds__(64) void mp_gram_kernel(GramArgs a) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int C = a.C, K = a.K, lane = threadIdx.x, slots = a.S * a.k;
    float* r = smem;                                           // C: the exact residual, when needed
    float* hgam = r + C;                                       // slots: gamma * sign of the picks
    uint16_t* hist = reinterpret_cast<uint16_t*>(hgam + slots);  // and their atoms
    uint16_t* cand = hist + ((slots + 1) & ~1);                // kGramMaxCand: atoms left
    const int tile = blockIdx.x;
    const float* x = a.tiles + (size_t)tile * C;
    float s[KPL];
    uint32_t out_of = 0;  // atoms past K
    int jc[KPL];          // this lane's atoms, clamped
#pragma unroll
    for (int i = 0; i < KPL; ++i) {
        const int j = lane + 64 * i;
        jc[i] = min(j, K - 1);
        s[i] = a.scores[(size_t)tile * K + jc[i]];
        if (j >= K) out_of |= 1u << i;
    }
    float dm = 0.f;
    bool odd = false;  // NaN or infinite (fmaxf would drop a NaN)
    for (int j = lane; j < K; j += 64) {
        const float g = a.sq[j];
        dm = fmaxf(dm, g);
        odd |= !(g >= 0.f);
    }
    const float dmax = __builtin_amdgcn_sqrtf(wave_max(dm)) * 1.01f;
    // the tile's norm, scaled by its largest magnitude
    float mx = 0.f;
    for (int c = lane; c < C; c += 64) {
        mx = fmaxf(mx, fabsf(x[c]));
        odd |= !(fabsf(x[c]) < INFINITY);
    }
    mx = wave_max(mx);
    float n2 = 0.f;
    if (mx > 0.f)
        for (int c = lane; c < C; c += 64) {
            const float v = x[c] / mx;
            n2 = fmaf(v, v, n2);
        }
    const float n0 = mx > 0.f ? mx * __builtin_amdgcn_sqrtf(csdr::wave_sum(n2)) * 1.01f : 0.f;
    const auto leave = [&] {
        if (lane == 0) a.list[atomicAdd(a.count, 1)] = tile;
    };
    if (__any(odd) || !(dmax >= 1e-12f && dmax <= 1e12f) ||
        !(n0 == 0.f || (n0 >= 1e-12f && n0 <= 1e12f))) {
        leave();
        return;
    }
    // a zero tile whose first pick, atom 0, is all zeros too stays zero: atom 0 at every pick
    if (n0 == 0.f) {
        bool live = false;
        for (int c = lane; c < C; c += 64) live |= a.D[c] != 0.f;
        for (int l = 0; l < a.S; ++l) live |= !(fabsf(a.gamma[l]) < INFINITY);  // 0 * inf
        if (!__any(live)) {
            for (int q = lane; q < slots; q += 64) a.codes[(size_t)tile * slots + q] = 0;
            return;
        }
    }
    const float u = 1.25f * 5.9604645e-8f * dmax;
    float rn2 = n0 * n0, nmax2 = rn2, len = 0.f;
    int upto = -1;  // picks applied to r (-1: r not loaded)
    int t = 0;
    for (int l = 0; l < a.S; ++l) {
        uint32_t used = out_of;
        const float gl = a.gamma[l];
        for (int st = 0; st < a.k; ++st, ++t) {
            float v[KPL];  // |score|, -1 for atoms used in this stage
            float m = 0.f;
#pragma unroll
            for (int i = 0; i < KPL; ++i) {
                v[i] = used >> i & 1 ? -1.f : fabsf(s[i]);
                m = fmaxf(m, v[i]);
            }
            m = wave_max(m);
            const float nmax = __builtin_amdgcn_sqrtf(nmax2) * 1.01f;
            const float nt =
                __builtin_amdgcn_sqrtf(rn2 + (1e-4f + 1e-6f * (float)t) * nmax2) * 1.01f;
            const float eps =
                u * ((float)(C / 16 + 16) * nt + (float)(2 * t) * nmax + n0 + len) + 1e-38f;
            if (!(m <= 1e30f && len <= 1e15f && eps < 1e30f)) {
                leave();
                return;
            }
            const float thr = m - 2.f * eps;
            // the atoms left: NaN stays in; a used one's -1 may only come in with thr < -1,
            // where eps is far past any score
            uint64_t left[KPL];
            int nc = 0;
#pragma unroll
            for (int i = 0; i < KPL; ++i) {
                left[i] = __ballot(!(v[i] < thr) && !(used >> i & 1));
                nc += __popcll(left[i]);
            }
            int bi = 0, sg = 1;
            if (nc == 1 && m > eps) {
                float sv = 0.f;
#pragma unroll
                for (int i = 0; i < KPL; ++i)
                    if (left[i]) {  // one of them
                        const int src = __ffsll((unsigned long long)left[i]) - 1;
                        bi = 64 * i + src;
                        sv = __builtin_bit_cast(
                            float,
                            __builtin_amdgcn_readlane(__builtin_bit_cast(int, s[i]), src));
                    }
                sg = sv >= 0.f ? 1 : -1;
            } else if (n0 == 0.f && t == 0) {
                // a zero tile: every projection is 0, atom 0 stands
            } else if (nc > kGramMaxCand) {
                leave();
                return;
            } else {
                // the residual up to date, as the reference updates it; four elements a lane
                // at a time, so that every pick's loads are independent of the last one's
                for (int c0 = lane; c0 < C; c0 += 256) {
                    float rv[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        rv[e] = upto < 0 ? x[min(c0 + 64 * e, C - 1)] : r[min(c0 + 64 * e, C - 1)];
#pragma unroll 4
                    for (int q = max(upto, 0); q < t; ++q) {
                        const uint16_t h = hist[q];
                        const float sc = hgam[q];
                        const float* d = a.D + (size_t)h * C;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            rv[e] = fmaf(-d[min(c0 + 64 * e, C - 1)], sc, rv[e]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (c0 + 64 * e < C) r[c0 + 64 * e] = rv[e];
                }
                upto = t;
                int n = 0;  // the atoms left, in ascending order
#pragma unroll
                for (int i = 0; i < KPL; ++i) {
                    if (left[i] >> lane & 1)
                        cand[n + __popcll(left[i] & ((1ull << lane) - 1))] =
                            (uint16_t)(lane + 64 * i);
                    n += __popcll(left[i]);
                }
                __syncthreads();
                // their projections in the reference's order, one per 16 lanes
                const int l16 = lane & 15, grp = lane >> 4;
                const int C16 = C & ~15, C8 = C & ~7;
                float bv = 0.f;  // sg: atom 0 used in this stage scores 0, a positive sign
                for (int q = 0; q < nc; q += 4) {
                    const int j = cand[min(q + grp, nc - 1)];
                    const float* d = a.D + (size_t)j * C;
                    float p = 0.f;
#pragma unroll 8
                    for (int c = l16; c < C16; c += 16) p = fmaf(d[c], r[c], p);
                    if (C8 > C16 && l16 < 8) p = fmaf(d[C16 + l16], r[C16 + l16], p);
                    p += __shfl_xor(p, 8, 16);
                    p += __shfl_xor(p, 4, 16);
                    p += __shfl_xor(p, 1, 16);
                    p += __shfl_xor(p, 2, 16);
                    for (int c = C8; c < C; ++c) p = fmaf(d[c], r[c], p);
                    if (fabsf(p) > bv) {  // ascending within a group: the first maximum
                        bv = fabsf(p);
                        bi = j;
                        sg = p >= 0.f ? 1 : -1;
                    } else if (j == 0 && bv == 0.f) {
                        sg = p >= 0.f ? 1 : -1;
                    }
                }
                // group 0 holds atom 0 when it is left: with no score above 0 its sign stands
#pragma unroll
                for (int off = 16; off <= 32; off <<= 1) {
                    const float ov = __shfl_xor(bv, off, 64);
                    const int oi = __shfl_xor(bi, off, 64), os = __shfl_xor(sg, off, 64);
                    if (ov > bv || (ov == bv && (oi < bi || (ov == 0.f && os < sg)))) {
                        bv = ov;
                        bi = oi;
                        sg = os;
                    }
                }
                bi = __builtin_amdgcn_readfirstlane(bi);
                sg = __builtin_amdgcn_readfirstlane(sg);
            }
            const float sc = gl * (float)sg;
            const float* g = a.gram + (size_t)bi * K;
            const float gb = a.sq[bi];
            float sb = 0.f;
#pragma unroll
            for (int i = 0; i < KPL; ++i) {
                if (i == bi >> 6)
                    sb = __builtin_bit_cast(
                        float,
                        __builtin_amdgcn_readlane(__builtin_bit_cast(int, s[i]), bi & 63));
                s[i] = fmaf(-sc, g[jc[i]], s[i]);
            }
            if (lane == (bi & 63)) used |= 1u << (bi >> 6);
            if (lane == 0) {
                a.codes[(size_t)tile * slots + t] =
                    (uint16_t)((bi & 0x7FFF) | (sg < 0 ? 0x8000 : 0));
                hist[t] = (uint16_t)bi;
                hgam[t] = sc;
            }
            rn2 += sc * (sc * gb - 2.f * sb);
            rn2 = rn2 >= 0.f ? rn2 : rn2 < 0.f ? 0.f : INFINITY;  // NaN: the tile leaves
            len += fabsf(sc) * __builtin_amdgcn_sqrtf(gb) * 1.01f;
            nmax2 = fmaxf(nmax2, rn2);
            __syncthreads();  // hist and cand before the next pick's reads and writes
        }
    }
}

// Workspace of the Gram path: the scores of a chunk of tiles, the Gram matrix, its
// diagonal, the numbers of a chunk's tiles left to mp_list_kernel and their count.
long long gram_chunk(long long n, int K) {
    return std::min<long long>(n, std::max<long long>(64, (long long)(kGramScoreBytes / 4) / K));
}
size_t gram_ws_bytes(long long n, int K) {
    const size_t chunk = (size_t)gram_chunk(n, K);
    return csdr::align_up(chunk * K * 4, 256) + csdr::align_up((size_t)K * K * 4, 256) +
           ((size_t)K + chunk + 1) * 4;
}

// mp_gram_kernel's LDS: the residual, the picks with their gains, the atoms left.
size_t gram_lds_bytes(int C, int S, int k) {
    const size_t slots = (size_t)S * k;
    return ((size_t)C + slots) * 4 + (((slots + 1) & ~(size_t)1) + kGramMaxCand) * 2;
}

// The Gram path does 2 (n + K) K C operations where mp_kernel does 2 n picks K C. It keeps every
// pick in LDS, mp_kernel none: more of them than fit in 64 KiB stay with that.
bool gram_pays(long long n, int C, int K, int S, int k) {
    return K <= kGramMaxK && C <= kGramMaxC && 2 * n * S * k >= n + K &&
           gram_lds_bytes(C, S, k) <= 64 * 1024 &&
           !std::getenv("CSDR_HSDR_TILES_PER_WG");  // that override names mp_kernel's form
}

int launch_dots(const float* X, long long M, const float* W, int R, int C, float* out,
                float* diag, int* zero, hipStream_t st) {
    const dim3 grid((unsigned)((M + 63) / 64), (unsigned)((R + 63) / 64));
    if (C % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(W) % 16 == 0)
        dots_f64_kernel<true><<<grid, kEThreads, 0, st>>>(X, M, W, R, C, out, diag, zero);
    else
        dots_f64_kernel<false><<<grid, kEThreads, 0, st>>>(X, M, W, R, C, out, diag, zero);
    CSDR_LAUNCH_CHECK("hsdr_encode products");
    return CSDR_OK;
}

int launch_mp_gram(const float* tiles, long long n, int C, const float* D, int K, int S, int k,
                   const float* gamma, uint16_t* codes, void* ws, hipStream_t st) {
    const long long chunk = gram_chunk(n, K);
    char* w = static_cast<char*>(ws);
    float* scores = reinterpret_cast<float*>(w);
    w += csdr::align_up((size_t)chunk * K * 4, 256);
    float* gram = reinterpret_cast<float*>(w);
    w += csdr::align_up((size_t)K * K * 4, 256);
    float* sq = reinterpret_cast<float*>(w);
    int* count = reinterpret_cast<int*>(sq + K);
    int rc = launch_dots(D, K, D, K, C, gram, sq, nullptr, st);
    if (rc != CSDR_OK) return rc;
    GramArgs a{};
    MpArgs b{};
    a.D = b.D = D;
    a.scores = scores;
    a.gram = gram;
    a.sq = sq;
    a.C = b.C = C;
    a.K = b.K = K;
    a.S = b.S = S;
    a.k = b.k = k;
    a.count = count;
    a.list = count + 1;
    b.count = count;
    b.list = count + 1;
    for (int l = 0; l < S; ++l) a.gamma[l] = b.gamma[l] = gamma[l];
    const size_t lds = gram_lds_bytes(C, S, k);
    const int tt = mp_tiles_per_wg(n, C, K);
    const int list_tt = tt >= 4 ? tt : 1;
    const size_t list_lds = mp_lds_bytes(list_tt, C, K);  // (no more than the soft limit)
    for (long long t0 = 0; t0 < n; t0 += chunk) {
        const long long nt = std::min(chunk, n - t0);
        a.tiles = b.tiles = tiles + (size_t)t0 * C;
        a.codes = b.codes = codes + (size_t)t0 * S * k;
        b.n = nt;
        rc = launch_dots(a.tiles, nt, D, K, C, scores, nullptr, count, st);
        if (rc != CSDR_OK) return rc;
        const unsigned grid = (unsigned)nt;
        if (K <= 256) mp_gram_kernel<4><<<grid, 64, lds, st>>>(a);
        else if (K <= 512) mp_gram_kernel<8><<<grid, 64, lds, st>>>(a);
        else if (K <= 1024) mp_gram_kernel<16><<<grid, 64, lds, st>>>(a);
        else mp_gram_kernel<32><<<grid, 64, lds, st>>>(a);
        const long long lgrid = list_tt == 1
                                    ? std::min<long long>(nt, 1024)
                                    : std::max<long long>((nt + list_tt - 1) / list_tt,
                                                          std::min<long long>(nt, kListFew));
        if (list_tt == 8) mp_list_kernel<8><<<(unsigned)lgrid, kEThreads, list_lds, st>>>(b);
        else if (list_tt == 4) mp_list_kernel<4><<<(unsigned)lgrid, kEThreads, list_lds, st>>>(b);
        else mp_list_kernel<1><<<(unsigned)lgrid, kEThreads, list_lds, st>>>(b);
        CSDR_LAUNCH_CHECK("hsdr_encode");
    }
    return CSDR_OK;
}

int check_mp_shape(long long n, int C, int K, int S, int k) {
    if (n < 0 || C <= 0 || K <= 0 || S <= 0 || k <= 0)
        return set_error(CSDR_E_INVALID, "hsdr_encode: bad shape");
    if (K > 32768) return set_error(CSDR_E_UNSUPPORTED, "hsdr_encode: at most 32768 atoms");
    if (S > kMaxStages) return set_error(CSDR_E_UNSUPPORTED, "hsdr_encode: at most 32 stages");
    if (k > K) return set_error(CSDR_E_INVALID, "hsdr_encode: more picks per stage than atoms");
    if (mp_tiles_per_wg(n, C, K) == 0)
        return set_error(CSDR_E_UNSUPPORTED, "hsdr_encode: tile and dictionary exceed LDS");
    return CSDR_OK;
}

// gram_ws: gram_ws_bytes(n, K) of device memory, or NULL for mp_kernel.
int launch_mp(const float* tiles, long long n, int C, const float* D, int K, int S, int k,
              const float* gamma, uint16_t* codes, void* gram_ws, hipStream_t st) {
    if (n == 0) return CSDR_OK;
    if (gram_ws) return launch_mp_gram(tiles, n, C, D, K, S, k, gamma, codes, gram_ws, st);
    MpArgs a{};
    a.tiles = tiles;
    a.D = D;
    a.codes = codes;
    a.n = n;
    a.C = C;
    a.K = K;
    a.S = S;
    a.k = k;
    a.tt = mp_tiles_per_wg(n, C, K);
    for (int l = 0; l < S; ++l) a.gamma[l] = gamma[l];
    const size_t lds = mp_lds_bytes(a.tt, C, K);
    const long long grid = (n + a.tt - 1) / a.tt;
    if (grid > 0x7fffffffLL) return set_error(CSDR_E_UNSUPPORTED, "hsdr_encode: too many tiles");
    auto go = [&](auto kern) {
        if (lds > 64 * 1024)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        kern<<<(unsigned)grid, kEThreads, lds, st>>>(a);
    };
    switch (a.tt) {
        case 8: go(&mp_kernel<8>); break;
        case 4: go(&mp_kernel<4>); break;
        case 2: go(&mp_kernel<2>); break;
        default: go(&mp_kernel<1>); break;
    }
    CSDR_LAUNCH_CHECK("hsdr_encode");
    return CSDR_OK;
}

// ---------------------------------------------------------------- K-SVD atom update

// atomUpdateStep (HierarchicalSDRStrategy.cpp:281-490) on the device, per refinement pass:
//  users_count / scan / fill: every atom's users in (tile, slot) order (:325-339) with their
//    sign * gamma, and 0.5 / the sum of gamma^2 over them in that order (fused, :428-437; 0
//    when the sum is <= 1e-12). Counts by LDS histograms, one workgroup scans them, and one
//    workgroup per atom then walks all codes: thread t takes the t-th run of them, counts its
//    users, and writes them behind those of the threads before it. On the host this was a
//    copy of the codes, a synchronisation and 0.5 ms per pass;
//  residual_kernel: residual = tile - sum over slots of gamma_l * sign * D[idx], slots in
//    order, each term fused (the reference's r[c] += scale * atom[c], :300-311), then tile -
//    recon (:316-320). A workgroup per tile: its codes are uniform (scalar loads) and a thread
//    keeps 4 elements, with the next slots' atom rows in flight (84 -> 24 us at 4864 x 896,
//    24 slots: a thread per element with a 64-bit division each). Short tiles share one, 16
//    threads each up to 64 elements and 64 up to 256 (16384 8 x 8 tiles 26 us a thread per
//    element, 18.6 a workgroup each, 8.3 here; 32768 4 x 4 tiles 14.2, 34.6, 11.6);
//  atom_sum_kernel: correction[c] = sum over the atom's users, in order, of sign * gamma *
//    residual (double, fused: :428-437), the new value atom + correction * (0.5 / sum gamma^2)
//    rounded to float (:448-458), in the atom's place (one that is not finite is re-seeded
//    whole). One thread per element; the users' rows are L2 reads whose
//    latency bounds it, so a workgroup takes 256 elements of one atom (K x C / 256 of them)
//    and eight rows are in flight;
//  atom_finish_kernel: per atom, a non-finite value flags it for the host's re-seed (:461), the
//    squared norm is summed in element order as the reference's loop does (:456), and atoms
//    longer than the cap are scaled back to the target norm (:482-487). Atoms without users
//    are re-seeded by the host (:411-425). Sum and finish: 273 -> 34 + 15 us at K = 512.
struct FitArgs {
    const float* tiles;
    const uint16_t* codes;
    float* D;
    float* res;     // n x C
    int* off;       // K + 1
    uint32_t* utile;
    double* ucoef;
    double* inv_w;  // K
    uint8_t* flag;  // K
    long long n, ncodes;
    int C, K, S, k;
    double cap, target;
    float gamma[kMaxStages];
};

__global__ __launch_bounds__(kEThreads) void users_count_kernel(FitArgs a) {
    extern __shared__ int hist_s[];
    for (int j = threadIdx.x; j < a.K; j += kEThreads) hist_s[j] = 0;
    __syncthreads();
    for (long long i = (long long)blockIdx.x * kEThreads + threadIdx.x; i < a.ncodes;
         i += (long long)gridDim.x * kEThreads)
        atomicAdd(&hist_s[a.codes[i] & 0x7FFF], 1);
    __syncthreads();
    for (int j = threadIdx.x; j < a.K; j += kEThreads)
        if (hist_s[j]) atomicAdd(&a.off[j + 1], hist_s[j]);
}

// Exclusive prefix sum over `v` of a 256-thread workgroup; the total in *total.
__device__ __forceinline__ int block_scan(int v, int* total) {
    __shared__ int wsum[kEThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int before = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < kEThreads / 64; ++w) {
        if (w < wave) before += wsum[w];
        sum += wsum[w];
    }
    __syncthreads();
    *total = sum;
    return before + x - v;
}

__global__ __launch_bounds__(kEThreads) void users_zero_kernel(FitArgs a) {
    for (int j = blockIdx.x * kEThreads + threadIdx.x; j <= a.K; j += gridDim.x * kEThreads)
        a.off[j] = 0;
}

__global__ __launch_bounds__(kEThreads) void users_scan_kernel(FitArgs a) {
    int base = 0;
    for (int j0 = 0; j0 < a.K; j0 += kEThreads) {
        const int j = j0 + threadIdx.x;
        const int c = j < a.K ? a.off[j + 1] : 0;
        int total;
        const int e = block_scan(c, &total);
        if (j < a.K) a.off[j + 1] = base + e + c;
        base += total;
    }
}

// Bound by the codes' way from L2: 64 of them (a 128-byte line) are in flight per thread and the
// first walk keeps its finds in LDS, so that the second one is needed only by a thread with more
// than kFillHits of them (4864 x 896, 24 slots, K = 512: 66 us with one 16-byte load in flight and
// two walks, 31 here; eight reads at a time for the sum of gamma^2 changed
// nothing).
constexpr int kFillHits = 8;

__global__ __launch_bounds__(kEThreads) void users_fill_kernel(FitArgs a) {
    __shared__ double gm_s[kEThreads];
    __shared__ uint32_t hit_s[kFillHits][kEThreads];  // 2 x position in the run + sign
    const int j = blockIdx.x, tid = threadIdx.x;
    const int u0 = a.off[j], u1 = a.off[j + 1];
    const int slots = a.S * a.k;
    const uint32_t want = (uint32_t)j;
    // runs of a multiple of 8 codes, read 16 bytes at a time (codes is 16-byte aligned)
    const long long run = (a.ncodes + (long long)kEThreads * 8 - 1) / (kEThreads * 8) * 8;
    const long long i0 = min(tid * run, a.ncodes);
    const int len = (int)(min(i0 + run, a.ncodes) - i0);
    const uint16_t* cd = a.codes + i0;
    auto walk = [&](auto&& use) {
        const int len8 = len & ~7;
        for (int i = 0; i < len8; i += 64) {  // pieces past the last one: that one, not looked at
            uint4 w[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                w[q] = *reinterpret_cast<const uint4*>(cd + min(i + 8 * q, len8 - 8));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t found = 0;
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const uint4& v = w[4 * h + q / 4];
                    const uint32_t x = q % 4 == 0 ? v.x : q % 4 == 1 ? v.y : q % 4 == 2 ? v.z : v.w;
                    found |= (x & 0x7FFF) == want ? 1u << (2 * q) : 0u;
                    found |= (x >> 16 & 0x7FFF) == want ? 2u << (2 * q) : 0u;
                }
                const int left = len8 - i - 32 * h;
                if (left < 32) found &= left > 0 ? (1u << left) - 1 : 0u;
                for (; found; found &= found - 1) use(i + 32 * h + __ffs(found) - 1);
            }
        }
        for (int i = len8; i < len; ++i)
            if ((cd[i] & 0x7FFFu) == want) use(i);
    };
    int mine = 0;
    if (u1 > u0)
        walk([&](int i) {
            if (mine < kFillHits) hit_s[mine][tid] = 2u * i + (cd[i] >> 15);
            ++mine;
        });
    int total;
    int p = u0 + block_scan(mine, &total);
    auto put_user = [&](int i, bool neg) {
        const long long tile = (i0 + i) / slots;
        const double gm = (double)a.gamma[(int)(i0 + i - tile * slots) / a.k];
        a.utile[p] = (uint32_t)tile;
        a.ucoef[p] = neg ? -gm : gm;
        ++p;
    };
    if (mine <= kFillHits) {
        for (int q = 0; q < mine; ++q) put_user(hit_s[q][tid] >> 1, hit_s[q][tid] & 1);
    } else {
        walk([&](int i) { put_user(i, cd[i] >> 15); });
    }
    __syncthreads();
    double w = 0.0;  // thread 0
    for (int b = u0; b < u1; b += kEThreads) {
        gm_s[tid] = b + tid < u1 ? a.ucoef[b + tid] : 0.0;
        __syncthreads();
        if (tid == 0)
            for (int q = 0; q < min(kEThreads, u1 - b); ++q) w = fma(gm_s[q], gm_s[q], w);
        __syncthreads();
    }
    if (tid == 0) a.inv_w[j] = w <= 1e-12 ? 0.0 : 0.5 / w;
}

template <int LPT>
__global__ __launch_bounds__(kEThreads) void residual_kernel(FitArgs a) {
    const int slots = a.S * a.k;
    const long long tile =
        LPT == kEThreads ? blockIdx.x
                         : (long long)blockIdx.x * (kEThreads / LPT) + threadIdx.x / LPT;
    if (tile >= a.n) return;
    const uint16_t* cd = a.codes + (size_t)tile * slots;
    const float* x = a.tiles + (size_t)tile * a.C;
    float* out = a.res + (size_t)tile * a.C;
    for (int c0 = threadIdx.x % LPT; c0 < a.C; c0 += 4 * LPT) {
        int c[4];
        float rec[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            c[e] = min(c0 + e * LPT, a.C - 1);
            rec[e] = 0.f;
        }
        int sl = 0;
        for (int l = 0; l < a.S; ++l) {
            const float g = a.gamma[l];
#pragma unroll 8
            for (int q = 0; q < a.k; ++q, ++sl) {
                const uint16_t v = cd[sl];
                const float scale = g * ((v & 0x8000) ? -1.0f : 1.0f);
                const float* d = a.D + (size_t)(v & 0x7FFF) * a.C;
#pragma unroll
                for (int e = 0; e < 4; ++e) rec[e] = fmaf(scale, d[c[e]], rec[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c0 + e * LPT < a.C) out[c0 + e * LPT] = x[c[e]] - rec[e];
    }
}

constexpr uint8_t kAtomKept = 0, kAtomNonFinite = 1, kAtomDead = 2;

__global__ __launch_bounds__(kEThreads) void atom_sum_kernel(FitArgs a) {
    constexpr int kU = 8;  // users' rows in flight
    const int j = blockIdx.x, c = blockIdx.y * kEThreads + threadIdx.x;
    const int u0 = a.off[j], u1 = a.off[j + 1];
    const double iw = a.inv_w[j];
    if (u0 == u1 || iw == 0.0 || c >= a.C) return;
    double corr = 0.0;
    int u = u0;
    for (; u + kU <= u1; u += kU) {
        float v[kU];
#pragma unroll
        for (int q = 0; q < kU; ++q) v[q] = a.res[(size_t)a.utile[u + q] * a.C + c];
#pragma unroll
        for (int q = 0; q < kU; ++q) corr = fma(a.ucoef[u + q], (double)v[q], corr);
    }
    for (; u < u1; ++u) corr = fma(a.ucoef[u], (double)a.res[(size_t)a.utile[u] * a.C + c], corr);
    // the new value through double; one that float cannot hold comes out infinite
    float& d = a.D[(size_t)j * a.C + c];
    d = (float)fma(corr, iw, (double)d);
}

__global__ __launch_bounds__(kEThreads) void atom_finish_kernel(FitArgs a) {
    extern __shared__ float nv[];  // C: the atom's new values
    __shared__ double nsq_s;
    const int j = blockIdx.x, tid = threadIdx.x, C = a.C;
    const bool dead = a.off[j] == a.off[j + 1];
    if (dead || a.inv_w[j] == 0.0) {  // no users, or sum of gamma^2 <= 1e-12: the atom stays
        if (tid == 0) a.flag[j] = dead ? kAtomDead : kAtomKept;
        return;
    }
    float* atom = a.D + (size_t)j * C;
    int bad = 0;
    for (int c = tid; c < C; c += kEThreads) {
        const float vf = atom[c];
        if (!isfinite(vf)) bad = 1;
        nv[c] = vf;
    }
    if (__syncthreads_or(bad)) {
        if (tid == 0) a.flag[j] = kAtomNonFinite;
        return;
    }
    if (tid == 0) {
        double sq = 0.0;
#pragma unroll 8
        for (int c = 0; c < C; ++c) sq = fma((double)nv[c], (double)nv[c], sq);
        nsq_s = sq;
        a.flag[j] = isfinite(sq) ? kAtomKept : kAtomNonFinite;
    }
    __syncthreads();
    const double nsq = nsq_s;
    if (!isfinite(nsq)) return;
    const double nn = sqrt(nsq);
    if (nn > a.cap) {
        const double sc = a.target / nn;
        for (int c = tid; c < C; c += kEThreads) atom[c] = (float)((double)nv[c] * sc);
    }
}

// ---------------------------------------------------------------- the initial dictionary

// hsdr_init.cpp's sums on the device, operation for operation (no contraction: its products and
// sums are rounded where that file rounds them; fma is one rounding on both). On the host
// the tile norms were a library call per element, 9 ms for 4864 x 896.
//  tile_norms_kernel: squared_norm_d of every tile, a lane per one of its four partial sums;
//  atom_norms_kernel: squared_norm of the picked tiles, a lane per one of its eight;
//  init_atoms_kernel: (tile * unit) * scale.
__global__ __launch_bounds__(kEThreads) void tile_norms_kernel(const float* __restrict__ tiles,
                                                               uint32_t n, uint32_t C,
                                                               double* __restrict__ out) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * (kEThreads / 4) + threadIdx.x / 4;
    const int j = threadIdx.x & 3;
    const float* t = tiles + (size_t)min(i, n - 1) * C;
    double a = 0.0;
    uint32_t c = 0;
#pragma unroll 4
    for (; c + 8 <= C; c += 8) {
        const double lo = t[c + j], hi = t[c + 4 + j];
        const double h2 = hi * hi;
        a = a + fma(lo, lo, h2);
    }
    const double a2 = a + __shfl_xor(a, 2, 4);        // lanes 0 + 2 and 1 + 3
    double total = a2 + __shfl_xor(a2, 1, 4);
    if (C - c >= 4) {
        const double t0 = t[c], t1 = t[c + 1], t2 = t[c + 2], t3 = t[c + 3];
        const double p2 = t2 * t2, p3 = t3 * t3;
        const double e0 = fma(t0, t0, p2), e1 = fma(t1, t1, p3);
        const double e = e0 + e1;
        total = total + e;
        c += 4;
    }
    for (; c < C; ++c) total = fma((double)t[c], (double)t[c], total);
    if (i < n && j == 0) out[i] = total;
}

__global__ __launch_bounds__(kEThreads) void atom_norms_kernel(const float* __restrict__ tiles,
                                                               const uint32_t* __restrict__ src,
                                                               uint32_t K, uint32_t C,
                                                               float* __restrict__ out) {
#pragma clang fp contract(off)
    const uint32_t a = blockIdx.x * (kEThreads / 8) + threadIdx.x / 8;
    const int l = threadIdx.x & 7;
    const float* d = tiles + (size_t)src[min(a, K - 1)] * C;
    float v = 0.f;
    uint32_t c = 0;
#pragma unroll 4
    for (; c + 8 <= C; c += 8) v = fmaf(d[c + l], d[c + l], v);
    const float h = v + __shfl_xor(v, 4, 8);   // h[i] = v[i + 4] + v[i]
    const float s = h + __shfl_xor(h, 2, 8);   // h[2] + h[0], h[3] + h[1]
    float sq = s + __shfl_xor(s, 1, 8);
    if (c + 4 <= C) {
        float p[4];
        for (int i = 0; i < 4; ++i) p[i] = d[c + i] * d[c + i];
        const float b0 = p[2] + p[0], b1 = p[3] + p[1];
        const float b = b1 + b0;
        sq = sq + b;
        c += 4;
    }
    for (; c < C; ++c) sq = fmaf(d[c], d[c], sq);
    if (a < K && l == 0) out[a] = sq;
}

__global__ __launch_bounds__(kEThreads) void init_atoms_kernel(const float* __restrict__ tiles,
                                                               const uint32_t* __restrict__ src,
                                                               const float* __restrict__ unit,
                                                               float scale, uint32_t C,
                                                               float* __restrict__ D) {
    const uint32_t j = blockIdx.x;
    const float* t = tiles + (size_t)src[j] * C;
    const float u = unit[j];
    for (uint32_t c = threadIdx.x; c < C; c += kEThreads) {
        const float d = t[c] * u;
        D[(size_t)j * C + c] = d * scale;
    }
}

// ---------------------------------------------------------------- compress (host side)

struct Geometry {
    uint32_t R, C, tr, tc, R_full, C_full, n_tiles, tile_dim, edge_floats;
    uint16_t K;
    uint8_t S, k;
};

// The strategy's geometry (compress :1130-1160; configFor :1024-1046 widens 1-row tiles to
// the whole row).
int geometry(uint32_t R, uint32_t C, uint16_t tile_rows, uint16_t tile_cols, uint16_t K,
             uint8_t S, uint8_t k, Geometry* g) {
    if (R == 0 || C == 0 || tile_rows == 0 || tile_cols == 0 || K == 0 || S == 0 || k == 0)
        return set_error(CSDR_E_INVALID, "hsdr_compress: bad shape or config");
    g->R = R;
    g->C = C;
    g->tr = tile_rows;
    g->tc = (tile_rows == 1 && C <= 0xFFFFu) ? C : tile_cols;
    g->R_full = R / g->tr * g->tr;
    g->C_full = C / g->tc * g->tc;
    if (g->R_full == 0 || g->C_full == 0)
        return set_error(CSDR_E_FORMAT, "HSDR: tensor too small to hold even one full tile");
    g->n_tiles = (g->R_full / g->tr) * (g->C_full / g->tc);
    g->tile_dim = g->tr * g->tc;
    if (g->n_tiles < K)
        return set_error(CSDR_E_FORMAT,
                         "HSDR: not enough tiles to fit the requested dictionary size");
    g->edge_floats = g->R_full * (C - g->C_full) + (R - g->R_full) * C;
    g->K = K;
    g->S = S;
    g->k = k;
    return CSDR_OK;
}

size_t stream_bytes(const Geometry& g) {
    return 36 + (size_t)g.S * 4 + (size_t)g.K * g.tile_dim * 4 +
           (size_t)g.n_tiles * g.S * g.k * 2 + (size_t)g.edge_floats * 4;
}

// A device allocation freed with its scope.
struct DevBuf {
    void* p = nullptr;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
    float* f() const { return static_cast<float*>(p); }
    uint16_t* u16() const { return static_cast<uint16_t*>(p); }
};

// The buffers of one fit or encode. The Gram path's workspace is asked for first (its allocation
// and the others' run beside the work already on the device) and left empty, for mp_kernel and
// the same codes, where that path does not pay or the memory cannot be had; it is given up again
// where a buffer that the call cannot do without finds no room.
struct Scratch {
    DevBuf gram;
    hipStream_t st;

    Scratch(long long n, int C, int K, int S, int k, hipStream_t stream) : st(stream) {
        if (gram_pays(n, C, K, S, k) && hipMalloc(&gram.p, gram_ws_bytes(n, K)) != hipSuccess) {
            gram.p = nullptr;
            (void)hipGetLastError();
        }
    }

    int need(DevBuf& b, size_t bytes) {
        hipError_t e = hipMalloc(&b.p, bytes);
        if (e != hipSuccess && gram.p) {
            (void)hipGetLastError();
            (void)hipStreamSynchronize(st);  // an encode may still be reading it
            (void)hipFree(gram.p);
            gram.p = nullptr;
            e = hipMalloc(&b.p, bytes);
        }
        if (e == hipSuccess) return CSDR_OK;
        b.p = nullptr;
        (void)hipGetLastError();
        return set_error(CSDR_E_HIP, "hsdr_compress: out of device memory (" +
                                         std::to_string(bytes) + " bytes)");
    }
};

#define RC(expr)                        \
    do {                                \
        const int rc_ = (expr);         \
        if (rc_ != CSDR_OK) return rc_; \
    } while (0)

// One atomUpdateStep per pass (HierarchicalSDRStrategy.cpp:281-490): users, residuals and
// updates on the device, the re-seeds on the host from the fit's generator (base seed :403).
struct Refine {
    DevBuf res, off, utile, ucoef, invw, flag;
    FitArgs fa{};

    int init(const Geometry& g, double mean_norm, const std::vector<float>& gamma,
             const float* d_tiles, float* d_D, const uint16_t* d_codes, Scratch& scratch) {
        const size_t slots = (size_t)g.S * g.k, ncodes = (size_t)g.n_tiles * slots;
        RC(scratch.need(res, (size_t)g.n_tiles * g.tile_dim * 4));
        RC(scratch.need(off, ((size_t)g.K + 1) * 4));
        RC(scratch.need(utile, std::max<size_t>(ncodes, 1) * 4));
        RC(scratch.need(ucoef, std::max<size_t>(ncodes, 1) * 8));
        RC(scratch.need(invw, (size_t)g.K * 8));
        RC(scratch.need(flag, (size_t)g.K));
        fa.tiles = d_tiles;
        fa.codes = d_codes;
        fa.D = d_D;
        fa.res = res.f();
        fa.off = static_cast<int*>(off.p);
        fa.utile = static_cast<uint32_t*>(utile.p);
        fa.ucoef = static_cast<double*>(ucoef.p);
        fa.inv_w = static_cast<double*>(invw.p);
        fa.flag = static_cast<uint8_t*>(flag.p);
        fa.n = g.n_tiles;
        fa.ncodes = (long long)ncodes;
        fa.C = (int)g.tile_dim;
        fa.K = g.K;
        fa.S = g.S;
        fa.k = g.k;
        fa.target = std::max(1e-6, mean_norm / std::sqrt((double)slots));  // :390-392
        fa.cap = 1.5 * fa.target;
        for (uint32_t l = 0; l < g.S; ++l) fa.gamma[l] = gamma[l];
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&atom_finish_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)(g.tile_dim * 4));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&users_count_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)g.K * 4);
        return CSDR_OK;
    }

    int pass(const float* tiles, std::mt19937& rng, hipStream_t st) {
        const uint32_t C = (uint32_t)fa.C, K = (uint32_t)fa.K;
        const uint64_t base_seed = static_cast<uint64_t>(rng()) ^ 0xA0B1C2D3u;
        users_zero_kernel<<<(K + kEThreads) / kEThreads, kEThreads, 0, st>>>(fa);
        const unsigned cgrid =
            (unsigned)std::min<long long>((fa.ncodes + 4 * kEThreads - 1) / (4 * kEThreads), 256);
        users_count_kernel<<<cgrid, kEThreads, K * 4, st>>>(fa);
        users_scan_kernel<<<1, kEThreads, 0, st>>>(fa);
        users_fill_kernel<<<K, kEThreads, 0, st>>>(fa);
        CSDR_LAUNCH_CHECK("hsdr_compress users");
        const auto residual = [&](auto kern, int lpt) {
            const long long per = kEThreads / lpt;
            kern<<<(unsigned)((fa.n + per - 1) / per), kEThreads, 0, st>>>(fa);
        };
        if (C <= 64) residual(&residual_kernel<16>, 16);
        else if (C <= 256) residual(&residual_kernel<64>, 64);
        else residual(&residual_kernel<kEThreads>, kEThreads);
        CSDR_LAUNCH_CHECK("hsdr_compress residual");
        atom_sum_kernel<<<dim3(K, (C + kEThreads - 1) / kEThreads), kEThreads, 0, st>>>(fa);
        atom_finish_kernel<<<K, kEThreads, (size_t)C * 4, st>>>(fa);
        CSDR_LAUNCH_CHECK("hsdr_compress atom update");
        std::vector<uint8_t> fl(K);
        CSDR_HIP_CHECK(hipMemcpyAsync(fl.data(), flag.p, K, hipMemcpyDeviceToHost, st));
        CSDR_HIP_CHECK(hipStreamSynchronize(st));
        std::vector<float> atom(C);
        for (uint32_t j = 0; j < K; ++j) {
            if (fl[j] == kAtomKept) continue;
            csdr::hsdr_reseed_atom(tiles, (uint32_t)fa.n, C, base_seed, j,
                                   fl[j] == kAtomDead ? 0x9E3779B1u : 0xB7E15163u, fa.target,
                                   atom.data());
            CSDR_HIP_CHECK(hipMemcpy(fa.D + (size_t)j * C, atom.data(), (size_t)C * 4,
                                     hipMemcpyHostToDevice));
        }
        return CSDR_OK;
    }
};

template <class T>
void put(std::vector<uint8_t>& out, const T& v) {
    const uint8_t* p = reinterpret_cast<const uint8_t*>(&v);
    out.insert(out.end(), p, p + sizeof(T));
}

// The initial dictionary of device tiles into d_D; returns the tiles' mean norm in *mean_norm
// (the square roots summed in tile order, as hsdr_init.cpp does).
int init_dictionary_device(const float* d_tiles, uint32_t n, uint32_t C, uint16_t K,
                           uint32_t slots, std::mt19937& rng, float* d_D, double* mean_norm,
                           Scratch& scratch, hipStream_t st) {
    DevBuf ws;  // n squared norms, then K picks, K squared norms, K factors
    RC(scratch.need(ws, (size_t)n * 8 + (size_t)K * 12));
    double* d_norm = static_cast<double*>(ws.p);
    uint32_t* d_src = reinterpret_cast<uint32_t*>(d_norm + n);
    float* d_sq = reinterpret_cast<float*>(d_src + K);
    float* d_unit = d_sq + K;
    std::vector<uint32_t> src(K);
    csdr::hsdr_init_picks(n, K, rng, src.data());
    CSDR_HIP_CHECK(hipMemcpyAsync(d_src, src.data(), (size_t)K * 4, hipMemcpyHostToDevice, st));
    tile_norms_kernel<<<(n + kEThreads / 4 - 1) / (kEThreads / 4), kEThreads, 0, st>>>(
        d_tiles, n, C, d_norm);
    atom_norms_kernel<<<(K + kEThreads / 8 - 1) / (kEThreads / 8), kEThreads, 0, st>>>(
        d_tiles, d_src, K, C, d_sq);
    CSDR_LAUNCH_CHECK("hsdr_compress norms");
    std::vector<double> norm(n);
    std::vector<float> sq(K), unit(K);
    CSDR_HIP_CHECK(hipMemcpyAsync(norm.data(), d_norm, (size_t)n * 8, hipMemcpyDeviceToHost, st));
    CSDR_HIP_CHECK(hipMemcpyAsync(sq.data(), d_sq, (size_t)K * 4, hipMemcpyDeviceToHost, st));
    CSDR_HIP_CHECK(hipStreamSynchronize(st));
    double sum = 0.0;
    for (double v : norm) sum += std::sqrt(v);
    *mean_norm = sum / (double)std::max<uint32_t>(1u, n);
    const float scale = csdr::hsdr_init_scales(sq.data(), K, slots, *mean_norm, unit.data());
    CSDR_HIP_CHECK(hipMemcpyAsync(d_unit, unit.data(), (size_t)K * 4, hipMemcpyHostToDevice, st));
    init_atoms_kernel<<<K, kEThreads, 0, st>>>(d_tiles, d_src, d_unit, scale, C, d_D);
    CSDR_LAUNCH_CHECK("hsdr_compress atoms");
    CSDR_HIP_CHECK(hipStreamSynchronize(st));  // the factors and the workspace are this frame's
    return CSDR_OK;
}

// fitHierarchicalKSVD (HierarchicalSDRStrategy.cpp:494-607) over tiles (n x tile_dim) in host
// memory: the dictionary initialisation from the fit's generator (mt19937(0xC0DE), :513),
// matching pursuit, then ksvd_iters atom-update passes each followed by matching pursuit again
// (:570-573); D (K x tile_dim, non-finite values zeroed as :592-601) and, when codes is not
// null, the final codes.
int fit_tiles(const float* tiles, uint32_t n_tiles, uint32_t tile_dim, uint16_t K,
              uint8_t S, uint8_t k, uint8_t ksvd_iters, const std::vector<float>& gamma,
              float* D, uint16_t* codes, hipStream_t st) {
    Geometry g{};
    g.n_tiles = n_tiles;
    g.tile_dim = tile_dim;
    g.K = K;
    g.S = S;
    g.k = k;
    if (ksvd_iters != 0 && tile_dim > 32768)
        return set_error(CSDR_E_UNSUPPORTED,
                         "hsdr_compress: K-SVD refinement takes tiles of at most 32768 values");
    int rc = check_mp_shape(n_tiles, (int)tile_dim, K, S, k);
    if (rc != CSDR_OK) return rc;
    const size_t ncodes = (size_t)n_tiles * S * k, kc = (size_t)K * tile_dim;
    Scratch scratch(n_tiles, (int)tile_dim, K, S, k, st);
    DevBuf d_tiles, d_D, d_codes;
    RC(scratch.need(d_tiles, (size_t)n_tiles * tile_dim * 4));
    RC(scratch.need(d_D, kc * 4));
    RC(scratch.need(d_codes, std::max<size_t>(ncodes * 2, 2)));
    CSDR_HIP_CHECK(hipMemcpyAsync(d_tiles.p, tiles, (size_t)n_tiles * tile_dim * 4,
                                  hipMemcpyHostToDevice, st));
    std::mt19937 rng(0xC0DE);  // the fit's generator (:513), through init and every pass
    double mean_norm = 0.0;
    RC(init_dictionary_device(d_tiles.f(), n_tiles, tile_dim, K, (uint32_t)S * k, rng, d_D.f(),
                              &mean_norm, scratch, st));
    const auto encode = [&] {
        return launch_mp(d_tiles.f(), n_tiles, (int)tile_dim, d_D.f(), K, S, k, gamma.data(),
                         d_codes.u16(), scratch.gram.p, st);
    };
    RC(encode());
    if (ksvd_iters) {
        Refine rf;
        RC(rf.init(g, mean_norm, gamma, d_tiles.f(), d_D.f(), d_codes.u16(), scratch));
        for (int it = 0; it < ksvd_iters; ++it) {  // atom update, then encode again (:570-573)
            RC(rf.pass(tiles, rng, st));
            RC(encode());
        }
    }
    CSDR_HIP_CHECK(hipMemcpyAsync(D, d_D.p, kc * 4, hipMemcpyDeviceToHost, st));
    if (codes)
        CSDR_HIP_CHECK(hipMemcpyAsync(codes, d_codes.p, ncodes * 2, hipMemcpyDeviceToHost, st));
    CSDR_HIP_CHECK(hipStreamSynchronize(st));
    for (size_t i = 0; i < kc; ++i)  // the fit's final sanitisation (:592-601)
        if (!std::isfinite(D[i])) D[i] = 0.0f;
    return CSDR_OK;
}

// Matching pursuit of host tiles against a fixed dictionary (encodeAllTilesAgainstDictionary,
// the encode of compressFP32WithExternalDictionary :1690-1754).
int encode_tiles(const float* tiles, uint32_t n_tiles, uint32_t tile_dim, const std::vector<float>& D,
                 uint16_t K, uint8_t S, uint8_t k, const std::vector<float>& gamma,
                 std::vector<uint16_t>& codes, hipStream_t st) {
    int rc = check_mp_shape(n_tiles, (int)tile_dim, K, S, k);
    if (rc != CSDR_OK) return rc;
    const size_t ncodes = (size_t)n_tiles * S * k;
    Scratch scratch(n_tiles, (int)tile_dim, K, S, k, st);
    DevBuf d_tiles, d_D, d_codes;
    RC(scratch.need(d_tiles, std::max<size_t>((size_t)n_tiles * tile_dim, 1) * 4));
    RC(scratch.need(d_D, D.size() * 4));
    RC(scratch.need(d_codes, std::max<size_t>(ncodes * 2, 2)));
    CSDR_HIP_CHECK(hipMemcpyAsync(d_tiles.p, tiles, (size_t)n_tiles * tile_dim * 4,
                                  hipMemcpyHostToDevice, st));
    CSDR_HIP_CHECK(hipMemcpyAsync(d_D.p, D.data(), D.size() * 4, hipMemcpyHostToDevice, st));
    rc = launch_mp(d_tiles.f(), n_tiles, (int)tile_dim, d_D.f(), K, S, k, gamma.data(),
                   d_codes.u16(), scratch.gram.p, st);
    if (rc != CSDR_OK) return rc;
    codes.resize(ncodes);
    CSDR_HIP_CHECK(hipMemcpyAsync(codes.data(), d_codes.p, ncodes * 2, hipMemcpyDeviceToHost, st));
    CSDR_HIP_CHECK(hipStreamSynchronize(st));
    return CSDR_OK;
}

// Tiles of an R x C matrix in row-major tile order (extractTiles :94-116), of its aligned
// top-left block.
std::vector<float> extract_tiles(const float* w, uint32_t R, uint32_t C, uint32_t tr,
                                 uint32_t tc) {
    const uint32_t nrt = R / tr, nct = C / tc;
    std::vector<float> tiles((size_t)nrt * nct * tr * tc);
    for (uint32_t br = 0; br < nrt; ++br)
        for (uint32_t bc = 0; bc < nct; ++bc) {
            float* dst = tiles.data() + (size_t)(br * nct + bc) * tr * tc;
            for (uint32_t r = 0; r < tr; ++r)
                std::memcpy(dst + (size_t)r * tc, w + (size_t)(br * tr + r) * C + (size_t)bc * tc,
                            sizeof(float) * tc);
        }
    return tiles;
}

// compressGroupedSegments' bucket key and its hash (HierarchicalSDRStrategy.cpp:2088-2120),
// so that the buckets come out of the same std::unordered_map in the same order.
struct GroupKey {
    uint16_t tile_rows, tile_cols, n_atoms;
    uint8_t n_stages, k;
    float decay;
    bool operator==(const GroupKey& o) const {
        return tile_rows == o.tile_rows && tile_cols == o.tile_cols && n_atoms == o.n_atoms &&
               n_stages == o.n_stages && k == o.k && decay == o.decay;
    }
};
struct GroupKeyHash {
    size_t operator()(const GroupKey& g) const {
        size_t h = std::hash<uint32_t>{}(((uint32_t)g.tile_rows << 16) | g.tile_cols);
        h ^= std::hash<uint32_t>{}(((uint32_t)g.n_atoms << 16) | ((uint32_t)g.n_stages << 8) | g.k) +
             0x9e3779b9 + (h << 6) + (h >> 2);
        h ^= std::hash<float>{}(g.decay) + 0x9e3779b9 + (h << 6) + (h >> 2);
        return h;
    }
};

}  // namespace

extern "C" {

CSDR_API int csdr_hsdr_encode(const float* tiles, size_t n_tiles, int tile_dim, const float* D,
                              int n_atoms, int n_stages, int k_per_stage,
                              const float* stage_scales, uint16_t* codes, void* hip_stream) {
    if ((n_tiles && (!tiles || !codes)) || !D || !stage_scales)
        return set_error(CSDR_E_INVALID, "hsdr_encode: null pointer");
    const int rc = check_mp_shape((long long)n_tiles, tile_dim, n_atoms, n_stages, k_per_stage);
    if (rc != CSDR_OK) return rc;
    // The Gram path's workspace is stream-ordered memory; a stream under capture (or one whose
    // state cannot be asked for) and an allocation that fails keep mp_kernel, which needs none.
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    void* ws = nullptr;
    if (n_tiles && gram_pays((long long)n_tiles, tile_dim, n_atoms, n_stages, k_per_stage)) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusActive;
        if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone ||
            hipMallocAsync(&ws, gram_ws_bytes((long long)n_tiles, n_atoms), st) != hipSuccess) {
            ws = nullptr;
            (void)hipGetLastError();
        }
    }
    const int mrc = launch_mp(tiles, (long long)n_tiles, tile_dim, D, n_atoms, n_stages,
                              k_per_stage, stage_scales, codes, ws, st);
    if (ws) (void)hipFreeAsync(ws, st);
    return mrc;
}

CSDR_API int csdr_hsdr_init_dictionary(const float* tiles, uint32_t n_tiles, uint32_t tile_dim,
                                       uint16_t n_atoms, uint8_t n_stages, uint8_t k_per_stage,
                                       float* D) {
    if (!tiles || !D || n_tiles == 0 || tile_dim == 0 || n_atoms == 0 || n_stages == 0 ||
        k_per_stage == 0)
        return set_error(CSDR_E_INVALID, "hsdr_init_dictionary: bad argument");
    csdr::hsdr_init_dictionary(tiles, n_tiles, tile_dim, n_atoms,
                               (uint32_t)n_stages * k_per_stage, D);
    return CSDR_OK;
}

CSDR_API size_t csdr_hsdr_compress_bytes(uint32_t rows, uint32_t cols, uint16_t tile_rows,
                                         uint16_t tile_cols, uint16_t n_atoms, uint8_t n_stages,
                                         uint8_t k_per_stage) {
    Geometry g;
    if (geometry(rows, cols, tile_rows, tile_cols, n_atoms, n_stages, k_per_stage, &g) !=
        CSDR_OK)
        return 0;
    return stream_bytes(g);
}

CSDR_API int csdr_hsdr_compress(const float* w, uint32_t rows, uint32_t cols, uint16_t tile_rows,
                                uint16_t tile_cols, uint16_t n_atoms, uint8_t n_stages,
                                uint8_t k_per_stage, uint8_t ksvd_iters, float stage_decay,
                                uint8_t* out, size_t out_bytes, void* hip_stream) {
    if (!w || !out) return set_error(CSDR_E_INVALID, "hsdr_compress: null pointer");
    Geometry g;
    int rc = geometry(rows, cols, tile_rows, tile_cols, n_atoms, n_stages, k_per_stage, &g);
    if (rc != CSDR_OK) return rc;
    if (out_bytes < stream_bytes(g))
        return set_error(CSDR_E_INVALID, "hsdr_compress: output buffer too small");
    if (ksvd_iters != 0 && g.tile_dim > 32768)
        return set_error(CSDR_E_UNSUPPORTED,
                         "hsdr_compress: K-SVD refinement takes tiles of at most 32768 values");
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    // tiles in row-major tile order (extractTiles :94-116) of the aligned block; whole-row
    // tiles lie in that order already
    std::vector<float> copied;
    if (!(g.tr == 1 && g.tc == g.C)) copied = extract_tiles(w, g.R_full, g.C, g.tr, g.tc);
    const float* tiles = copied.empty() ? w : copied.data();
    std::vector<float> gamma(g.S), D((size_t)g.K * g.tile_dim);
    for (uint32_t l = 0; l < g.S; ++l) gamma[l] = std::pow(stage_decay, (float)l);
    std::vector<uint16_t> codes((size_t)g.n_tiles * g.S * g.k);
    rc = fit_tiles(tiles, g.n_tiles, g.tile_dim, g.K, g.S, g.k, ksvd_iters, gamma, D.data(),
                   codes.data(), st);
    if (rc != CSDR_OK) return rc;

    // serialisation (:1197-1237): header, stage scales, D, packed codes, edge strips
    uint8_t* o = out;
    const auto bytes = [&](const void* p, size_t n) {
        if (n) std::memcpy(o, p, n);
        o += n;
    };
    std::vector<uint8_t> s{'H', 'S', 'D', 'R'};
    put<uint32_t>(s, 2);
    put<uint32_t>(s, g.R);
    put<uint32_t>(s, g.C);
    put<uint32_t>(s, g.n_tiles);
    put<uint16_t>(s, (uint16_t)g.tr);
    put<uint16_t>(s, (uint16_t)g.tc);
    put<uint16_t>(s, g.K);
    put<uint8_t>(s, g.S);
    put<uint8_t>(s, g.k);
    put<float>(s, stage_decay);
    put<uint32_t>(s, g.edge_floats * 4);
    bytes(s.data(), s.size());
    bytes(gamma.data(), gamma.size() * 4);
    bytes(D.data(), D.size() * 4);
    bytes(codes.data(), codes.size() * 2);
    for (uint32_t r = 0; r < g.R_full; ++r)
        bytes(w + (size_t)r * g.C + g.C_full, (size_t)(g.C - g.C_full) * 4);
    bytes(w + (size_t)g.R_full * g.C, (size_t)(g.R - g.R_full) * g.C * 4);
    return CSDR_OK;
}

CSDR_API int csdr_hsda_build(int n, const char* const* names, const float* const* w,
                             const uint32_t* rows, const uint32_t* cols,
                             const uint8_t* original_types, uint16_t tile_rows,
                             uint16_t tile_cols, uint16_t n_atoms, uint8_t n_stages,
                             uint8_t k_per_stage, uint8_t ksvd_iters, float stage_decay,
                             uint32_t max_tiles_for_fit, uint8_t** out, size_t* out_size,
                             uint8_t* skipped, void* hip_stream) {
    if (n <= 0 || !names || !w || !rows || !cols || !out || !out_size)
        return set_error(CSDR_E_INVALID, "hsda_build: bad argument");
    if (tile_rows == 0 || tile_cols == 0 || n_atoms == 0 || n_stages == 0 || k_per_stage == 0)
        return set_error(CSDR_E_INVALID, "hsda_build: bad config");
    *out = nullptr;
    *out_size = 0;
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    try {
        // configFor per segment (1-row tiles widen to the row), suitability (:2147-2190:
        // shape divisible by the tile; the caller's matrices are fp32), buckets by config
        std::vector<GroupKey> keys(n);
        std::unordered_map<GroupKey, std::vector<size_t>, GroupKeyHash> buckets;
        std::vector<uint8_t> skip(n, 0);
        for (int i = 0; i < n; ++i) {
            if (!names[i] || !w[i]) return set_error(CSDR_E_INVALID, "hsda_build: null entry");
            GroupKey key{tile_rows, (tile_rows == 1 && cols[i] <= 0xFFFFu) ? (uint16_t)cols[i]
                                                                          : tile_cols,
                         n_atoms, n_stages, k_per_stage, stage_decay};
            keys[i] = key;
            if (rows[i] == 0 || cols[i] == 0 || rows[i] % key.tile_rows ||
                cols[i] % key.tile_cols) {
                skip[i] = 1;
                continue;
            }
            buckets[key].push_back((size_t)i);
        }
        std::vector<float> gamma(n_stages);
        for (uint32_t l = 0; l < n_stages; ++l) gamma[l] = std::pow(stage_decay, (float)l);
        struct Dict {
            GroupKey key;
            std::vector<float> atoms;
        };
        struct Entry {
            size_t seg, dict;
            std::vector<uint16_t> codes;
            uint32_t n_tiles;
        };
        std::vector<Dict> dicts;
        std::vector<Entry> entries;
        for (auto& kv : buckets) {
            const GroupKey& key = kv.first;
            const uint32_t tr = key.tile_rows, tc = key.tile_cols, tile_dim = tr * tc;
            uint64_t total = 0;
            for (size_t i : kv.second) total += (uint64_t)(rows[i] / tr) * (cols[i] / tc);
            const uint32_t pooled_count = total > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)total;
            const uint32_t cap = (max_tiles_for_fit > 0 && total > max_tiles_for_fit)
                                     ? max_tiles_for_fit
                                     : pooled_count;
            const bool reservoir = cap < pooled_count;
            std::vector<float> pool((size_t)cap * tile_dim);
            std::mt19937 res_rng(0xC0DECAFEu ^ cap);  // :2277
            uint64_t seen = 0;
            uint32_t fill = 0;
            std::vector<size_t> pooled_segs;
            std::vector<std::vector<float>> seg_tiles;
            for (size_t i : kv.second) {
                // per-segment non-finite gate (:2324-2358): probe 1 in 256, then sanitise and
                // skip the segment when more than 1e-3 of it is bad. The sanitised values are
                // also what the segment is encoded from, in every tile mode; the reference
                // re-encodes 2-D segments from the raw values (:2373, :2474-2475), letting
                // NaN / Inf into matching pursuit (a deliberate difference)
                std::vector<float> m(w[i], w[i] + (size_t)rows[i] * cols[i]);
                bool any_bad = false;
                for (size_t j = 0; j < m.size(); j += 256)
                    if (!std::isfinite(m[j])) {
                        any_bad = true;
                        break;
                    }
                if (any_bad) {
                    size_t bad = 0;
                    for (float& v : m)
                        if (!std::isfinite(v)) {
                            v = 0.0f;
                            ++bad;
                        }
                    if ((double)bad / std::max<size_t>(1, m.size()) > 1e-3) {
                        skip[i] = 1;
                        continue;
                    }
                }
                std::vector<float> t = (tr == 1 && tc == cols[i])
                                           ? std::move(m)
                                           : extract_tiles(m.data(), rows[i], cols[i], tr, tc);
                const uint32_t nt = (rows[i] / tr) * (cols[i] / tc);
                for (uint32_t j = 0; j < nt; ++j) {
                    const float* src = t.data() + (size_t)j * tile_dim;
                    if (!reservoir || fill < cap) {
                        std::memcpy(pool.data() + (size_t)fill * tile_dim, src, tile_dim * 4);
                        ++fill;
                    } else {
                        std::uniform_int_distribution<uint64_t> dist(0, seen);
                        const uint64_t r = dist(res_rng);
                        if (r < cap) std::memcpy(pool.data() + r * tile_dim, src, tile_dim * 4);
                    }
                    ++seen;
                }
                pooled_segs.push_back(i);
                seg_tiles.push_back(std::move(t));
            }
            pool.resize((size_t)fill * tile_dim);
            for (float& v : pool)  // pool integrity (:2403-2419)
                if (!std::isfinite(v)) v = 0.0f;
            if (fill < key.n_atoms) {  // too small to fit the dictionary: the bucket is skipped
                for (size_t i : pooled_segs) skip[i] = 1;
                continue;
            }
            Dict d;
            d.key = key;
            d.atoms.resize((size_t)key.n_atoms * tile_dim);
            int rc = fit_tiles(pool.data(), fill, tile_dim, key.n_atoms, key.n_stages, key.k,
                               ksvd_iters, gamma, d.atoms.data(), nullptr, st);
            if (rc != CSDR_OK) return rc;
            const size_t di = dicts.size();
            dicts.push_back(std::move(d));
            for (size_t q = 0; q < pooled_segs.size(); ++q) {
                const size_t i = pooled_segs[q];
                Entry e;
                e.seg = i;
                e.dict = di;
                e.n_tiles = (rows[i] / tr) * (cols[i] / tc);
                rc = encode_tiles(seg_tiles[q].data(), e.n_tiles, tile_dim, dicts[di].atoms,
                                  key.n_atoms, key.n_stages, key.k, gamma, e.codes, st);
                if (rc != CSDR_OK) return rc;
                std::vector<float>().swap(seg_tiles[q]);
                entries.push_back(std::move(e));
            }
        }
        // SharedDictArchive::writeToStream (:1967-2002)
        std::vector<uint8_t> s;
        s.insert(s.end(), {'H', 'S', 'D', 'A'});
        put<uint32_t>(s, 1);
        put<uint32_t>(s, (uint32_t)dicts.size());
        put<uint32_t>(s, (uint32_t)entries.size());
        for (const Dict& d : dicts) {
            // the 20-byte HierarchicalSDRConfig (HierarchicalSDRStrategy.hpp:43-58); its two
            // padding bytes (10-11) written as zeros
            put<uint16_t>(s, d.key.tile_rows);
            put<uint16_t>(s, d.key.tile_cols);
            put<uint16_t>(s, d.key.n_atoms);
            put<uint8_t>(s, d.key.n_stages);
            put<uint8_t>(s, d.key.k);
            put<uint8_t>(s, ksvd_iters);
            put<uint8_t>(s, 0);  // reserved_pad
            put<uint16_t>(s, 0);
            put<float>(s, d.key.decay);
            put<uint32_t>(s, max_tiles_for_fit);
            put<uint32_t>(s, (uint32_t)gamma.size());
            for (float x : gamma) put<float>(s, x);
            put<uint32_t>(s, (uint32_t)d.atoms.size());
            for (float x : d.atoms) put<float>(s, x);
        }
        for (const Entry& e : entries) {
            const size_t i = e.seg;
            const std::string name = names[i];
            const GroupKey& key = dicts[e.dict].key;
            put<uint32_t>(s, (uint32_t)name.size());
            s.insert(s.end(), name.begin(), name.end());
            put<uint32_t>(s, (uint32_t)e.dict);
            put<uint64_t>(s, (uint64_t)rows[i] * cols[i] * 4);
            put<uint8_t>(s, original_types ? original_types[i] : (uint8_t)1);
            // compressFP32WithExternalDictionary's HSDC stream (:1732-1754): 32-byte header,
            // packed codes
            put<uint32_t>(s, (uint32_t)(32 + e.codes.size() * 2));
            s.insert(s.end(), {'H', 'S', 'D', 'C'});
            put<uint32_t>(s, 1);
            put<uint32_t>(s, rows[i]);
            put<uint32_t>(s, cols[i]);
            put<uint32_t>(s, e.n_tiles);
            put<uint16_t>(s, key.tile_rows);
            put<uint16_t>(s, key.tile_cols);
            put<uint16_t>(s, key.n_atoms);
            put<uint8_t>(s, key.n_stages);
            put<uint8_t>(s, key.k);
            put<float>(s, key.decay);
            for (uint16_t c : e.codes) put<uint16_t>(s, c);
        }
        uint8_t* buf = static_cast<uint8_t*>(std::malloc(std::max<size_t>(s.size(), 1)));
        if (!buf) return set_error(CSDR_E_INVALID, "hsda_build: out of host memory");
        std::memcpy(buf, s.data(), s.size());
        *out = buf;
        *out_size = s.size();
        if (skipped) std::memcpy(skipped, skip.data(), skip.size());
    } catch (const std::exception& ex) {
        return set_error(CSDR_E_INVALID, std::string("hsda_build: ") + ex.what());
    }
    return CSDR_OK;
}

CSDR_API void csdr_free_buffer(void* p) { std::free(p); }

}  // extern "C"
