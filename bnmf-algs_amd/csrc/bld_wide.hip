// bld_wide.hip — pass kernel for instances whose fibers are deeper than the
// fused passes hold in registers (z > 64). The reference puts no bound on z
// (check_bld_params, src/bld/util_details.hpp:20-28; its kernels loop over
// any z, cuda_src/bld_mult/bld_mult_cuda_kernels.cu:119-255).
//
// Mapping: one wavefront per block; a work item is a tile of kWideRows rows
// x kWideCols columns of one instance, walked row by row. For each fiber
// (i, j) the 64 lanes cover k = lane, lane + 64, ... (a fiber of z > 64
// elements is at least 260 contiguous bytes, so every access is coalesced)
// and the per-fiber sums (S_ij+, nom, denom; S_mult and the exp-row norm of
// the additive step) are butterfly reductions across the wave, which leave
// the same value in every lane (each step adds a commutative pair). Phase B
// re-reads the fiber (it was just read: cache hits) and evaluates the
// element's gradient again rather than keeping z values per lane, so one
// kernel serves every z with no register arrays and no LDS. Up to z = 256 the
// sums and step passes run bld_wide_regs_kernel instead (below).
//
// The tile owns its partial-sum slots: part_pjk[ti][j][k] for its columns
// (summed over its rows, in row order) and part_ipk[tj][i][k] for its rows
// (summed over its columns, in column order); each slot is written by the
// lane that owns k, first by a store, then by read-add-store, so results are
// deterministic and independent of the rest of the launch. The prep kernel
// reduces them as it reduces the fused passes' partials.
//
// Reference operations: update_grad_plus bld_mult_funcs.hpp:177-192, nom
// :242-259, denom :272-290, update_S :307-327; bld_add's step
// src/bld/bld_add.hpp:137-181; the log-marginal's lgamma(S+1) terms
// alloc_model_funcs.hpp:179-194.

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "bld_types.hpp"
#include "digamma.hpp"
#include "pass_common.hpp"

namespace bnmf {

template <typename T, typename ACC, int MODE, int PSI>
__global__ void __launch_bounds__(64)
    bld_wide_kernel(const BldInst* __restrict__ insts, const PassItem* __restrict__ items,
                    const uint32_t* __restrict__ n_items_p) {
    const uint32_t n_items = *n_items_p;
    const uint32_t lane = threadIdx.x;
    for (uint32_t it = blockIdx.x; it < n_items; it += gridDim.x) {
        const PassItem item = items[it];
        const BldInst* __restrict__ I = insts + item.inst;
        const uint32_t x = I->x, y = I->y, z = I->z;
        const uint32_t i0 = item.ti * kWideRows, i1 = min(x, i0 + kWideRows);
        const uint32_t j0 = item.tj * kWideCols, j1 = min(y, j0 + kWideCols);
        // S_src and S are the same tensor after the first pass: no restrict
        const BNMF_GLOBAL T* Ssrc = gconst<T>(I->S_src);
        BNMF_GLOBAL T* Sdst = gmut<T>(I->S);
        BNMF_GLOBAL ACC* __restrict__ pjk = gmut<ACC>(I->part_pjk) + (size_t)item.ti * y * z;
        BNMF_GLOBAL ACC* __restrict__ ipk = gmut<ACC>(I->part_ipk) + (size_t)item.tj * x * z;
        const double eps = I->eps;
        const bool fast_psi = I->nonneg != 0u;
        double eta = 0.0;
        // additive step size 0.1 / (iteration + 1)^0.55 (bld_add.hpp:101-103);
        // *iter counts the iterations started, this one included
        if constexpr (MODE == PASS_ADD) eta = 0.1 / pow((double)*I->iter, 0.55);
        double lg_sum = 0.0;

        for (uint32_t i = i0; i < i1; ++i) {
            const BNMF_GLOBAL T* __restrict__ psia_i = gconst<T>(I->psia) + (size_t)i * z;
            const BNMF_GLOBAL T* __restrict__ psiA = gconst<T>(I->psiA);
            for (uint32_t j = j0; j < j1; ++j) {
                const size_t f = ((size_t)i * y + j) * z;
                const BNMF_GLOBAL T* src = Ssrc + f;
                BNMF_GLOBAL T* dst = Sdst + f;
                const BNMF_GLOBAL T* __restrict__ pb = gconst<T>(I->psib) + (size_t)j * z;
                const bool row0 = i == i0, col0 = j == j0;
                // the new element's contribution to the tile's partial sums
                auto add_partials = [&](uint32_t k, T sn) {
                    const size_t a = (size_t)j * z + k, b = (size_t)i * z + k;
                    pjk[a] = row0 ? ACC(sn) : pjk[a] + ACC(sn);
                    ipk[b] = col0 ? ACC(sn) : ipk[b] + ACC(sn);
                };
                if constexpr (MODE == PASS_SUMS || MODE == PASS_SCORE) {
                    ACC fs = ACC(0);
                    for (uint32_t k = lane; k < z; k += 64) {
                        const T s = src[k];
                        add_partials(k, s);
                        fs += ACC(s);
                        if constexpr (MODE == PASS_SCORE) lg_sum += lgamma((double)s + 1.0);
                    }
                    if constexpr (MODE == PASS_SUMS) {
                        fs = wave_sum(fs);
                        if (lane == 0 && I->sijp != nullptr) gmut<ACC>(I->sijp)[(size_t)i * y + j] = fs;
                    }
                } else if constexpr (MODE == PASS_UPDATE) {
                    const T xv = gconst<T>(I->X)[(size_t)i * y + j];
                    if constexpr (sizeof(T) == 8) {
                        // FP64 plain form: the reference's operations
                        // (X_reciprocal :95, nom :254, denom :284-285,
                        // update :319-323)
                        const T xr = T(1.0) / (xv + eps);
                        auto grad = [&](uint32_t k, T s) { return pb[k] - psi_sp1<PSI, T>(s); };
                        T sumS = T(0), nom = T(0), den = T(0);
                        for (uint32_t k = lane; k < z; k += 64) {
                            const T s = src[k];
                            const T g = grad(k, s);
                            sumS += s;
                            nom += s * xr * (psiA[k] - psia_i[k]);
                            den += s * xr * g;
                        }
                        sumS = wave_sum(sumS);
                        nom = wave_sum(nom);
                        den = wave_sum(den);
                        const T x_over_s = xv / (sumS + eps);
                        for (uint32_t k = lane; k < z; k += 64) {
                            const T s = src[k];
                            const T gm = psiA[k] - psia_i[k];
                            const T sn = as_stored(s * ((grad(k, s) + nom) * x_over_s / (gm + den + eps)));
                            dst[k] = sn;
                            add_partials(k, sn);
                        }
                    } else {
                        // FP32 bulk: eps = 1e-50 flushes to zero in float; the
                        // reference's double-promoted guard makes an X_ij = 0
                        // or all-zero fiber update to exactly 0, taken
                        // explicitly, and an exact-zero denominator (a single
                        // row with beta = 1) updates to 0 rather than 0/0
                        const float epsf = static_cast<float>(eps);
                        const bool live = xv > 0.0f;
                        const float xr = live ? 1.0f / (xv + epsf) : 0.0f;
                        auto grad = [&](uint32_t k, float s) {
                            const float ps = fast_psi ? psi_ge1_f32(s + 1.0f) : psi_sp1<PSI_F32, float>(s);
                            return pb[k] - ps;
                        };
                        float sumS = 0.0f, nom = 0.0f, den = 0.0f;
                        for (uint32_t k = lane; k < z; k += 64) {
                            const float s = src[k];
                            const float g = grad(k, s);
                            sumS += s;
                            const float t = s * xr;
                            nom = fmaf(t, psiA[k] - psia_i[k], nom);
                            den = fmaf(t, g, den);
                        }
                        sumS = wave_sum(sumS);
                        nom = wave_sum(nom);
                        den = wave_sum(den);
                        const bool upd = live && sumS != 0.0f;
                        const float x_over_s = upd ? xv / (sumS + epsf) : 0.0f;
                        float den_e = den + epsf;
                        if (den_e == 0.0f) den_e = FLT_MIN;
                        for (uint32_t k = lane; k < z; k += 64) {
                            const float s = src[k];
                            const float gm = psiA[k] - psia_i[k];
                            const float fct = (grad(k, s) + nom) * x_over_s * recip_fast<float>(gm + den_e);
                            const float sn = as_stored(upd ? s * fct : 0.0f);
                            dst[k] = sn;
                            add_partials(k, sn);
                        }
                    }
                } else {
                    // bld::bld_add's step (src/bld/bld_add.hpp:137-181):
                    // grad_S = psi(beta_eph) - psi(S+1) - psi(A) + psi(alpha_eph),
                    // S_mult = sum_k S grad_S, Z = log S + eps + eta S (X grad_S
                    // - S_mult), S = X exp(Z) / (|exp(Z)|_1 + 1e-50). exp(Z) is
                    // kept in S between the two reductions (each lane rereads
                    // only the elements it wrote).
                    const T xv = gconst<T>(I->X)[(size_t)i * y + j];
                    auto grad = [&](uint32_t k, T s) -> T {
                        if constexpr (sizeof(T) == 8) {
                            const T ps = psi_sp1<PSI, T>(s);
                            return ((pb[k] - ps) - psiA[k]) + psia_i[k];
                        } else {
                            const float ps = fast_psi ? psi_ge1_f32(s + 1.0f) : psi_sp1<PSI_F32, float>(s);
                            return (pb[k] - ps) - (psiA[k] - psia_i[k]);
                        }
                    };
                    T smult = T(0);
                    for (uint32_t k = lane; k < z; k += 64) {
                        const T s = src[k];
                        if constexpr (sizeof(T) == 8)
                            smult += s * grad(k, s);
                        else
                            smult = fmaf(s, grad(k, s), smult);
                    }
                    smult = wave_sum(smult);
                    T norm = T(0);
                    for (uint32_t k = lane; k < z; k += 64) {
                        const T s = src[k];
                        T e;
                        if constexpr (sizeof(T) == 8) {
                            T zk = log(s) + eps;
                            zk += eta * s * (xv * grad(k, s) - smult);
                            e = exp(zk);
                        } else {
                            // exp(log s + t) = s exp(t): one rounding of s
                            // instead of log's (0 stays 0)
                            const float etaf = static_cast<float>(eta);
                            e = s * __expf((etaf * s) * fmaf(xv, grad(k, s), -smult));
                        }
                        dst[k] = e;
                        norm += e;
                    }
                    norm = wave_sum(norm);
                    T scale = T(1);
                    if constexpr (sizeof(T) == 8) {
                        norm += 1e-50;
                    } else {
                        // the reference's 1e-50 guard underflows in float: an
                        // all-zero exp row (X = 0) is taken explicitly
                        scale = norm > 0.0f ? xv / norm : 0.0f;
                    }
                    for (uint32_t k = lane; k < z; k += 64) {
                        const T e = dst[k];
                        T sn;
                        if constexpr (sizeof(T) == 8)
                            sn = as_stored(xv * (e / norm));
                        else
                            sn = as_stored(e * scale);
                        dst[k] = sn;
                        add_partials(k, sn);
                    }
                }
            }
        }
        if constexpr (MODE == PASS_SCORE) {
            lg_sum = wave_sum(lg_sum);
            if (lane == 0) I->score[(size_t)item.ti * I->n_tj + item.tj] = lg_sum;
        }
    }
}

// Sum over the wavefront, the value wave_sum gives (the same pairs in the same
// order: lanes 32 apart, 16, 8, 4, 2, 1) without going through LDS: swaps of
// half wavefronts and of 16-lane rows, then rotations within a row, whose
// lanes repeat with period 8, 4 and 2 by then.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_row(float v) {
    return __builtin_bit_cast(float, dpp_u32<CTRL>(__builtin_bit_cast(uint32_t, v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_row(double v) {
    const uint2 u = __builtin_bit_cast(uint2, v);
    return __builtin_bit_cast(double, make_uint2(dpp_u32<CTRL>(u.x), dpp_u32<CTRL>(u.y)));
}
template <bool WIDE>
__device__ __forceinline__ auto swap_u32(uint32_t v) {
    if constexpr (WIDE)
        return __builtin_amdgcn_permlane32_swap(v, v, false, false);
    else
        return __builtin_amdgcn_permlane16_swap(v, v, false, false);
}
template <bool WIDE>
__device__ __forceinline__ float pair_sum(float v) {
    const auto r = swap_u32<WIDE>(__builtin_bit_cast(uint32_t, v));
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
template <bool WIDE>
__device__ __forceinline__ double pair_sum(double v) {
    const uint2 u = __builtin_bit_cast(uint2, v);
    const auto lo = swap_u32<WIDE>(u.x);
    const auto hi = swap_u32<WIDE>(u.y);
    return __builtin_bit_cast(double, make_uint2((uint32_t)lo[0], (uint32_t)hi[0])) +
           __builtin_bit_cast(double, make_uint2((uint32_t)lo[1], (uint32_t)hi[1]));
}
template <typename T>
__device__ __forceinline__ T wave_sum_reg(T v) {
    v = pair_sum<true>(v);
    v = pair_sum<false>(v);
    v += dpp_row<0x128>(v);  // row_ror:8
    v += dpp_row<0x124>(v);  // row_ror:4
    v += dpp_row<0x122>(v);  // row_ror:2
    v += dpp_row<0x121>(v);  // row_ror:1
    return v;
}

// 64 (NK - 1) < z <= 64 NK, NK 2 to 4: the same tile, sums and order by a block of
// eight wavefronts with the fibers in registers. Wavefront w owns the tile's
// columns w and w + 8 and walks the rows: NK elements of each fiber per lane
// (the next row's are in flight), the gradient evaluated once, its columns'
// partial sums in registers. The new row goes to LDS (two buffers, one barrier
// per row), where one wavefront per 64 k, another each row, adds it up in
// column order. Bit-identical to bld_wide_kernel, whose partials go through
// global memory: per fiber two dependent reads and writes of them, two reads
// of the fiber and 18 shuffles by one wavefront per tile. 320 x 448 x 100 in
// FP32, where memory traffic of 115 MB sets the bound: 664 -> 56 us (2 TB/s; 560
// blocks of 16 dependent rows leave latency between them), 100 iterations with
// S fetched 77 -> 12 ms. Deeper fibers would not fit the registers and keep
// bld_wide_kernel.
constexpr uint32_t kWideWaves = 8;
constexpr int kWideNk = 4;

template <typename T, int MODE, int PSI, int NK>
__global__ void __launch_bounds__(64 * kWideWaves)
    bld_wide_regs_kernel(const BldInst* __restrict__ insts, const PassItem* __restrict__ items,
                         const uint32_t* __restrict__ n_items_p) {
    constexpr uint32_t C = kWideCols / kWideWaves;
    __shared__ T rowbuf[2][kWideCols][64 * NK];
    const uint32_t n_items = *n_items_p;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t buf = 0;
    for (uint32_t it = blockIdx.x; it < n_items; it += gridDim.x) {
        const PassItem item = items[it];
        const BldInst* __restrict__ I = insts + item.inst;
        const uint32_t x = I->x, y = I->y, z = I->z;
        const uint32_t i0 = item.ti * kWideRows, i1 = min(x, i0 + kWideRows);
        const uint32_t j0 = item.tj * kWideCols, nj = min(y - j0, kWideCols);
        // S_src and S are the same tensor after the first pass: no restrict
        const BNMF_GLOBAL T* const Ssrc = gconst<T>(I->S_src);
        BNMF_GLOBAL T* const Sdst = gmut<T>(I->S);
        BNMF_GLOBAL T* __restrict__ const pjk = gmut<T>(I->part_pjk) + ((size_t)item.ti * y + j0) * z;
        BNMF_GLOBAL T* __restrict__ const ipk = gmut<T>(I->part_ipk) + (size_t)item.tj * x * z;
        const BNMF_GLOBAL T* __restrict__ const psia = gconst<T>(I->psia);
        const BNMF_GLOBAL T* __restrict__ const X = gconst<T>(I->X);
        const double eps = I->eps;
        const bool fast_psi = I->nonneg != 0u;
        double eta = 0.0;
        if constexpr (MODE == PASS_ADD) eta = 0.1 / pow((double)*I->iter, 0.55);
        (void)eta;

        T psiA[NK], pa[NK], pb[C][NK], sum[C][NK], next[C][NK], xn[C];
#pragma unroll
        for (int m = 0; m < NK; ++m) {
            const uint32_t k = lane + 64u * m;
            const bool in = k < z;
            if constexpr (MODE != PASS_SUMS) {
                psiA[m] = in ? gconst<T>(I->psiA)[k] : T(0);
                pa[m] = in ? psia[(size_t)i0 * z + k] : T(0);
            }
#pragma unroll
            for (uint32_t c = 0; c < C; ++c) {
                const uint32_t f = w + c * kWideWaves;
                const bool on = in && f < nj;
                if constexpr (MODE != PASS_SUMS) pb[c][m] = on ? gconst<T>(I->psib)[(size_t)(j0 + f) * z + k] : T(0);
                next[c][m] = on ? Ssrc[((size_t)i0 * y + j0 + f) * z + k] : T(0);
                sum[c][m] = T(0);
            }
        }
#pragma unroll
        for (uint32_t c = 0; c < C; ++c) {
            const uint32_t f = w + c * kWideWaves;
            if constexpr (MODE != PASS_SUMS) xn[c] = f < nj ? X[(size_t)i0 * y + j0 + f] : T(0);
        }

        for (uint32_t i = i0; i < i1; ++i) {
            T s[C][NK], xv[C], gm[NK], pa_i[NK];
            const uint32_t i2 = i + 1u < i1 ? i + 1u : i;
#pragma unroll
            for (int m = 0; m < NK; ++m) {
                const uint32_t k = lane + 64u * m;
                if constexpr (MODE != PASS_SUMS) {
                    pa_i[m] = pa[m];
                    gm[m] = psiA[m] - pa[m];
                    pa[m] = k < z ? psia[(size_t)i2 * z + k] : T(0);
                }
#pragma unroll
                for (uint32_t c = 0; c < C; ++c) {
                    const uint32_t f = w + c * kWideWaves;
                    s[c][m] = next[c][m];
                    if (i2 != i && k < z && f < nj) next[c][m] = Ssrc[((size_t)i2 * y + j0 + f) * z + k];
                }
            }
#pragma unroll
            for (uint32_t c = 0; c < C; ++c) {
                const uint32_t f = w + c * kWideWaves;
                if constexpr (MODE != PASS_SUMS) {
                    xv[c] = xn[c];
                    xn[c] = f < nj ? X[(size_t)i2 * y + j0 + f] : T(0);
                }
            }
#pragma unroll
            for (uint32_t c = 0; c < C; ++c) {
                const uint32_t f = w + c * kWideWaves;
                if (f >= nj) continue;
                BNMF_GLOBAL T* const dst = Sdst + ((size_t)i * y + j0 + f) * z;
                auto in = [&](int m) { return 64u * (m + 1u) <= 64u * (NK - 1u) || lane + 64u * m < z; };
                // the new element: stored, and added to its column and row
                auto put = [&](int m, T sn) {
                    if constexpr (MODE != PASS_SUMS) dst[lane + 64u * m] = sn;
                    sum[c][m] = i == i0 ? sn : sum[c][m] + sn;
                    rowbuf[buf][f][lane + 64u * m] = sn;
                };
                if constexpr (MODE == PASS_SUMS) {
                    T fs = T(0);
#pragma unroll
                    for (int m = 0; m < NK; ++m)
                        if (in(m)) {
                            put(m, s[c][m]);
                            fs += s[c][m];
                        }
                    fs = wave_sum_reg(fs);
                    if (lane == 0 && I->sijp != nullptr) gmut<T>(I->sijp)[(size_t)i * y + j0 + f] = fs;
                } else if constexpr (MODE == PASS_UPDATE) {
                    T g[NK];
                    if constexpr (sizeof(T) == 8) {
                        const T xr = T(1.0) / (xv[c] + eps);
                        T sumS = T(0), nom = T(0), den = T(0);
#pragma unroll
                        for (int m = 0; m < NK; ++m)
                            if (in(m)) {
                                const T sv = s[c][m];
                                g[m] = pb[c][m] - psi_sp1<PSI, T>(sv);
                                sumS += sv;
                                nom += sv * xr * gm[m];
                                den += sv * xr * g[m];
                            }
                        sumS = wave_sum_reg(sumS);
                        nom = wave_sum_reg(nom);
                        den = wave_sum_reg(den);
                        const T x_over_s = xv[c] / (sumS + eps);
#pragma unroll
                        for (int m = 0; m < NK; ++m)
                            if (in(m)) put(m, as_stored(s[c][m] * ((g[m] + nom) * x_over_s / (gm[m] + den + eps))));
                    } else {
                        const float epsf = static_cast<float>(eps);
                        const bool live = xv[c] > 0.0f;
                        const float xr = live ? 1.0f / (xv[c] + epsf) : 0.0f;
                        float sumS = 0.0f, nom = 0.0f, den = 0.0f;
#pragma unroll
                        for (int m = 0; m < NK; ++m)
                            if (in(m)) {
                                const float sv = s[c][m];
                                const float ps = fast_psi ? psi_ge1_f32(sv + 1.0f) : psi_sp1<PSI_F32, float>(sv);
                                g[m] = pb[c][m] - ps;
                                sumS += sv;
                                const float t = sv * xr;
                                nom = fmaf(t, gm[m], nom);
                                den = fmaf(t, g[m], den);
                            }
                        sumS = wave_sum_reg(sumS);
                        nom = wave_sum_reg(nom);
                        den = wave_sum_reg(den);
                        const bool upd = live && sumS != 0.0f;
                        const float x_over_s = upd ? xv[c] / (sumS + epsf) : 0.0f;
                        float den_e = den + epsf;
                        if (den_e == 0.0f) den_e = FLT_MIN;
#pragma unroll
                        for (int m = 0; m < NK; ++m)
                            if (in(m)) {
                                const float fct = (g[m] + nom) * x_over_s * recip_fast<float>(gm[m] + den_e);
                                put(m, as_stored(upd ? s[c][m] * fct : 0.0f));
                            }
                    }
                } else {
                    T g[NK], e[NK];
                    T smult = T(0);
#pragma unroll
                    for (int m = 0; m < NK; ++m)
                        if (in(m)) {
                            const T sv = s[c][m];
                            if constexpr (sizeof(T) == 8) {
                                const T ps = psi_sp1<PSI, T>(sv);
                                g[m] = ((pb[c][m] - ps) - psiA[m]) + pa_i[m];
                                smult += sv * g[m];
                            } else {
                                const float ps = fast_psi ? psi_ge1_f32(sv + 1.0f) : psi_sp1<PSI_F32, float>(sv);
                                g[m] = (pb[c][m] - ps) - gm[m];
                                smult = fmaf(sv, g[m], smult);
                            }
                        }
                    smult = wave_sum_reg(smult);
                    T norm = T(0);
#pragma unroll
                    for (int m = 0; m < NK; ++m)
                        if (in(m)) {
                            const T sv = s[c][m];
                            if constexpr (sizeof(T) == 8) {
                                T zk = log(sv) + eps;
                                zk += eta * sv * (xv[c] * g[m] - smult);
                                e[m] = exp(zk);
                            } else {
                                const float etaf = static_cast<float>(eta);
                                e[m] = sv * __expf((etaf * sv) * fmaf(xv[c], g[m], -smult));
                            }
                            norm += e[m];
                        }
                    norm = wave_sum_reg(norm);
                    T scale = T(1);
                    if constexpr (sizeof(T) == 8)
                        norm += 1e-50;
                    else
                        scale = norm > 0.0f ? xv[c] / norm : 0.0f;
#pragma unroll
                    for (int m = 0; m < NK; ++m)
                        if (in(m)) {
                            if constexpr (sizeof(T) == 8)
                                put(m, as_stored(xv[c] * (e[m] / norm)));
                            else
                                put(m, as_stored(e[m] * scale));
                        }
                }
            }
            __syncthreads();
            // the row's sums; a buffer is written again only after the next
            // barrier, which every reader reaches when it is done
            const uint32_t m = (w + (i - i0) * NK) % kWideWaves, k = lane + 64u * m;
            if (m < NK && k < z) {
                T r = rowbuf[buf][0][k];
#pragma unroll 5
                for (uint32_t f = 1; f < nj; ++f) r += rowbuf[buf][f][k];
                ipk[(size_t)i * z + k] = r;
            }
            buf ^= 1u;
        }
#pragma unroll
        for (uint32_t c = 0; c < C; ++c) {
            const uint32_t f = w + c * kWideWaves;
#pragma unroll
            for (int m = 0; m < NK; ++m) {
                const uint32_t k = lane + 64u * m;
                if (f < nj && k < z) pjk[(size_t)f * z + k] = sum[c][m];
            }
        }
    }
}

template <typename T, int MODE, int PSI>
static hipError_t launch_wide_regs(int nk, dim3 grid, hipStream_t st, const BldInst* insts, const PassItem* items,
                                   const uint32_t* n_items) {
    const dim3 block(64 * kWideWaves);
    switch (nk) {
        case 2: hipLaunchKernelGGL((bld_wide_regs_kernel<T, MODE, PSI, 2>), grid, block, 0, st, insts, items, n_items); break;
        case 3: hipLaunchKernelGGL((bld_wide_regs_kernel<T, MODE, PSI, 3>), grid, block, 0, st, insts, items, n_items); break;
        case 4: hipLaunchKernelGGL((bld_wide_regs_kernel<T, MODE, PSI, 4>), grid, block, 0, st, insts, items, n_items); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

int wide_regs_nk(uint32_t z) { return z <= 64u * kWideNk ? (int)((z + 63u) / 64u) : 0; }

template <typename T, typename ACC, int MODE, int PSI>
static hipError_t launch_wide_t(dim3 grid, hipStream_t st, const BldInst* insts, const PassItem* items,
                                const uint32_t* n_items) {
    hipLaunchKernelGGL((bld_wide_kernel<T, ACC, MODE, PSI>), grid, dim3(64), 0, st, insts, items, n_items);
    return hipGetLastError();
}

// dtype 0 = float, 1 = double; psi and mode as for launch_pass; nk 2 to 4: every
// instance of the launch has 64 (nk - 1) < z <= 64 nk, 0: any z
hipError_t launch_pass_wide(int dtype, int psi, int mode, int nk, dim3 grid, hipStream_t st, const BldInst* insts,
                            const PassItem* items, const uint32_t* n_items) {
    if (nk > 0 && mode != PASS_SCORE) {
        if (dtype == 0) {
            switch (mode) {
                case PASS_UPDATE: return launch_wide_regs<float, PASS_UPDATE, PSI_F32>(nk, grid, st, insts, items, n_items);
                case PASS_SUMS: return launch_wide_regs<float, PASS_SUMS, PSI_F32>(nk, grid, st, insts, items, n_items);
                case PASS_ADD: return launch_wide_regs<float, PASS_ADD, PSI_F32>(nk, grid, st, insts, items, n_items);
            }
            return hipErrorInvalidValue;
        }
        switch (mode) {
            case PASS_UPDATE:
                if (psi == PSI_F64_APPR)
                    return launch_wide_regs<double, PASS_UPDATE, PSI_F64_APPR>(nk, grid, st, insts, items, n_items);
                return launch_wide_regs<double, PASS_UPDATE, PSI_F64_EXACT>(nk, grid, st, insts, items, n_items);
            case PASS_SUMS: return launch_wide_regs<double, PASS_SUMS, PSI_F64_EXACT>(nk, grid, st, insts, items, n_items);
            case PASS_ADD: return launch_wide_regs<double, PASS_ADD, PSI_F64_APPR>(nk, grid, st, insts, items, n_items);
        }
        return hipErrorInvalidValue;
    }
    if (dtype == 0) {
        switch (mode) {
            case PASS_UPDATE: return launch_wide_t<float, float, PASS_UPDATE, PSI_F32>(grid, st, insts, items, n_items);
            case PASS_SUMS: return launch_wide_t<float, float, PASS_SUMS, PSI_F32>(grid, st, insts, items, n_items);
            case PASS_SCORE: return launch_wide_t<float, double, PASS_SCORE, PSI_F32>(grid, st, insts, items, n_items);
            case PASS_ADD: return launch_wide_t<float, float, PASS_ADD, PSI_F32>(grid, st, insts, items, n_items);
        }
    } else {
        switch (mode) {
            case PASS_UPDATE:
                if (psi == PSI_F64_APPR)
                    return launch_wide_t<double, double, PASS_UPDATE, PSI_F64_APPR>(grid, st, insts, items, n_items);
                return launch_wide_t<double, double, PASS_UPDATE, PSI_F64_EXACT>(grid, st, insts, items, n_items);
            case PASS_SUMS: return launch_wide_t<double, double, PASS_SUMS, PSI_F64_EXACT>(grid, st, insts, items, n_items);
            case PASS_SCORE: return launch_wide_t<double, double, PASS_SCORE, PSI_F64_EXACT>(grid, st, insts, items, n_items);
            case PASS_ADD:
                // the additive solver evaluates every psi with psi_appr
                return launch_wide_t<double, double, PASS_ADD, PSI_F64_APPR>(grid, st, insts, items, n_items);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace bnmf
