// bld_appr_live.hip — the approximate solver's FP64 iteration
// (bld_appr.hpp:320-348) over the nonempty entries of X, for z <= 64.
//
// In factored form an entry with X_ij = 0 contributes nothing to any sum of an
// iteration (S_ijk, orig_over_appr and orig_over_appr_squared are all
// proportional to X_ij), so a count matrix costs what its counts cost. X is kept
// as lists of its nonempty entries by row and by column. A wavefront (four
// for long lists) takes one row or column: groups of G lanes (G = z rounded up
// to a power of two) hold k and walk its entries, 64 / G at a time, the other
// factor's row arriving as one contiguous read; X_hat and the fiber sums A and B
// are sums over the group, and what is summed over the row or column stays in
// the lane. So a row's S_i+k, psi(alpha_eph), and the numerator, denominator,
// step and normalisation of its nu are finished where they are summed: no
// per-tile partials, no prep and no factor kernel. A half-step is three
// launches:
//   sums   rows: S_i+k, psi(alpha_eph), column sums of alpha_eph per block;
//          columns: S_+jk, psi(beta_eph)
//   psi(A) from those sums
//   step   rows (nu) or columns (mu): the two sums of update_nu / update_mu
//          (:105-226, bld_appr.hip), the step and the normalisation
// mu is held transposed (y x z) during a solve, so both factors' rows are
// contiguous in k.
//
// What bounds a launch on a sparse matrix is latency: a wavefront's walk is a
// chain of dependent reads (list, factor row), group sums and psi, with the
// next entry's reads in flight while the current one is evaluated; on a full
// one it is the FP64 arithmetic of psi and of three divisions. Per iteration,
// dense passes before, lists now: 1024 x 1024 x 32, 975 -> 73 us at 2 % nonempty
// entries, 131 at 10 %, 307 at 30 %; 384 x 384 x 32, 492 -> 51 us at 10 %; 16
// instances of up to 384 x 384 x 32 (100 iterations with S fetched), 96 -> 16 ms.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "bld_types.hpp"
#include "digamma.hpp"
#include "pass_common.hpp"

namespace bnmf {

namespace {

template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const int2 u = __builtin_bit_cast(int2, v);
    const int lo = __builtin_amdgcn_update_dpp(0, u.x, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, u.y, CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, make_int2(lo, hi));
}

// Sum over aligned groups of G lanes, the same value in each of them: quad
// permutes, then mirrors of 8 and 16 lanes (whose halves are uniform by then),
// then shuffles.
template <int G>
__device__ __forceinline__ double group_sum(double v) {
    if constexpr (G >= 2) v += dpp<0xB1>(v);   // quad_perm 1 0 3 2
    if constexpr (G >= 4) v += dpp<0x4E>(v);   // quad_perm 2 3 0 1
    if constexpr (G >= 8) v += dpp<0x141>(v);  // row_half_mirror
    if constexpr (G >= 16) v += dpp<0x140>(v); // row_mirror
    if constexpr (G >= 32) v += __shfl_xor(v, 16);
    if constexpr (G >= 64) v += __shfl_xor(v, 32);
    return v;
}

__device__ __forceinline__ double psi_appr(double v) { return psi_sel<PSI_F64_APPR, double>(v); }

// What the block's lists are: rows (entries name columns) or columns.
enum LiveSide : int { SIDE_ROWS = 0, SIDE_COLS = 1 };

// Sums of two accumulators over the wavefront's groups and the wavefronts of
// the list, in a fixed order; valid in the first wavefront's lanes.
template <int G>
__device__ __forceinline__ void list_sum(double& a, double& b, uint32_t wpl, double (*red)[2][64]) {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
#pragma unroll
    for (int off = G; off < 64; off <<= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if (wpl > 1u) {
        red[w][0][lane] = a;
        red[w][1][lane] = b;
        __syncthreads();
        a = (red[0][0][lane] + red[1][0][lane]) + (red[2][0][lane] + red[3][0][lane]);
        b = (red[0][1][lane] + red[1][1][lane]) + (red[2][1][lane] + red[3][1][lane]);
    }
}

// STEP 0: sums; 1: step. own: the list's factor row; other: the entries' factor.
template <int G, int SIDE, int STEP>
__device__ __forceinline__ void live_list(const ApprInst& I, uint32_t first, uint32_t wpl, double (*red)[2][64], double* asum) {
    constexpr uint32_t F = 64u / G;
    const uint32_t lane = threadIdx.x & 63u, w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t k = lane & (G - 1u), grp = lane / G, z = I.z;
    const uint32_t n_lists = SIDE == SIDE_ROWS ? I.x : I.y;
    const uint32_t list = first + (wpl > 1u ? 0u : w);
    const bool on = list < n_lists, act = on && k < z;
    const uint32_t kc = k < z ? k : 0u;
    BNMF_GLOBAL double* const own = gmut<double>(SIDE == SIDE_ROWS ? I.nu : I.muT);
    const BNMF_GLOBAL double* const other = gconst<double>(SIDE == SIDE_ROWS ? I.muT : I.nu);
    const BNMF_GLOBAL uint32_t* const ptr = gconst<uint32_t>(SIDE == SIDE_ROWS ? I.rptr : I.cptr);
    const BNMF_GLOBAL uint32_t* const idx = gconst<uint32_t>(SIDE == SIDE_ROWS ? I.ridx : I.cidx);
    const BNMF_GLOBAL double* const xs = gconst<double>(SIDE == SIDE_ROWS ? I.rxv : I.cxv);
    const double eps = I.eps;
    const uint32_t b = on ? ptr[list] : 0u, e = on ? ptr[list + 1u] : 0u;
    const size_t at = (size_t)(on ? list : 0u) * z + kc;
    const double own_k = act ? own[at] : 0.0;
    // step: grad_minus of the row, or psi(beta_eph) of the column
    double side_k = 0.0, pA = 0.0;
    if constexpr (STEP == 1) {
        pA = gconst<double>(I.psiA)[kc];
        side_k = SIDE == SIDE_ROWS ? pA - gconst<double>(I.psia)[at] : gconst<double>(I.psib)[at];
    }
    // zero, or NaN once the solve has lost psi(A): an empty list's factor is then
    // lost too, as 0 times a gradient makes it in the dense passes
    double n = pA - pA, d = 0.0;
    const uint32_t stride = F * (wpl > 1u ? 4u : 1u), off = grp + (wpl > 1u ? w * F : 0u);
    // the next entry's factor row is in flight while the current one is evaluated
    uint32_t t = b + off;
    uint32_t j0 = t < e ? idx[t] : 0u, j1 = t + stride < e ? idx[t + stride] : 0u;
    double x0 = t < e ? xs[t] : 0.0, x1 = t + stride < e ? xs[t + stride] : 0.0;
    double o0 = other[(size_t)j0 * z + kc];
    double p0 = 0.0;
    const BNMF_GLOBAL double* const psi_o = gconst<double>(SIDE == SIDE_ROWS ? I.psib : I.psia);
    if constexpr (STEP == 1) p0 = psi_o[(size_t)j0 * z + kc];
    // every group of the wavefront walks as long as the longest
    const uint32_t steps = e > b ? (e - b + stride - 1u) / stride : 0u;
    for (uint32_t s = 0; s < steps; ++s) {
        const double xv = x0;
        const double ok = act ? o0 : 0.0;
        const double pk = p0;
        x0 = x1;
        o0 = other[(size_t)j1 * z + kc];
        if constexpr (STEP == 1) p0 = psi_o[(size_t)j1 * z + kc];
        t += stride;
        j1 = t + stride < e ? idx[t + stride] : 0u;
        x1 = t + stride < e ? xs[t + stride] : 0.0;
        // X_hat (update_X_hat :12-15), orig_over_appr (:17-32), S (:34-48)
        const double nm = own_k * ok;
        const double h = group_sum<G>(nm);
        const double oa = xv > 0.0 ? xv / (h + eps) : 0.0;
        const double s_k = oa * nm;
        if constexpr (STEP == 0) {
            n += s_k;
        } else {
            const double oa2 = xv > 0.0 ? xv / (h * h + eps) : 0.0;
            const double gm = SIDE == SIDE_ROWS ? side_k : pA - pk;
            const double gp = (SIDE == SIDE_ROWS ? pk : side_k) - psi_appr(s_k + 1.0);
            const double A = group_sum<G>(k < z ? nm * gm : 0.0), B = group_sum<G>(k < z ? nm * gp : 0.0);
            n += ok * (oa * gp + oa2 * A);
            d += ok * (oa * gm + oa2 * B);
        }
    }
    list_sum<G>(n, d, wpl, red);
    const bool write = act && grp == 0u && (wpl == 1u || w == 0u);
    if constexpr (STEP == 0) {
        if constexpr (SIDE == SIDE_ROWS) {
            const double eph = n + (on ? I.alpha[list] : 1.0);
            if (write) gmut<double>(I.psia)[at] = psi_appr(eph);
            // the block's sum of alpha_eph over its rows, in row order
            if (wpl > 1u) {
                if (write) gmut<double>(I.partA)[(size_t)first * z + k] = eph;
            } else {
                if (grp == 0u) asum[w * 64u + k] = act ? eph : 0.0;
                __syncthreads();
                if (w == 0u && grp == 0u && k < z)
                    gmut<double>(I.partA)[(size_t)(first / 4u) * z + k] =
                        ((asum[k] + asum[64u + k]) + asum[128u + k]) + asum[192u + k];
            }
        } else {
            if (write) gmut<double>(I.psib)[at] = psi_appr(n + I.beta[kc]);
        }
    } else {
        const double v = k < z ? own_k * (n / (d + eps)) : 0.0;
        const double rs = group_sum<G>(v) + eps;
        if (write) own[at] = v / rs;
    }
}

template <int SIDE, int STEP>
__device__ __forceinline__ void live_lists(const ApprInst& I, uint32_t first, uint32_t wpl, double (*red)[2][64], double* asum) {
    switch (I.zq_log2) {
        case 0: return live_list<1, SIDE, STEP>(I, first, wpl, red, asum);
        case 1: return live_list<2, SIDE, STEP>(I, first, wpl, red, asum);
        case 2: return live_list<4, SIDE, STEP>(I, first, wpl, red, asum);
        case 3: return live_list<8, SIDE, STEP>(I, first, wpl, red, asum);
        case 4: return live_list<16, SIDE, STEP>(I, first, wpl, red, asum);
        case 5: return live_list<32, SIDE, STEP>(I, first, wpl, red, asum);
        default: return live_list<64, SIDE, STEP>(I, first, wpl, red, asum);
    }
}

}  // namespace

// One block per item: ti the first list, tj its side, pad the wavefronts per
// list (1: four lists, 4: one). STEP 0: both sides; 1: the items' own side.
template <int STEP>
__global__ void __launch_bounds__(256)
    bld_appr_live_kernel(const ApprInst* __restrict__ insts, const PassItem* __restrict__ items) {
    __shared__ double red[4][2][64];
    __shared__ double asum[256];
    const PassItem item = items[blockIdx.x];
    const ApprInst& I = insts[item.inst];
    if (item.tj == SIDE_ROWS)
        live_lists<SIDE_ROWS, STEP>(I, item.ti, item.pad, red, asum);
    else
        live_lists<SIDE_COLS, STEP>(I, item.ti, item.pad, red, asum);
}

// psi(A), A the sum of alpha_eph over the rows: a block per instance and four
// k, 64 threads to each k's block sums.
__global__ void __launch_bounds__(256) bld_appr_psiA_kernel(const ApprInst* __restrict__ insts) {
    __shared__ double part[4][4];
    const ApprInst& I = insts[blockIdx.x];
    if (I.rptr == nullptr) return;
    const uint32_t k0 = blockIdx.y * 4u, z = I.z, nA = I.nA;
    if (k0 >= z) return;
    const uint32_t kq = threadIdx.x & 3u, r0 = threadIdx.x >> 2;
    const uint32_t k = min(k0 + kq, z - 1u);
    const BNMF_GLOBAL double* const p = gconst<double>(I.partA);
    double s = 0.0;
#pragma unroll 4
    for (uint32_t r = r0; r < nA; r += 64u) s += p[(size_t)r * z + k];
#pragma unroll
    for (int off = 4; off < 64; off <<= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63u) < 4u) part[threadIdx.x >> 6][kq] = s;
    __syncthreads();
    if (threadIdx.x < 4u && k0 + threadIdx.x < z) {
        const double A = (part[0][kq] + part[1][kq]) + (part[2][kq] + part[3][kq]);
        gmut<double>(I.psiA)[k] = psi_appr(A);
    }
}

// The lists, a wavefront per row, then per column (whose reads four
// neighbours share). Counts: rows, then columns; ~0u marks a list that
// holds a negative X_ij or one near the type's range.
__global__ void __launch_bounds__(256)
    bld_appr_count_kernel(const double* __restrict__ X, uint32_t x, uint32_t y, double most, uint32_t* __restrict__ counts) {
    const uint32_t lane = threadIdx.x & 63u, row_blocks = (x + 3u) / 4u;
    const bool rows = blockIdx.x < row_blocks;
    const uint32_t list = (rows ? blockIdx.x : blockIdx.x - row_blocks) * 4u + (threadIdx.x >> 6);
    if (list >= (rows ? x : y)) return;
    const uint32_t len = rows ? y : x;
    const size_t at = rows ? (size_t)list * y : list, step = rows ? 1 : y;
    uint32_t n = 0;
    bool bad = false;
#pragma unroll 4
    for (uint32_t t = lane; t < len; t += 64u) {
        const double v = X[at + t * step];
        n += v != 0.0;
        bad = bad || !(v >= 0.0 && v <= most);
    }
    n = wave_sum(n);
    const bool any = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 0) counts[rows ? list : x + list] = any ? ~0u : n;
}

__global__ void __launch_bounds__(256)
    bld_appr_fill_kernel(const double* __restrict__ X, uint32_t x, uint32_t y, const uint32_t* __restrict__ rptr,
                         uint32_t* __restrict__ ridx, double* __restrict__ rxv, const uint32_t* __restrict__ cptr,
                         uint32_t* __restrict__ cidx, double* __restrict__ cxv) {
    const uint32_t lane = threadIdx.x & 63u, row_blocks = (x + 3u) / 4u;
    const bool rows = blockIdx.x < row_blocks;
    const uint32_t list = (rows ? blockIdx.x : blockIdx.x - row_blocks) * 4u + (threadIdx.x >> 6);
    if (list >= (rows ? x : y)) return;
    const uint32_t len = rows ? y : x;
    const size_t from = rows ? (size_t)list * y : list, step = rows ? 1 : y;
    uint32_t* __restrict__ const idx = rows ? ridx : cidx;
    double* __restrict__ const xv = rows ? rxv : cxv;
    uint32_t at = rows ? rptr[list] : cptr[list];
#pragma unroll 4
    for (uint32_t t0 = 0; t0 < len; t0 += 64u) {
        const uint32_t t = t0 + lane;
        const double v = t < len ? X[from + t * step] : 0.0;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(v != 0.0);
        if (v != 0.0) {
            const uint32_t p = at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            idx[p] = t;
            xv[p] = v;
        }
        at += (uint32_t)__popcll(m);
    }
}

// dst (n x m) = src (m x n) transposed; one thread per element of dst
__global__ void __launch_bounds__(256)
    bld_appr_transpose_kernel(double* __restrict__ dst, const double* __restrict__ src, uint32_t n, uint32_t m) {
    const size_t e = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (e >= (size_t)n * m) return;
    const size_t r = e / m, c = e - r * m;
    dst[e] = src[c * n + r];
}

// ----------------------------------------------------------- launchers
hipError_t launch_appr_live(int step, uint32_t n, hipStream_t st, const ApprInst* insts, const PassItem* items) {
    if (n == 0) return hipSuccess;
    if (step == 0)
        hipLaunchKernelGGL(bld_appr_live_kernel<0>, dim3(n), dim3(256), 0, st, insts, items);
    else
        hipLaunchKernelGGL(bld_appr_live_kernel<1>, dim3(n), dim3(256), 0, st, insts, items);
    return hipGetLastError();
}

hipError_t launch_appr_psiA(uint32_t n_inst, uint32_t zmax, hipStream_t st, const ApprInst* insts) {
    hipLaunchKernelGGL(bld_appr_psiA_kernel, dim3(n_inst, (zmax + 3u) / 4u), dim3(256), 0, st, insts);
    return hipGetLastError();
}

hipError_t launch_appr_count(const double* X, uint32_t x, uint32_t y, uint32_t* counts, hipStream_t st) {
    hipLaunchKernelGGL(bld_appr_count_kernel, dim3((x + 3u) / 4u + (y + 3u) / 4u), dim3(256), 0, st, X, x, y, 1e200,
                       counts);
    return hipGetLastError();
}

hipError_t launch_appr_fill(const double* X, uint32_t x, uint32_t y, const uint32_t* rptr, uint32_t* ridx, double* rxv,
                            const uint32_t* cptr, uint32_t* cidx, double* cxv, hipStream_t st) {
    hipLaunchKernelGGL(bld_appr_fill_kernel, dim3((x + 3u) / 4u + (y + 3u) / 4u), dim3(256), 0, st, X, x, y, rptr, ridx,
                       rxv, cptr, cidx, cxv);
    return hipGetLastError();
}

hipError_t launch_appr_transpose(double* dst, const double* src, uint32_t n, uint32_t m, hipStream_t st) {
    hipLaunchKernelGGL(bld_appr_transpose_kernel, dim3((unsigned)(((size_t)n * m + 255) / 256)), dim3(256), 0, st, dst,
                       src, n, m);
    return hipGetLastError();
}

}  // namespace bnmf
