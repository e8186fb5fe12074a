// bld_tiny.hip — bld_mult in FP64 for instances of one tile and at most
// kTinyElems elements: every iteration of a solve in one launch, a block per
// instance, the tensor and all of its sums in LDS.
//
// A small instance gives each of an iteration's three launches (step, prep,
// psi(A)) a microsecond of work; what it waits for is the launches, the trip of
// the sums through the L2 between them and three digamma chains in a row. Here
// an iteration is four stretches between block barriers:
//   sums    S_i+k (a wavefront per row), S_+jk (a thread per column and k)
//   psi     psi(A), psi(alpha_eph), psi(beta_eph) and every psi(S + 1), none of
//           which needs another: a thread per value
//   fibers  S_ij+, nom and denom (two or four lanes per fiber)
//   update  a thread per element
// so one digamma chain is left of the three. Every sum runs in the order of the
// step pass, the prep kernel and the psi(A) kernel (bld_pass_f64.hip,
// bld_kernels.hip) with their operations, so an instance gives the same bits
// here and in a batch with larger ones, which runs those. What bounds it is
// latency (the digamma chain, LDS, four barriers) up to about 500 elements, then
// the FP64 rate of its one CU.
//
// Measured on one MI355X, an iteration here and by three launches: 8x10x3 3.8 us
// against 13.2 (2000 of them 31 -> 8 ms), 10x20x5 4.7 against 17.2, 8x16x16 7.2
// against 19.1, 64x32x2 18.6 against 47.8, 4x16x64 12.8 against 20.9, and with
// mostly zero counts 12.4 against 15.7 (packed fibers). 256 of 8x32x16 at once 12.1
// against 23.1, 1024 of them 48 against 55: the line of kTinyElems lies where the
// gain for full batches ends and the LDS for one block does. Beyond 1024 instances,
// those of few rows take the passes (Batch::plan).
//
// Reference operations: src/bld/bld_mult/bld_mult_funcs.hpp (X_reciprocal :95,
// alpha_eph :130-141, beta_eph :152-163, grad_plus :177-192, grad_minus
// :213-220, nom :242-259, denom :272-290, update_S :307-327).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "bld_types.hpp"
#include "bnmf_internal.hpp"
#include "digamma.hpp"
#include "pass_common.hpp"

namespace bnmf {

namespace {

constexpr uint32_t kTinyThreads = 1024;
constexpr uint32_t kTinyClasses = 4;  // row classes of S_+jk: the step pass's wavefronts

template <int PSI, uint32_t LPF>
__device__ __forceinline__ void tiny_solve(const BldInst* __restrict__ I, uint32_t iters, double* __restrict__ lds) {
    const uint32_t tid = threadIdx.x, NT = blockDim.x, lane = tid & 63u;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), waves = NT >> 6;
    const uint32_t x = I->x, y = I->y, z = I->z, rw = I->rw;
    const uint32_t F = x * y, E = F * z, xz = x * z, yz = y * z;
    const double eps = I->eps;
    const float inv_z = I->inv_z, inv_y = 1.0f / (float)y;
    double* const S = lds;           // E
    double* const ps = S + E;        // psi(S + 1), E
    double* const xs = ps + E;       // X, F
    double* const xr = xs + F;       // X_reciprocal, F
    double* const fs = xr + F;       // nom, denom, X / S_ij+ of a fiber, 3 F
    double* const psib = fs + 3 * F; // S_+jk, then psi(beta_eph), yz
    double* const aeph = psib + yz;  // alpha_eph, xz
    double* const psia = aeph + xz;  // psi(alpha_eph), xz
    double* const psiA = psia + xz;  // psi(A), z
    double* const al = psiA + z;     // alpha, x
    double* const be = al + x;       // beta, z

    for (uint32_t e = tid; e < E; e += NT) S[e] = gconst<double>(I->S_src)[e];
    for (uint32_t f = tid; f < F; f += NT) {
        const double v = gconst<double>(I->X)[f];
        xs[f] = v;
        xr[f] = 1.0 / (v + eps);
    }
    for (uint32_t i = tid; i < x; i += NT) al[i] = I->alpha[i];
    for (uint32_t k = tid; k < z; k += NT) be[k] = I->beta[k];
    // the step pass's lane (fiber, p): chunks m0 .. m0 + mcount - 1 of rw
    // elements, visited as m0 + (u ^ xm)
    const uint32_t p = tid % LPF;
    const uint32_t nchunk = z / rw, cp = (nchunk + LPF - 1u) / LPF;
    const uint32_t xmask = nchunk % LPF == 0u ? min(cp & (0u - cp), 4u) - 1u : 0u;
    const uint32_t m0 = min(p * cp, nchunk), mcount = min(cp, nchunk - m0);
    const uint32_t zq = I->zq, kq = lane & (zq - 1u), part = lane >> I->zq_log2, L = 64u >> I->zq_log2;
    __syncthreads();

    for (uint32_t t = 0;; ++t) {
        const bool last = t == iters;
        // S_i+k: eight strided partial sums a lane, their tree, then the parts
        for (uint32_t i = w; i < x; i += waves) {
            double r[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) r[v] = 0.0;
            if (kq < z) {
                const double* const row = S + i * yz + kq;
                for (uint32_t f0 = part; f0 < y; f0 += 8u * L) {
#pragma unroll
                    for (int v = 0; v < 8; ++v) {
                        const uint32_t j = f0 + (uint32_t)v * L;
                        if (j < y) r[v] += row[j * z];
                    }
                }
            }
            double rs = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
            for (uint32_t off = zq; off < 64u; off <<= 1) rs += __shfl_xor(rs, (int)off);
            if (part == 0u && kq < z) {
                if (last)
                    gmut<double>(I->part_ipk)[i * z + kq] = rs;
                else
                    aeph[i * z + kq] = rs + al[i];
            }
        }
        // S_+jk: the rows of each class in order, then the classes
        for (uint32_t e = tid; e < yz; e += NT) {
            double c[kTinyClasses];
#pragma unroll
            for (uint32_t v = 0; v < kTinyClasses; ++v) c[v] = 0.0;
            for (uint32_t i0 = 0; i0 < x; i0 += kTinyClasses) {
#pragma unroll
                for (uint32_t v = 0; v < kTinyClasses; ++v)
                    if (i0 + v < x) c[v] += S[(i0 + v) * yz + e];
            }
            const double s = ((c[0] + c[1]) + c[2]) + c[3];
            if (last)
                gmut<double>(I->part_pjk)[e] = s;
            else
                psib[e] = s + be[e - fiber_of(e, inv_z) * z];
        }
        if (last) break;
        __syncthreads();

        // every digamma: psi(A) first, whose sum over the rows goes by prep
        // chunks (at most four)
        const uint32_t n_psi = z + xz + yz + E;
        for (uint32_t u = tid; u < n_psi; u += NT) {
            double a, *out;
            if (u < z) {
                double A = 0.0;
                for (uint32_t r0 = 0; r0 < x; r0 += kPrepRows) {
                    double c = 0.0;
                    for (uint32_t r = r0; r < min(x, r0 + kPrepRows); ++r) c += aeph[r * z + u];
                    A += c;
                }
                a = A;
                out = psiA + u;
            } else if (u < z + xz) {
                a = aeph[u - z];
                out = psia + (u - z);
            } else if (u < z + xz + yz) {
                out = psib + (u - z - xz);
                a = *out;
            } else {
                a = S[u - z - xz - yz] + 1.0;
                out = ps + (u - z - xz - yz);
            }
            *out = psi_sel<PSI, double>(a);
        }
        __syncthreads();

        for (uint32_t f = tid / LPF; f < F; f += NT / LPF) {
            const uint32_t i = fiber_of(f, inv_y), j = f - i * y, xm = j & xmask;
            const double *const sf = S + f * z, *const pf = ps + f * z, *const pb = psib + j * z, *const pa = psia + i * z;
            const double xrf = xr[f];
            double sumS = 0.0, nom = 0.0, den = 0.0;
            bool slow = false;
            for (uint32_t u = 0; u < mcount; ++u) {
                const uint32_t mm = (m0 + (u ^ xm)) * rw;
                for (uint32_t k = mm; k < mm + rw; ++k) {
                    const double sk = sf[k];
                    bool fast = true;
                    if constexpr (PSI == PSI_F64_EXACT) {
                        const double xa = sk + 1.0;
                        fast = xa >= 1.0 && xa < 10.0;
                        slow = slow || !fast;
                    }
                    sumS += sk;
                    nom += sk * xrf * (psiA[k] - pa[k]);
                    const double dn = den + sk * xrf * (pb[k] - pf[k]);
                    den = fast ? dn : den;
                }
            }
            // the step pass adds the denom terms of elements with S + 1
            // outside [1, 10) after the others
            if (slow) {
                for (uint32_t u = 0; u < mcount; ++u) {
                    const uint32_t mm = (m0 + (u ^ xm)) * rw;
                    for (uint32_t k = mm; k < mm + rw; ++k) {
                        const double sk = sf[k], xa = sk + 1.0;
                        if (!(xa >= 1.0 && xa < 10.0)) den += sk * xrf * (pb[k] - pf[k]);
                    }
                }
            }
#pragma unroll
            for (uint32_t o = 1; o < LPF; o <<= 1) {
                sumS += __shfl_xor(sumS, (int)o);
                nom += __shfl_xor(nom, (int)o);
                den += __shfl_xor(den, (int)o);
            }
            if (p == 0u) {
                fs[f * 3u] = nom;
                fs[f * 3u + 1u] = den;
                fs[f * 3u + 2u] = xs[f] / (sumS + eps);
            }
        }
        __syncthreads();

        for (uint32_t e = tid; e < E; e += NT) {
            const uint32_t f = fiber_of(e, inv_z), k = e - f * z, i = fiber_of(f, inv_y), j = f - i * y;
            const double nom = fs[f * 3u], den = fs[f * 3u + 1u], x_over_s = fs[f * 3u + 2u];
            const double g = psib[j * z + k] - ps[e], gm = psiA[k] - psia[i * z + k];
            S[e] = as_stored(S[e] * div_moderate((g + nom) * x_over_s, gm + den + eps));
        }
        __syncthreads();
    }
    for (uint32_t e = tid; e < E; e += NT) gmut<double>(I->S)[e] = S[e];
}

template <int PSI>
__global__ void __launch_bounds__(kTinyThreads) bld_tiny_kernel(const BldInst* __restrict__ insts, uint32_t iters) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const BldInst* __restrict__ I = insts + blockIdx.x;
    if ((size_t)I->x * I->y * I->z == 0) return;
    if (I->z <= 32u)
        tiny_solve<PSI, 2>(I, iters, reinterpret_cast<double*>(lds_raw));
    else
        tiny_solve<PSI, 4>(I, iters, reinterpret_cast<double*>(lds_raw));
}

}  // namespace

size_t tiny_lds(uint32_t x, uint32_t y, uint32_t z) {
    const size_t F = (size_t)x * y;
    return (2 * F * z + 5 * F + (size_t)y * z + 2 * (size_t)x * z + 2 * z + x) * 8;
}

// threads: one per digamma of the largest instance, as far as a block goes
uint32_t tiny_threads(uint32_t x, uint32_t y, uint32_t z) {
    const uint32_t n = z + (x + y) * z + x * y * z;
    return n >= kTinyThreads ? kTinyThreads : (n + 63u) / 64u * 64u;
}

hipError_t launch_tiny(int psi, uint32_t n_inst, uint32_t threads, size_t lds, hipStream_t st, const BldInst* insts,
                       uint32_t iters) {
    if (psi == PSI_F64_APPR)
        hipLaunchKernelGGL(bld_tiny_kernel<PSI_F64_APPR>, dim3(n_inst), dim3(threads), lds, st, insts, iters);
    else
        hipLaunchKernelGGL(bld_tiny_kernel<PSI_F64_EXACT>, dim3(n_inst), dim3(threads), lds, st, insts, iters);
    return hipGetLastError();
}

hipError_t init_tiny_attributes() {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(bld_tiny_kernel<PSI_F64_EXACT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTinyLds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(bld_tiny_kernel<PSI_F64_APPR>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTinyLds);
    return e;
}

}  // namespace bnmf
