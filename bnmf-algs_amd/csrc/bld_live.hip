// bld_live.hip — the step passes (bld_mult's multiplicative update, bld_add's
// additive step, FP32 and FP64, z <= 64) over the nonempty fibers of an
// instance.
//
// A count matrix has far fewer counts than entries: with the benchmark's
// model (column totals around 40) 96 % of X is zero at 1024 rows and 98 % at
// 2048. A fiber with X_ij = 0 is zero in S0 and stays zero, so the dense pass
// spends almost all its traffic moving zeros. Here the nonempty fibers of each
// pass tile are kept packed (LiveTile, bld_types.hpp), and a block does one
// tile: the step for its fibers, whatever their rows, then the tile's partial
// sums S_+jk and S_i+k, which the prep kernel reduces as it reduces the dense
// pass's.
//
// The results are those of the dense pass bit for bit (zeros apart from their
// sign): the same operations per element, the fiber sums in the dense pass's
// visit order, and each partial sum in its order with the zero terms left
// out. So an instance may run either kernel, alone or among others. Rows and
// columns of a tile without a fiber are not written: the sums-only pass that
// starts a solve leaves zeros there.
//
// FP32: a lane per fiber. The packed S holds groups of 64 fibers, chunk (four
// elements) by chunk in each lane's own visit order, so a wavefront's load or
// store of S is 1 KiB contiguous and needs no LDS; psi(beta_eph) and
// psi(alpha_eph) rows are gathered through the L1 (neighbouring lanes share
// columns). FP64: a thread per element, because an FP64 digamma is a chain of
// some 500 cycles that a lane with a whole half-fiber would walk 16 times; the
// fiber sums are formed from LDS by the dense pass's two (four) lanes.
//
// What bounds a block is the chain of dependent loads (tile record, fibers,
// gathered rows), each a first touch past the L2, and the barriers between the
// step and the partial sums, not bytes; a launch has one block per tile, two
// to four resident per CU. Measured on one MI355X (kernel trace), one pass of
// the benchmark's counts: 2048 x 2048 x 64 FP32 32 us against 470 us for the
// dense pass, 1024 x 1024 x 32 FP64 29 us against 151 us, 100 x 100 x 17 FP64 with
// a third of X nonempty (8-row tiles) 12 us against some 19 us. Up to which share
// it pays: LivePlan::most_share.
//
// Reference operations: src/bld/bld_mult/bld_mult_funcs.hpp (X_reciprocal
// :95, grad_plus :177-192, nom :242-259, denom :272-290, update_S :307-327),
// src/bld/bld_add.hpp:137-181.

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "bld_types.hpp"
#include "digamma.hpp"
#include "pass_common.hpp"

namespace bnmf {

namespace {

constexpr uint32_t kClasses = 4;   // row classes of S_+jk: the dense block's wavefronts
constexpr uint32_t kWaves32 = 4;   // wavefronts per block
constexpr uint32_t kWaves64 = 8;
constexpr uint32_t kElems64 = 2;   // FP64: elements a thread evaluates at once

__host__ __device__ constexpr uint32_t odd(uint32_t v) { return v | 1u; }

// fiber stride of the value buffer that holds kc elements of each: an odd
// number of 16-byte groups (FP32) or of doubles spreads the lanes over the banks
template <typename T>
__host__ __device__ constexpr uint32_t live_val_stride(uint32_t kc) {
    return sizeof(T) == 4 ? 4u * odd(kc / 4u) : odd(kc);
}
// elements of k (a multiple of 4) the value buffer holds at once for n fibers
// and a fiber of zeros in `bytes` of LDS
template <typename T>
__host__ __device__ inline uint32_t live_kc(uint32_t z, uint32_t n, size_t bytes) {
    uint32_t kc = (z + 3u) / 4u * 4u;
    while (kc > 4u && (size_t)(n + 1u) * live_val_stride<T>(kc) * sizeof(T) > bytes) kc -= 4u;
    return kc;
}

// FP64: fibers of a set (a block's fiber sums, four elements a thread at most), where its launch's fullest tile has `most`
__host__ __device__ constexpr uint32_t live_fibers64(uint32_t z, uint32_t most) {
    const uint32_t f = 64u * kWaves64 * 4u / z, g = f < 128u ? f : 128u;
    return g < most ? g : most;
}
// LDS before the value buffer: the row and column tables, the maps of the
// rows with more than four fibers and, in FP64, psi(alpha_eph) of the rows,
// psi(A), the gradients of the fibers held at once and three values a fiber
template <typename T>
__host__ __device__ constexpr size_t live_lds_fixed(uint32_t z, uint32_t tile_cols, uint32_t rows, uint32_t most) {
    const uint32_t full = most / 5u < rows ? most / 5u : rows;
    size_t b = (size_t)(tile_cols + rows) * 16u + (size_t)full * tile_cols * 2u;
    if (sizeof(T) == 8)
        b += round16((size_t)(rows + 1u) * z * 8u) + round16((size_t)live_fibers64(z, most) * (odd(z) + 3u) * 8u);
    return b;
}

// Element k of fiber q (tile column c) in a tile's packed S.
template <typename T>
__device__ __forceinline__ size_t live_index(const LiveTile* t, uint32_t q, uint32_t c, uint32_t k) {
    if constexpr (sizeof(T) == 4) {
        const uint32_t ng = (t->z + 3u) / 4u, m = (k >> 2) ^ ((c >> t->xs) & t->xm);
        return ((size_t)(q >> 6) * ng + m) * 256u + (q & 63u) * 4u + (k & 3u);
    } else {
        return (size_t)q * t->z + k;
    }
}

// S_i+k of one element over a tile row of TW columns, in the dense pass's
// order: columns part + (v + 8 t) L, summed over t, the eight sums v in a fixed
// tree, the L parts in the tree of its xor shuffles. map: the row's fiber
// numbers, empty columns naming a fiber of zeros.
template <typename T, uint32_t L, uint32_t TW>
__device__ __forceinline__ T live_row_sum(const T* vk, uint32_t vs, const uint16_t* map) {
    typedef uint32_t U4 __attribute__((ext_vector_type(4)));
    U4 m4[TW / 8];
#pragma unroll
    for (uint32_t i = 0; i < TW / 8; ++i) m4[i] = ((const U4*)map)[i];
    T pend[7], x = T(0);
#pragma unroll
    for (uint32_t part = 0; part < (L < TW ? L : TW); ++part) {
        T s[8];
#pragma unroll
        for (uint32_t v = 0; v < 8; ++v) {
            s[v] = T(0);
#pragma unroll
            for (uint32_t t = 0; t < 8; ++t) {
                const uint32_t f = part + (v + 8u * t) * L;
                if (f < TW) s[v] += vk[((m4[f / 8u][(f % 8u) / 2u] >> (16u * (f % 2u))) & 0xffffu) * vs];
            }
        }
        x = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
#pragma unroll
        for (uint32_t l = 0; l < 7; ++l) {
            if ((part >> l) & 1u) {
                x = pend[l] + x;
            } else {
                pend[l] = x;
                break;
            }
        }
    }
    return x;
}
// The same for L = 1 << l_log2 known at run time: a loop over the parts (the
// unrolled forms of every L would be most of a kernel's code, and a launch's
// blocks run it once, out of a cold instruction cache).
template <typename T, uint32_t TW>
__device__ __forceinline__ T live_row_sum_loop(uint32_t l_log2, const T* vk, uint32_t vs, const uint16_t* map) {
    const uint32_t L = 1u << l_log2, parts = min(L, TW);
    T pend[6], x = T(0);
#pragma unroll
    for (uint32_t l = 0; l < 6; ++l) pend[l] = T(0);
    for (uint32_t part = 0; part < parts; ++part) {
        T s[8];
#pragma unroll
        for (uint32_t v = 0; v < 8; ++v) {
            const uint32_t f = part + v * L;
            s[v] = f < TW ? vk[map[f] * vs] : T(0);
        }
        for (uint32_t f0 = part + 8u * L; f0 < TW; f0 += 8u * L) {
#pragma unroll
            for (uint32_t v = 0; v < 8; ++v)
                if (f0 + v * L < TW) s[v] += vk[map[f0 + v * L] * vs];
        }
        x = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
        bool carry = true;
#pragma unroll
        for (uint32_t l = 0; l < 6; ++l) {
            const bool right = (part >> l) & 1u;
            if (carry && right) x = pend[l] + x;
            if (carry && !right) pend[l] = x;
            carry = carry && right;
        }
    }
    return x;
}

// The tile's row and column tables (rows first) and the fuller rows' maps into LDS.
template <uint32_t TW, uint32_t NT>
__device__ __forceinline__ void live_stage_tables(const LiveTile& t, LiveRow* rt) {
    typedef uint32_t U4 __attribute__((ext_vector_type(4)));
    const BNMF_GLOBAL U4* rd = (const BNMF_GLOBAL U4*)gconst<LiveRow>(t.rdesc);
    const BNMF_GLOBAL U4* cd = (const BNMF_GLOBAL U4*)gconst<LiveCol>(t.cdesc);
    U4* const o = reinterpret_cast<U4*>(rt);
    const uint32_t n = (uint32_t)t.rows + t.cols;
    for (uint32_t e = threadIdx.x; e < n; e += NT) o[e] = e < t.rows ? rd[e] : cd[e - t.rows];
    const BNMF_GLOBAL U4* sm = (const BNMF_GLOBAL U4*)gconst<uint16_t>(t.smap);
    const uint32_t nm = (uint32_t)(t.rows - t.rows4) * (TW / 8u);
    for (uint32_t e = threadIdx.x; e < nm; e += NT) o[n + e] = sm[e];
}
template <uint32_t TW>
__device__ __forceinline__ uint32_t live_table_bytes(const LiveTile& t) {
    return (uint32_t)(t.rows + t.cols) * 16u + (uint32_t)(t.rows - t.rows4) * TW * 2u;
}

// The tile's partial sums over elements k0 <= k < k0 + kn from vals (element
// k of fiber q at q * vs + k - k0, fiber n zeros), in the dense pass's order:
// a thread per (row, k), then per (column, k). A row of at most four fibers
// takes the shape of its sum from its table entry; a fuller row walks its tile
// row with the empty columns as zeros (pipelined LDS reads without a branch).
// A column adds the rows of one class in order, then the classes in order.
// L: lane parts of a row (64 / next power of two >= z), 0: known at run time.
template <typename T, uint32_t TW, uint32_t NT, uint32_t L>
__device__ __forceinline__ void live_partials(const LiveTile& t, const LiveRow* rt, const T* vals, uint32_t vs,
                                              uint32_t k0, uint32_t kn) {
    const uint32_t z = t.z, tid = threadIdx.x;
    const float inv_kn = 1.0f / (float)kn;
    {
        BNMF_GLOBAL T* const out = gmut<T>(t.part_ipk) + k0;
        const uint32_t ef = t.rows4 * kn, es = t.rows * kn;
#pragma unroll 2
        for (uint32_t e = tid; e < ef; e += NT) {
            const uint32_t i = fiber_of(e, inv_kn), k = e - i * kn;
            const LiveRow d = rt[i];
            const T* const vk = vals + k;
            const T a = vk[d.q[0] * vs], b = vk[d.q[1] * vs], c = vk[d.q[2] * vs], f = vk[d.q[3] * vs];
            const T ab = a + b, bc = b + c, cf = c + f;
            T s = ab + cf;
            s = d.shape == 0u ? (ab + c) + f : s;
            s = d.shape == 1u ? (a + bc) + f : s;
            s = d.shape == 3u ? a + (bc + f) : s;
            s = d.shape == 4u ? a + (b + cf) : s;
            out[(size_t)d.row * z + k] = s;
        }
        const uint16_t* const mp = reinterpret_cast<const uint16_t*>(rt + t.rows + t.cols);
        for (uint32_t e = ef + tid; e < es; e += NT) {
            const uint32_t i = fiber_of(e, inv_kn), k = e - i * kn, r = rt[i].row;
            const uint16_t* const mr = mp + (i - t.rows4) * TW;
            T sum;
            if constexpr (L > 0)
                sum = live_row_sum<T, L, TW>(vals + k, vs, mr);
            else
                sum = live_row_sum_loop<T, TW>(6u - t.zq_log2, vals + k, vs, mr);
            out[(size_t)r * z + k] = sum;
        }
    }
    {
        const LiveCol* const ct = reinterpret_cast<const LiveCol*>(rt + t.rows);
        BNMF_GLOBAL T* const out = gmut<T>(t.part_pjk) + k0;
        const uint32_t ec = t.cols * kn;
        for (uint32_t e = tid; e < ec; e += NT) {
            const uint32_t a = fiber_of(e, inv_kn), k = e - a * kn;
            const LiveCol d = ct[a];
            const uint32_t m = d.end[3];
            const T* const v = vals + d.q0 * vs + k;
            T sum = T(0), cls = T(0);
            for (uint32_t i = 0; i < m; i += 4u) {
                T f[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) f[u] = v[min(i + u, m - 1u) * vs];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) {
                    const uint32_t at = i + u;
                    if (at < m) {
                        if (at == d.end[0] || at == d.end[1] || at == d.end[2]) {
                            sum += cls;
                            cls = T(0);
                        }
                        cls += f[u];
                    }
                }
            }
            out[(size_t)d.col * z + k] = sum + cls;
        }
    }
}

// psi(s + 1) of U elements. The exact digamma's recurrence (psi_1to10) runs
// for all of them in one loop and their rational parts interleave, so a
// thread's chains overlap; the operations on each are psi_1to10's. Returns
// whether an argument lies outside [1, 10), whose value is then meaningless.
template <int PSI, uint32_t U>
__device__ __forceinline__ bool live_psi(const double (&s)[U], double (&ps)[U]) {
    if constexpr (PSI != PSI_F64_EXACT) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) ps[u] = psi_sp1<PSI, double>(s[u]);
        return false;
    } else {
        double y[U], num[U], den[U];
        bool slow = false;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const double xa = s[u] + 1.0;
            const bool fast = xa >= 1.0 && xa < 10.0;
            slow = slow || !fast;
            y[u] = fast ? xa - 1.0 : 0.0;
            num[u] = 0.0;
            den[u] = 1.0;
        }
        for (;;) {
            bool more = false;
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) more = more || y[u] >= 1.0;
            if (!more) break;
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                const bool on = y[u] >= 1.0;
                num[u] = on ? fma(num[u], y[u], den[u]) : num[u];
                den[u] = on ? den[u] * y[u] : den[u];
                y[u] = on ? y[u] - 1.0 : y[u];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            double q;
            const double p = psi1p_rat(y[u], &q);
            ps[u] = div_moderate(fma(p, den[u], q * num[u]), q * den[u]);
        }
        return slow;
    }
}

}  // namespace

// FP32, z in (4 NG - 4, 4 NG]. The arithmetic is bld_pass_f32z_kernel's; the
// products the compiler contracts there (nom and den scaled by X_reciprocal,
// the exp-row norm) are written as the FMAs they become.
template <int NG, int MODE>
__device__ __forceinline__ void live_step_f32(const LiveTile& t, unsigned char* lds_raw, uint32_t lds_bytes) {
    typedef float V4 __attribute__((ext_vector_type(4)));
    typedef float V4u __attribute__((ext_vector_type(4), aligned(4)));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t z = t.z, n = t.n, xs = t.xs, xmask = t.xm;
    const float epsf = static_cast<float>(t.eps);
    LiveRow* const rt = reinterpret_cast<LiveRow*>(lds_raw);
    const uint32_t fixed = live_table_bytes<kTileCols>(t);
    float* const vals = reinterpret_cast<float*>(lds_raw + fixed);
    const uint32_t kc = live_kc<float>(z, n, lds_bytes - fixed), vs = live_val_stride<float>(kc);
    const bool whole = kc >= z;  // vals holds whole fibers

    BNMF_GLOBAL V4* const Sc = (BNMF_GLOBAL V4*)gmut<float>(t.Sc);
    const BNMF_GLOBAL float* __restrict__ xg = gconst<float>(t.xv);
    const BNMF_GLOBAL uint16_t* __restrict__ fg = gconst<uint16_t>(t.fib);
    const BNMF_GLOBAL float* __restrict__ pb_g = gconst<float>(t.psib);
    const BNMF_GLOBAL float* __restrict__ pa_g = gconst<float>(t.psia);
    const BNMF_GLOBAL float* __restrict__ pA_g = gconst<float>(t.psiA);

    V4 s[NG];
    uint32_t rc = 0;
    float xv = 0.0f;
    auto load_group = [&](uint32_t g) {
        rc = fg[g * 64u + lane];
        const BNMF_GLOBAL V4* src = Sc + (size_t)g * (NG * 64u) + lane;
#pragma unroll
        for (int m = 0; m < NG; ++m) s[m] = src[m * 64];
        xv = xg[g * 64u + lane];
    };
    if (w * 64u < n) load_group(w);
    live_stage_tables<kTileCols, 64u * kWaves32>(t, rt);
    if (threadIdx.x < vs) vals[n * vs + threadIdx.x] = 0.0f;  // the fiber of zeros
    // additive step size 0.1 / (iteration + 1)^0.55 (bld_add.hpp:101-103)
    float etaf = 0.0f;
    if constexpr (MODE == PASS_ADD) etaf = static_cast<float>(0.1 / pow((double)*t.iter, 0.55));

    for (uint32_t g = w; g * 64u < n; g += kWaves32) {
        const uint32_t q = g * 64u + lane;
        const uint32_t c = rc & 63u, r = rc >> 6;
        float gp[4 * NG], gm[4 * NG];
        const uint32_t hsw = (c >> xs) & xmask;
        // psi(beta_eph) and grad_minus in visit order; a last chunk's
        // elements past z are read (the row's successor in the workspace)
        // and not used
        const BNMF_GLOBAL float* const pbr = pb_g + c * z;
        const BNMF_GLOBAL float* const par = pa_g + r * z;
#pragma unroll
        for (int m = 0; m < NG; ++m) {
            const uint32_t mm = ((uint32_t)m ^ hsw) * 4u;
            const V4 pb = *(const BNMF_GLOBAL V4u*)(pbr + mm);
            const V4 pa = *(const BNMF_GLOBAL V4u*)(par + mm);
            const V4 pA = *(const BNMF_GLOBAL V4u*)(pA_g + mm);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                gp[4 * m + v] = pb[v];
                gm[4 * m + v] = pA[v] - pa[v];
            }
        }
        if constexpr (MODE == PASS_ADD) {
            float smult = 0.0f;
#pragma unroll
            for (int k = 0; k < 4 * NG; ++k) {
                if (k < 4 * NG - 4 || (uint32_t)k < z) {
                    const float sk = s[k / 4][k % 4];
                    const float gr = (gp[k] - psi_ge1_f32(sk + 1.0f)) - gm[k];
                    gp[k] = gr;
                    smult = fmaf(sk, gr, smult);
                }
            }
            float norm = 0.0f;
#pragma unroll
            for (int k = 0; k < 4 * NG; ++k) {
                if (k < 4 * NG - 4 || (uint32_t)k < z) {
                    const float sk = s[k / 4][k % 4];
                    const float ex = __expf((etaf * sk) * fmaf(xv, gp[k], -smult));
                    gp[k] = sk * ex;
                    norm = fmaf(sk, ex, norm);
                }
            }
            const float scale = norm > 0.0f ? xv / norm : 0.0f;
#pragma unroll
            for (int k = 0; k < 4 * NG; ++k)
                s[k / 4][k % 4] = (k < 4 * NG - 4 || (uint32_t)k < z) ? as_stored(gp[k] * scale) : 0.0f;
        } else {
            float sumS = 0.0f, nom = 0.0f, den = 0.0f;
#pragma unroll
            for (int k = 0; k < 4 * NG; ++k) {
                if (k < 4 * NG - 4 || (uint32_t)k < z) {
                    const float sk = s[k / 4][k % 4];
                    const float gr = gp[k] - psi_ge1_f32(sk + 1.0f);
                    gp[k] = gr;
                    sumS += sk;
                    nom = fmaf(sk, gm[k], nom);
                    den = fmaf(sk, gr, den);
                }
            }
            const bool upd = xv > 0.0f && sumS != 0.0f;
            const float xh = upd ? 1.0f / (xv + epsf) : 0.0f;
            const float qf = upd ? (sumS + epsf) / xv : 0.0f;
            const float dq = upd ? fmaxf(fmaf(den, xh, epsf) * qf, FLT_MIN) : __builtin_inff();
#pragma unroll
            for (int k = 0; k < 4 * NG; ++k) {
                if (k < 4 * NG - 4 || (uint32_t)k < z) {
                    const float rr = recip_fast<float>(fmaf(gm[k], qf, dq));
                    s[k / 4][k % 4] = as_stored(s[k / 4][k % 4] * (fmaf(nom, xh, gp[k]) * rr));
                } else {
                    s[k / 4][k % 4] = 0.0f;
                }
            }
        }
        if (q < n) {
            BNMF_GLOBAL V4* dst = Sc + (size_t)g * (NG * 64u) + lane;
#pragma unroll
            for (int m = 0; m < NG; ++m) {
                dst[m * 64] = s[m];
                if (whole) *reinterpret_cast<V4*>(vals + q * vs + ((uint32_t)m ^ hsw) * 4u) = s[m];
            }
        }
        if ((g + kWaves32) * 64u < n) load_group(g + kWaves32);
    }

    for (uint32_t k0 = 0; k0 < z; k0 += kc) {
        const uint32_t kn = min(kc, z - k0);
        if (!whole) {
            // elements k0 .. k0 + kc - 1 of every fiber, as this wavefront stored them
            if (k0) __syncthreads();
            for (uint32_t g = w; g * 64u < n; g += kWaves32) {
                const uint32_t q = g * 64u + lane;
                if (q < n) {
                    const uint32_t hsw = ((fg[q] & 63u) >> xs) & xmask;
                    for (uint32_t m = k0 / 4u; m < (k0 + kn + 3u) / 4u; ++m)
                        *reinterpret_cast<V4*>(vals + q * vs + (m * 4u - k0)) =
                            Sc[((size_t)g * NG + (m ^ hsw)) * 64u + lane];
                }
            }
        }
        __syncthreads();
        live_partials<float, kTileCols, 64u * kWaves32, NG == 1 ? 0u : NG == 2 ? 8u : NG <= 4 ? 4u : NG <= 8 ? 2u : 1u>(t, rt, vals, vs, k0, kn);
    }
}

// One launch for every depth up to 32 (LAST = 8) or from 33 to 64 (LAST = 16):
// a batch's instances of a dozen depths, a few hundred blocks each, fill the
// GPU together and finish with one tail instead of one per depth (60 instances
// of z 4 to 32: iteration 80 us against 145 us with a launch per ceil(z / 4),
// part of it from fullest tiles first and from weighing the streams by packed
// elements). The registers are those of the deepest case.
template <int LAST, int MODE>
__global__ void __launch_bounds__(64 * kWaves32) __attribute__((amdgpu_waves_per_eu(LAST <= 8 ? 3 : 2)))
    bld_live_f32_kernel(const LiveTile* __restrict__ tiles, uint32_t lds_bytes) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const LiveTile t = tiles[blockIdx.x];
    switch (LAST - (t.z + 3u) / 4u) {
        case 7: live_step_f32<LAST - 7, MODE>(t, lds_raw, lds_bytes); break;
        case 6: live_step_f32<LAST - 6, MODE>(t, lds_raw, lds_bytes); break;
        case 5: live_step_f32<LAST - 5, MODE>(t, lds_raw, lds_bytes); break;
        case 4: live_step_f32<LAST - 4, MODE>(t, lds_raw, lds_bytes); break;
        case 3: live_step_f32<LAST - 3, MODE>(t, lds_raw, lds_bytes); break;
        case 2: live_step_f32<LAST - 2, MODE>(t, lds_raw, lds_bytes); break;
        case 1: live_step_f32<LAST - 1, MODE>(t, lds_raw, lds_bytes); break;
        default: live_step_f32<LAST, MODE>(t, lds_raw, lds_bytes); break;
    }
}

// FP64, LPF lanes per fiber in the dense pass: a thread evaluates kElems64
// elements at a time of a set of whole fibers; the gradients meet the fiber
// sums through LDS.
template <int LPF, int RW, int MODE, int PSI>
__device__ __forceinline__ void live_step_f64(const LiveTile& t, unsigned char* lds_raw, uint32_t lds_bytes) {
    constexpr uint32_t NT = 64u * kWaves64;
    constexpr uint32_t TW = 64u / LPF;  // tile columns
    constexpr uint32_t U = kElems64;
    const uint32_t tid = threadIdx.x;
    const uint32_t z = t.z, n = t.n;
    const double eps = t.eps;
    const float inv_z = t.inv_z;
    const uint32_t fb = live_fibers64(z, n), ws = odd(z);
    LiveRow* const rt = reinterpret_cast<LiveRow*>(lds_raw);
    double* const pa_l = reinterpret_cast<double*>(lds_raw + live_table_bytes<TW>(t));  // psi(alpha_eph) of the rows
    double* const pA_l = pa_l + t.trows * z;                                            // psi(A)
    double* const gb = pA_l + z;                                            // gradients (exp(Z) later), fiber stride ws
    double* const fs = gb + fb * ws;                                        // per fiber: nom, den, X / S (S_mult, X, norm)
    double* const vals = fs + fb * 3u;
    const uint32_t used = (uint32_t)((unsigned char*)vals - lds_raw);
    const uint32_t kc = live_kc<double>(z, n, lds_bytes - used), vs = live_val_stride<double>(kc);
    const bool whole = kc >= z;

    BNMF_GLOBAL double* const Sc = gmut<double>(t.Sc);
    const BNMF_GLOBAL double* __restrict__ xg = gconst<double>(t.xv);
    const BNMF_GLOBAL uint16_t* __restrict__ fg = gconst<uint16_t>(t.fib);

    const BNMF_GLOBAL double* __restrict__ pb_g = gconst<double>(t.psib);

    // elements e and e + NT of a set of fibers from q0 on
    double s[U], pb[U];
    uint32_t f[U], k[U], rc[U];
    auto load = [&](uint32_t q0, uint32_t e0, uint32_t ne) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t e = min(e0 + u * NT, ne - 1u);
            f[u] = fiber_of(e, inv_z);
            k[u] = e - f[u] * z;
            rc[u] = fg[q0 + f[u]];
            s[u] = Sc[(size_t)q0 * z + e];
        }
    };
    const uint32_t fl = tid / LPF, p = tid % LPF;
    if (n) load(0, tid, min(fb, n) * z);
    {
        const BNMF_GLOBAL double* __restrict__ pa = gconst<double>(t.psia);
        for (uint32_t e = tid; e < t.trows * z; e += NT) pa_l[e] = pa[e];
        if (tid < z) pA_l[tid] = gconst<double>(t.psiA)[tid];
        live_stage_tables<TW, NT>(t, rt);
        if (tid < vs) vals[n * vs + tid] = 0.0;  // the fiber of zeros
    }
    // additive step size 0.1 / (iteration + 1)^0.55 (bld_add.hpp:101-103)
    double eta = 0.0;
    if constexpr (MODE == PASS_ADD) eta = 0.1 / pow((double)*t.iter, 0.55);

    // the dense pass's lane (fiber, p): chunks m0 .. m0 + mcount - 1 of RW
    // elements, visited as m0 + (u ^ xm)
    const uint32_t nchunk = z / RW, cp = (nchunk + LPF - 1u) / LPF;
    const uint32_t xr_mask = nchunk % LPF == 0u ? min(cp & (0u - cp), 4u) - 1u : 0u;
    const uint32_t m0 = min(p * cp, nchunk), mcount = min(cp, nchunk - m0);
    __syncthreads();

    for (uint32_t q0 = 0; q0 < n; q0 += fb) {
        const uint32_t nf = min(fb, n - q0), ne = nf * z;
        // the fiber this thread helps to sum
        const uint32_t ff = fl;
        const bool sums = ff < nf;
        const uint32_t rcs = sums ? fg[q0 + ff] : 0u;
        const double xv = sums ? xg[q0 + ff] : 0.0;
        const auto value = [&](uint32_t q, uint32_t kk) -> double {
            return whole ? vals[q * vs + kk] : Sc[(size_t)q * z + kk];
        };
        // the additive step adds psi(alpha_eph) last (its operation order)
        const auto grad = [&](uint32_t rcu, uint32_t kk, double pbu, double psu) -> double {
            return MODE == PASS_UPDATE ? pbu - psu : ((pbu - psu) - pA_l[kk]) + pa_l[(rcu >> 6) * z + kk];
        };
        bool slow_arg = false;
        for (uint32_t e0 = tid; e0 < ne; e0 += U * NT) {
            if (e0 != tid || q0 != 0u) load(q0, e0, ne);
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) pb[u] = pb_g[(rc[u] & 63u) * z + k[u]];
            double ps[U];
            slow_arg = live_psi<PSI, U>(s, ps) || slow_arg;
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                if (e0 + u * NT < ne) {
                    gb[f[u] * ws + k[u]] = grad(rc[u], k[u], pb[u], ps[u]);
                    if (whole) vals[(q0 + f[u]) * vs + k[u]] = s[u];
                }
            }
        }
        if constexpr (PSI == PSI_F64_EXACT) {
            if (slow_arg) {
                // this thread's elements again, those outside [1, 10)
#pragma unroll 1
                for (uint32_t e = tid; e < ne; e += NT) {
                    const uint32_t fe = fiber_of(e, inv_z), ke = e - fe * z, re = fg[q0 + fe];
                    const double xa = value(q0 + fe, ke) + 1.0;
                    if (!(xa >= 1.0 && xa < 10.0))
                        gb[fe * ws + ke] = grad(re, ke, pb_g[(re & 63u) * z + ke], psi_f64_general(xa));
                }
            }
        }
        __syncthreads();
        // fiber sums by the dense pass's lanes, in their visit order
        const uint32_t xm = (rcs & 63u) & xr_mask;
        const double* const gr = gb + ff * ws;
        auto sval = [&](uint32_t kk) -> double { return value(q0 + ff, kk); };
        if (sums) {
            if constexpr (MODE == PASS_UPDATE) {
                const double* const pr = pa_l + (rcs >> 6) * z;
                const double xr = 1.0 / (xv + eps);
                double sumS = 0.0, nom = 0.0, den = 0.0;
                bool slow = false;
#pragma unroll 2
                for (uint32_t u = 0; u < mcount; ++u) {
                    const uint32_t mm = (m0 + (u ^ xm)) * RW;
#pragma unroll
                    for (uint32_t v = 0; v < RW; ++v) {
                        const double sk = sval(mm + v);
                        bool fast = true;
                        if constexpr (PSI == PSI_F64_EXACT) {
                            const double xa = sk + 1.0;
                            fast = xa >= 1.0 && xa < 10.0;
                            slow = slow || !fast;
                        }
                        sumS += sk;
                        nom += sk * xr * (pA_l[mm + v] - pr[mm + v]);
                        const double dn = den + sk * xr * gr[mm + v];
                        den = fast ? dn : den;
                    }
                }
                // the dense pass adds the denom terms of elements with S + 1
                // outside [1, 10) after the others
                if (slow) {
                    for (uint32_t u = 0; u < mcount; ++u) {
                        const uint32_t mm = (m0 + (u ^ xm)) * RW;
                        for (uint32_t v = 0; v < RW; ++v) {
                            const double sk = sval(mm + v), xa = sk + 1.0;
                            if (!(xa >= 1.0 && xa < 10.0)) den += sk * xr * gr[mm + v];
                        }
                    }
                }
#pragma unroll
                for (int o = 1; o < LPF; o <<= 1) {
                    sumS += __shfl_xor(sumS, o);
                    nom += __shfl_xor(nom, o);
                    den += __shfl_xor(den, o);
                }
                if (p == 0u) {
                    fs[ff * 3u] = nom;
                    fs[ff * 3u + 1u] = den;
                    fs[ff * 3u + 2u] = xv / (sumS + eps);
                }
            } else {
                double smult = 0.0;
#pragma unroll 4
                for (uint32_t u = 0; u < mcount; ++u) {
                    const uint32_t mm = (m0 + (u ^ xm)) * RW;
#pragma unroll
                    for (uint32_t v = 0; v < RW; ++v) smult += sval(mm + v) * gr[mm + v];
                }
#pragma unroll
                for (int o = 1; o < LPF; o <<= 1) smult += __shfl_xor(smult, o);
                if (p == 0u) {
                    fs[ff * 3u] = smult;
                    fs[ff * 3u + 1u] = xv;
                }
            }
        }
        __syncthreads();
        // the new elements: e and e + NT at a time
        auto store = [&](uint32_t e, uint32_t fe, uint32_t ke, double v) {
            Sc[(size_t)q0 * z + e] = v;
            if (whole) vals[(q0 + fe) * vs + ke] = v;
        };
        if constexpr (MODE == PASS_UPDATE) {
#pragma unroll 2
            for (uint32_t e = tid; e < ne; e += NT) {
                const uint32_t fe = fiber_of(e, inv_z), ke = e - fe * z, re = (uint32_t)fg[q0 + fe] >> 6;
                const double nom = fs[fe * 3u], den = fs[fe * 3u + 1u], x_over_s = fs[fe * 3u + 2u];
                const double g = gb[fe * ws + ke], gm = pA_l[ke] - pa_l[re * z + ke], sk = value(q0 + fe, ke);
                store(e, fe, ke, as_stored(sk * div_moderate((g + nom) * x_over_s, gm + den + eps)));
            }
        } else {
            // exp(Z) and its norm along the fiber
#pragma unroll 1
            for (uint32_t e = tid; e < ne; e += NT) {
                const uint32_t fe = fiber_of(e, inv_z), ke = e - fe * z;
                const double smult = fs[fe * 3u], xf = fs[fe * 3u + 1u], g = gb[fe * ws + ke], sk = value(q0 + fe, ke);
                double zk = log(sk) + eps;
                zk += eta * sk * (xf * g - smult);
                gb[fe * ws + ke] = exp(zk);
            }
            __syncthreads();
            if (sums) {
                double norm = 0.0;
#pragma unroll 4
                for (uint32_t u = 0; u < mcount; ++u) {
                    const uint32_t mm = (m0 + (u ^ xm)) * RW;
#pragma unroll
                    for (uint32_t v = 0; v < RW; ++v) norm += gr[mm + v];
                }
#pragma unroll
                for (int o = 1; o < LPF; o <<= 1) norm += __shfl_xor(norm, o);
                if (p == 0u) fs[ff * 3u + 2u] = norm + 1e-50;
            }
            __syncthreads();
            for (uint32_t e = tid; e < ne; e += NT) {
                const uint32_t fe = fiber_of(e, inv_z), ke = e - fe * z;
                store(e, fe, ke, as_stored(fs[fe * 3u + 1u] * (gb[fe * ws + ke] / fs[fe * 3u + 2u])));
            }
        }
        if (q0 + fb < n) __syncthreads();
    }

    for (uint32_t k0 = 0; k0 < z; k0 += kc) {
        const uint32_t kn = min(kc, z - k0);
        __syncthreads();
        if (!whole) {
            // elements k0 .. k0 + kc - 1 of every fiber of the tile
            const float inv_kn = 1.0f / (float)kn;
            for (uint32_t q0 = 0; q0 < n; q0 += 256u) {
                const uint32_t ne = min(256u, n - q0) * kn;
                for (uint32_t e = tid; e < ne; e += NT) {
                    const uint32_t ff = fiber_of(e, inv_kn), kk = e - ff * kn;
                    vals[(q0 + ff) * vs + kk] = Sc[(size_t)(q0 + ff) * z + k0 + kk];
                }
            }
            __syncthreads();
        }
        live_partials<double, TW, NT, 0u>(t, rt, vals, vs, k0, kn);
    }
}

template <int LPF, int MODE, int PSI>
__global__ void __launch_bounds__(64 * kWaves64) __attribute__((amdgpu_waves_per_eu(4)))
    bld_live_f64_kernel(const LiveTile* __restrict__ tiles, uint32_t lds_bytes) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const LiveTile t = tiles[blockIdx.x];
    if (t.z % 2u == 0u)
        live_step_f64<LPF, 2, MODE, PSI>(t, lds_raw, lds_bytes);
    else
        live_step_f64<LPF, 1, MODE, PSI>(t, lds_raw, lds_bytes);
}

// ------------------------------------------------------- packing, unpacking
// Nonempty fibers of each tile, one wavefront per tile; ~0u marks an
// instance the packed form is not for: an X_ij above `most` (near the type's
// range) or not finite.
template <typename T>
__global__ void __launch_bounds__(64)
    bld_live_count_kernel(const BldInst* __restrict__ insts, const PassItem* __restrict__ items, T most,
                          uint32_t* __restrict__ counts) {
    const uint32_t lane = threadIdx.x;
    const PassItem item = items[blockIdx.x];
    const BldInst* __restrict__ I = insts + item.inst;
    const uint32_t i0 = item.ti * I->ti_rows, i1 = min(I->x, i0 + I->ti_rows), y = I->y;
    const uint32_t j0 = item.tj * I->tile_cols, nj = min(I->tile_cols, y - j0);
    const BNMF_GLOBAL T* __restrict__ X = gconst<T>(I->X) + j0;
    uint32_t cnt = 0;
    bool bad = false;
    if (lane < nj)
        for (uint32_t i = i0; i < i1; ++i) {
            const T v = X[(size_t)i * y + lane];
            cnt += v != T(0);
            bad = bad || !(v <= most);
        }
    cnt = wave_sum(cnt);
    if (__builtin_amdgcn_ballot_w64(bad) != 0) cnt = ~0u;
    if (lane == 0) counts[blockIdx.x] = cnt;
}

// The lists of each tile, one wavefront per tile.
template <typename T>
__global__ void __launch_bounds__(64)
    bld_live_build_kernel(const BldInst* __restrict__ insts, LiveTile* __restrict__ tiles) {
    __shared__ unsigned long long mask[kLiveRows];
    const uint32_t lane = threadIdx.x;
    LiveTile* __restrict__ t = tiles + blockIdx.x;
    const BldInst* __restrict__ I = insts + t->inst;
    const uint32_t y = I->y, tw = I->tile_cols, n = t->n, rows = t->trows;
    const uint32_t j0 = t->tj * tw, nj = t->tcols;
    const BNMF_GLOBAL T* __restrict__ X = gconst<T>(I->X) + (size_t)t->ti * I->ti_rows * y + j0;
    for (uint32_t r = 0; r < rows; ++r) {
        const bool on = lane < nj && X[(size_t)r * y + lane] != T(0);
        const unsigned long long m = __builtin_amdgcn_ballot_w64(on);
        if (lane == 0) mask[r] = m;
    }
    __syncthreads();
    // fibers by (column, class, row): a lane per column
    uint32_t total = 0;
    for (uint32_t r = 0; r < rows; ++r) total += (uint32_t)(mask[r] >> lane) & 1u;
    uint32_t pos = total;  // inclusive scan over the columns
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t v = (uint32_t)__shfl_up((int)pos, o);
        if (lane >= (uint32_t)o) pos += v;
    }
    pos -= total;
    BNMF_GLOBAL uint16_t* fib = (BNMF_GLOBAL uint16_t*)t->fib;
    BNMF_GLOBAL T* xv = (BNMF_GLOBAL T*)t->xv;
    BNMF_GLOBAL uint16_t* map = (BNMF_GLOBAL uint16_t*)t->map;
    // FP32: the lanes past the last fiber of its group of 64 read their place
    // and X; whatever their S is stays theirs
    if (sizeof(T) == 4 && n + lane < (n + 63u) / 64u * 64u) {
        fib[n + lane] = 0;
        xv[n + lane] = T(0);
    }
    const uint32_t q0 = pos;
    uint32_t per[kClasses] = {0u, 0u, 0u, 0u};
    for (uint32_t cls = 0; cls < kClasses; ++cls) {
        for (uint32_t r = cls; r < rows; r += kClasses) {
            const bool on = (mask[r] >> lane) & 1u;
            if (lane < tw) map[r * tw + lane] = (uint16_t)(on ? pos : n);
            if (on) {
                fib[pos] = (uint16_t)(r << 6 | lane);
                xv[pos] = X[(size_t)r * y + lane];
                ++pos;
                ++per[cls];
            }
        }
    }
    const unsigned long long cols = __builtin_amdgcn_ballot_w64(total != 0u);
    if (total != 0u) {
        LiveCol d{(uint16_t)q0, (uint16_t)lane, {0, 0, 0, 0}, 0u};
        uint32_t end = 0;
        for (uint32_t c = 0; c < kClasses; ++c) d.end[c] = (uint16_t)(end += per[c]);
        const_cast<LiveCol*>(t->cdesc)[(uint32_t)__popcll(cols & ((1ull << lane) - 1ull))] = d;
    }
    // rows: those with at most four fibers, then the fuller ones. A fiber's
    // place in its row's sum is its column's (part, v, t), part highest:
    // sums split at the highest bit in which neighbours differ, and those
    // of one (part, v) run in order
    const uint32_t pl = 6u - I->zq_log2;
    auto place = [&](uint32_t c) { return (c & ((1u << pl) - 1u)) << 6 | ((c >> pl) & 7u) << 3 | c >> pl >> 3; };
    __threadfence_block();
    __syncthreads();
    LiveRow* rd = const_cast<LiveRow*>(t->rdesc);
    BNMF_GLOBAL uint16_t* smap = (BNMF_GLOBAL uint16_t*)t->smap;
    uint32_t at = 0, few = 0;
    for (uint32_t pass = 0; pass < 2u; ++pass) {
        for (uint32_t r0 = 0; r0 < rows; r0 += 64u) {
            const uint32_t r = r0 + lane;
            const unsigned long long m = r < rows ? mask[r] : 0ull;
            const uint32_t cnt = (uint32_t)__popcll(m);
            const bool take = cnt != 0u && (pass == 0u) == (cnt <= 4u);
            const unsigned long long b = __builtin_amdgcn_ballot_w64(take);
            if (take) {
                LiveRow d{(uint16_t)r, 2, {(uint16_t)n, (uint16_t)n, (uint16_t)n, (uint16_t)n}, 0u};
                if (cnt <= 4u) {
                    uint32_t col[4], key[4];
                    unsigned long long left = m;
                    for (uint32_t u = 0; u < 4u; ++u) {
                        col[u] = left ? (uint32_t)__builtin_ctzll(left) : 0u;
                        key[u] = left ? place(col[u]) : ~0u;
                        left &= left - 1ull;
                    }
                    for (uint32_t u = 0; u < 3u; ++u)  // by place
                        for (uint32_t v = 0; v < 3u - u; ++v)
                            if (key[v] > key[v + 1u]) {
                                const uint32_t tk = key[v], tc = col[v];
                                key[v] = key[v + 1u], col[v] = col[v + 1u];
                                key[v + 1u] = tk, col[v + 1u] = tc;
                            }
                    for (uint32_t u = 0; u < cnt; ++u) d.q[u] = map[r * tw + col[u]];
                    // how far apart neighbours are: the bit at which their
                    // subtrees meet, 0 within one (part, v)
                    auto gap = [&](uint32_t u) {
                        const uint32_t xo = (key[u] ^ key[u + 1u]) >> 3;
                        return xo ? 32u - (uint32_t)__builtin_clz(xo) : 0u;
                    };
                    // a run of equal gaps (one (part, v), in order) leans left
                    if (cnt == 3u) d.shape = gap(0) <= gap(1) ? 0 : 1;
                    if (cnt == 4u) {
                        const uint32_t g0 = gap(0), g1 = gap(1), g2 = gap(2);
                        if (g2 >= g0 && g2 >= g1)
                            d.shape = g0 <= g1 ? 0 : 1;
                        else if (g1 >= g0)
                            d.shape = 2;
                        else
                            d.shape = g1 <= g2 ? 3 : 4;
                    }
                }
                const uint32_t pos = at + (uint32_t)__popcll(b & ((1ull << lane) - 1ull));
                rd[pos] = d;
                if (pass != 0u)
                    for (uint32_t c = 0; c < tw; ++c) smap[(pos - few) * tw + c] = map[r * tw + c];
            }
            at += (uint32_t)__popcll(b);
        }
        if (pass == 0u) few = at;
    }
    if (lane == 0) {
        t->rows4 = (uint16_t)few;
        t->rows = (uint16_t)at;
        t->cols = (uint16_t)__popcll(cols);
    }
}

// Packed S of each tile from its instance's S_src.
template <typename T>
__global__ void __launch_bounds__(256)
    bld_live_gather_kernel(const BldInst* __restrict__ insts, const LiveTile* __restrict__ tiles) {
    const LiveTile* __restrict__ t = tiles + blockIdx.x;
    const BldInst* __restrict__ I = insts + t->inst;
    const uint32_t z = t->z, y = I->y, n = t->n;
    const BNMF_GLOBAL T* __restrict__ src =
        gconst<T>(I->S_src) + ((size_t)t->ti * I->ti_rows * y + t->tj * I->tile_cols) * z;
    BNMF_GLOBAL T* __restrict__ Sc = gmut<T>(t->Sc);
    const BNMF_GLOBAL uint16_t* __restrict__ fib = gconst<uint16_t>(t->fib);
    for (uint32_t e = threadIdx.x; e < n * z; e += 256u) {
        const uint32_t q = e / z, k = e - q * z, rc = fib[q], c = rc & 63u;
        Sc[live_index<T>(t, q, c, k)] = src[((size_t)(rc >> 6) * y + c) * z + k];
    }
}

// S from its packed form: the nonempty fibers, and zeros. Where psi(A), which
// sums every element, is not finite, the last step has made NaN of every
// element (0 * inf), also of the empty fibers'.
template <typename T>
__global__ void __launch_bounds__(256)
    bld_live_scatter_kernel(const BldInst* __restrict__ insts, const LiveTile* __restrict__ tiles) {
    __shared__ uint32_t bad;
    const uint32_t tid = threadIdx.x;
    const LiveTile* __restrict__ t = tiles + blockIdx.x;
    const BldInst* __restrict__ I = insts + t->inst;
    const uint32_t z = t->z, y = I->y, tw = I->tile_cols, n = t->n, rows = t->trows;
    const uint32_t j0 = t->tj * tw, nj = t->tcols;
    const float inv_z = t->inv_z;
    const BNMF_GLOBAL uint16_t* __restrict__ map = gconst<uint16_t>(t->map);
    const BNMF_GLOBAL T* __restrict__ Sc = gconst<T>(t->Sc);
    if (tid == 0) bad = 0u;
    __syncthreads();
    if (tid < z) {
        const T a = gconst<T>(I->psiA)[tid];
        if (!(a - a == T(0))) atomicOr(&bad, 1u);
    }
    __syncthreads();
    const T fill = bad ? T(__builtin_nanf("")) : T(0);
    BNMF_GLOBAL T* __restrict__ dst = gmut<T>(I->S) + ((size_t)t->ti * I->ti_rows * y + j0) * z;
    for (uint32_t r = 0; r < rows; ++r) {
        for (uint32_t e = tid; e < nj * z; e += 256u) {
            const uint32_t c = fiber_of(e, inv_z), q = map[r * tw + c];
            const T v = q < n ? Sc[live_index<T>(t, q, c, e - c * z)] : fill;
            __builtin_nontemporal_store(v, &dst[(size_t)r * y * z + e]);
        }
    }
}

// ---------------------------------------------------------------- launchers
// dynamic LDS of a block whose tile has n fibers, with kc elements of k in the
// value buffer at once
size_t live_lds_need(int dtype, uint32_t z, uint32_t tile_cols, uint32_t rows, uint32_t n, uint32_t kc) {
    if (dtype == 0)
        return live_lds_fixed<float>(z, tile_cols, rows, n) + round16((size_t)(n + 1u) * live_val_stride<float>(kc) * 4);
    return live_lds_fixed<double>(z, tile_cols, rows, n) + round16((size_t)(n + 1u) * live_val_stride<double>(kc) * 8);
}

// packed elements a group of fibers takes, and the fibers of a group
void live_group(int dtype, uint32_t z, uint32_t* elems, uint32_t* fibers) {
    *elems = dtype == 0 ? (z + 3u) / 4u * 256u : z;
    *fibers = dtype == 0 ? 64u : 1u;
}

template <int LAST, int MODE>
static hipError_t live32(uint32_t n, hipStream_t st, const LiveTile* tiles, uint32_t lds) {
    if (n == 0)  // set-up
        return hipFuncSetAttribute(reinterpret_cast<const void*>(bld_live_f32_kernel<LAST, MODE>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
    hipLaunchKernelGGL((bld_live_f32_kernel<LAST, MODE>), dim3(n), dim3(64 * kWaves32), lds, st, tiles, lds);
    return hipGetLastError();
}

template <int LPF, int MODE, int PSI>
static hipError_t live64(uint32_t n, hipStream_t st, const LiveTile* tiles, uint32_t lds) {
    if (n == 0)  // set-up
        return hipFuncSetAttribute(reinterpret_cast<const void*>(bld_live_f64_kernel<LPF, MODE, PSI>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
    hipLaunchKernelGGL((bld_live_f64_kernel<LPF, MODE, PSI>), dim3(n), dim3(64 * kWaves64), lds, st, tiles, lds);
    return hipGetLastError();
}

// Step pass (PASS_UPDATE or PASS_ADD) over the packed fibers of n tiles; big:
// the instances' depths are 33 to 64, else at most 32.
hipError_t launch_pass_live(int dtype, int psi, int mode, bool big, uint32_t n, hipStream_t st, const LiveTile* tiles,
                            uint32_t lds) {
    if (mode == PASS_ADD) {
        if (dtype == 0)
            return big ? live32<16, PASS_ADD>(n, st, tiles, lds) : live32<8, PASS_ADD>(n, st, tiles, lds);
        return big ? live64<4, PASS_ADD, PSI_F64_APPR>(n, st, tiles, lds)
                   : live64<2, PASS_ADD, PSI_F64_APPR>(n, st, tiles, lds);
    }
    if (mode != PASS_UPDATE) return hipErrorInvalidValue;
    if (dtype == 0)
        return big ? live32<16, PASS_UPDATE>(n, st, tiles, lds) : live32<8, PASS_UPDATE>(n, st, tiles, lds);
    if (psi == PSI_F64_APPR)
        return big ? live64<4, PASS_UPDATE, PSI_F64_APPR>(n, st, tiles, lds)
                   : live64<2, PASS_UPDATE, PSI_F64_APPR>(n, st, tiles, lds);
    return big ? live64<4, PASS_UPDATE, PSI_F64_EXACT>(n, st, tiles, lds)
               : live64<2, PASS_UPDATE, PSI_F64_EXACT>(n, st, tiles, lds);
}

hipError_t init_live_attributes() {
    hipError_t e = hipSuccess;
    for (int big = 0; big < 2 && e == hipSuccess; ++big) {
        e = launch_pass_live(0, PSI_F32, PASS_UPDATE, big, 0, nullptr, nullptr, 0);
        if (e == hipSuccess) e = launch_pass_live(0, PSI_F32, PASS_ADD, big, 0, nullptr, nullptr, 0);
        if (e == hipSuccess) e = launch_pass_live(1, PSI_F64_EXACT, PASS_UPDATE, big, 0, nullptr, nullptr, 0);
        if (e == hipSuccess) e = launch_pass_live(1, PSI_F64_APPR, PASS_UPDATE, big, 0, nullptr, nullptr, 0);
        if (e == hipSuccess) e = launch_pass_live(1, PSI_F64_APPR, PASS_ADD, big, 0, nullptr, nullptr, 0);
    }
    return e;
}

hipError_t launch_live_count(int dtype, const BldInst* insts, const PassItem* items, uint32_t n, uint32_t* counts,
                             hipStream_t st) {
    if (dtype == 0)
        hipLaunchKernelGGL(bld_live_count_kernel<float>, dim3(n), dim3(64), 0, st, insts, items, 1e30f, counts);
    else
        hipLaunchKernelGGL(bld_live_count_kernel<double>, dim3(n), dim3(64), 0, st, insts, items, 1e200, counts);
    return hipGetLastError();
}

hipError_t launch_live_build(int dtype, const BldInst* insts, LiveTile* tiles, uint32_t n, hipStream_t st) {
    if (dtype == 0)
        hipLaunchKernelGGL(bld_live_build_kernel<float>, dim3(n), dim3(64), 0, st, insts, tiles);
    else
        hipLaunchKernelGGL(bld_live_build_kernel<double>, dim3(n), dim3(64), 0, st, insts, tiles);
    return hipGetLastError();
}

hipError_t launch_live_gather(int dtype, const BldInst* insts, const LiveTile* tiles, uint32_t n, hipStream_t st) {
    if (dtype == 0)
        hipLaunchKernelGGL(bld_live_gather_kernel<float>, dim3(n), dim3(256), 0, st, insts, tiles);
    else
        hipLaunchKernelGGL(bld_live_gather_kernel<double>, dim3(n), dim3(256), 0, st, insts, tiles);
    return hipGetLastError();
}

hipError_t launch_live_scatter(int dtype, const BldInst* insts, const LiveTile* tiles, uint32_t n, hipStream_t st) {
    if (dtype == 0)
        hipLaunchKernelGGL(bld_live_scatter_kernel<float>, dim3(n), dim3(256), 0, st, insts, tiles);
    else
        hipLaunchKernelGGL(bld_live_scatter_kernel<double>, dim3(n), dim3(256), 0, st, insts, tiles);
    return hipGetLastError();
}

}  // namespace bnmf
