// bld_appr_host.cpp — host side of the approximate BLD solver bld::bld_appr
// (src/bld/bld_appr.hpp:287-372): planning, HBM layout and the captured
// per-iteration launch sequence of the kernels in bld_appr.hip.
//
// The reference materialises S, grad_plus and four x*y*z loops per
// half-step on the host. Here the factors nu (x*z) and mu (z*y) stay on the
// device, S is formed per fiber inside each pass from X and the factors, and
// an iteration is, per half-step: sums pass, prep + psi(A) (shared with the
// multiplicative solver), step pass, factor update — captured once into a
// hipGraph and replayed.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "bnmf_internal.hpp"

namespace bnmf {

namespace {
constexpr size_t kAlign = 256;
size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }
uint32_t ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Rows per tile: enough tiles to give an instance's launch about one block
// per 2048 fibers, between 16 and 512 blocks, with tiles of 4 to 64 rows.
// The plan depends on the shape only, so an instance gives the same bits
// alone and batched. Measured on MI355X: 1024x1024x32 alone, 512 blocks
// (32-row tiles) 314 us per iteration against 518 us at 256 or fewer, and
// 2048 or 8192 blocks slower again (more tiles add column partials that the
// factor and prep kernels must reduce); the 256-instance batch (x, y up to
// 512), 3524 us per iteration at 512 blocks per instance, 2706 us at 128,
// 2566 us at 16 (the factor kernel's partial sums over row tiles dominate
// once every instance has many short tiles). BNMF_APPR_BLOCKS sets a fixed
// target for every instance instead, for experiments.
uint32_t appr_ti_rows(uint32_t x, uint32_t y, uint32_t n_tj) {
    static const uint32_t fixed_target = [] {
        const char* e = std::getenv("BNMF_APPR_BLOCKS");
        const long v = e ? std::strtol(e, nullptr, 10) : 0L;
        return v > 0 ? (uint32_t)std::min<long>(v, 1 << 20) : 0u;
    }();
    const uint64_t by_size = ((uint64_t)x * y) / 2048u;
    const uint32_t target =
        fixed_target ? fixed_target : (uint32_t)std::min<uint64_t>(std::max<uint64_t>(by_size, 16u), 512u);
    const uint32_t want = std::max<uint32_t>(1, target / std::max<uint32_t>(n_tj, 1));
    uint32_t ti = ceil_div(x, want);
    ti = (ti + 3) / 4 * 4;
    return std::min<uint32_t>(std::max<uint32_t>(ti, 4), 64);
}

uint32_t zq_of(uint32_t z) {
    uint32_t q = 1;
    while (q < z) q <<= 1;
    return q;
}
// Wavefronts per list: four once the mean list keeps one busy for more than a
// dozen entries per group.
uint32_t list_waves(size_t entries, uint32_t lists, uint32_t z) {
    return (double)entries * zq_of(z) > 768.0 * lists ? 4u : 1u;
}
// Largest share of nonempty entries at which an FP64 instance runs over them
// (bld_appr_live.hip), where lanes past z count as work too. Measured per
// iteration, lists against dense passes: 1024x1024x32 131 us against 975 at a
// share of 0.1 and 856 against 1000 full; 64 of 200x200x17 (17 of 32 lanes in
// use) 1072 against 1520 at 0.5 and 1865 against 1529 full; 64 of 400x40x10, 282
// against 405 and 459 against 419. An instance so small that its launches are
// all latency takes the lists always (8x10x3: 24 against 40).
double live_share(size_t x, size_t y, uint32_t z) { return x * y * zq_of(z) <= 8192 ? 1.0 : 0.9 * z / zq_of(z); }
// Longest list (entries times lanes per entry) that one block may be left to
// walk where the dense passes would spread it over the chip: 20000x100x20, 633 us
// against 1725 at lists of 2000; at 6000 both would take about 1750.
double list_budget(double elements) { return std::max(65536.0, elements / 256.0); }

bool within(const double* p, size_t n, double lo, double hi) {
    for (size_t t = 0; t < n; ++t)
        if (!(p[t] >= lo && p[t] <= hi)) return false;
    return true;
}
}  // namespace

// May the instance run over its nonempty entries only? An empty one then has
// to contribute exactly 0, so the gradients it multiplies must be finite:
// parameters, eps and starting factors of ordinary size. Whatever else the
// caller gives takes the dense passes, and so does FP32: its solves carry
// rounding errors of up to 1e-5 after 200 iterations, which sums taken in
// another order, or in double, would replace by other results.
bool ApprBatch::live_candidate(const ApprSpec& s, double eps) const {
    const size_t x = s.x, y = s.y, z = s.z;
    if (dtype_ != BNMF_F64 || z > kFusedZ || x * y == 0 || x * y > 0xffffffffull) return false;
    if (!(eps >= 1e-200 && eps <= 1.0)) return false;
    if (!within(s.alpha, x, 1e-6, 1e30) || !within(s.beta, z, 1e-6, 1e30)) return false;
    auto tame = [](const void* p, size_t n) { return !p || within(static_cast<const double*>(p), n, 0.0, 1e100); };
    return tame(s.nu0, x * z) && tame(s.mu0, z * y) && LivePlan::worth(dtype_, s.X, x, y, live_share(x, y, s.z));
}

// The lists of the instances that are sparse enough, in one allocation; none
// if it cannot be had. counts: (x + y) words per candidate, in order.
void ApprBatch::plan_live(uint32_t* counts, std::vector<ApprInst>& ai, std::vector<BldInst>& bi) {
    char* const base = arena_.as<char>();
    size_t total = 0;
    for (const L_& l : lay_)
        if (l.live) {
            BNMF_HIP(launch_appr_count(arena_.as<double>(l.off_X), l.x, l.y, counts + total, nullptr));
            total += (size_t)l.x + l.y;
        }
    if (total == 0) return;
    std::vector<uint32_t> cnt(total);
    BNMF_HIP(hipMemcpy(cnt.data(), counts, total * 4, hipMemcpyDeviceToHost));

    std::vector<uint32_t> ptr;  // per instance: x + 1 row offsets, y + 1 column offsets
    std::vector<size_t> off_ptr(lay_.size()), off_ent(lay_.size());
    size_t at = 0, ent_bytes = 0;
    for (size_t n = 0; n < lay_.size(); ++n) {
        L_& l = lay_[n];
        if (!l.live) continue;
        const uint32_t* const c = cnt.data() + at;
        at += (size_t)l.x + l.y;
        size_t entries = 0;
        uint32_t longest = 0;
        bool bad = false;
        for (size_t i = 0; i < (size_t)l.x + l.y; ++i) {
            bad = bad || c[i] == ~0u;
            longest = std::max(longest, c[i]);
            if (i < l.x) entries += c[i];
        }
        l.live = !bad && (double)entries <= live_share(l.x, l.y, l.z) * (double)l.x * (double)l.y &&
                 (double)longest * zq_of(l.z) <= list_budget((double)l.x * l.y * l.z);
        if (!l.live) continue;
        l.entries = entries;
        off_ptr[n] = ptr.size();
        uint32_t sum = 0;
        for (size_t i = 0; i < l.x; ++i) {
            ptr.push_back(sum);
            sum += c[i];
        }
        ptr.push_back(sum);
        sum = 0;
        for (size_t j = 0; j < l.y; ++j) {
            ptr.push_back(sum);
            sum += c[l.x + j];
        }
        ptr.push_back(sum);
        off_ent[n] = ent_bytes;
        ent_bytes += 2 * (align_up(entries * 4 + 4) + align_up(entries * 8 + 8));
    }
    if (ptr.empty()) return;
    const size_t ptr_bytes = align_up(ptr.size() * 4);
    void* p = nullptr;
    if (hipMalloc(&p, ptr_bytes + ent_bytes) != hipSuccess) {
        (void)hipGetLastError();
        for (L_& l : lay_) l.live = false;
        return;
    }
    lists_.ptr = p;
    lists_.bytes = ptr_bytes + ent_bytes;
    BNMF_HIP(hipMemcpy(p, ptr.data(), ptr.size() * 4, hipMemcpyHostToDevice));
    for (size_t n = 0; n < lay_.size(); ++n) {
        const L_& l = lay_[n];
        if (!l.live) continue;
        const size_t oi = align_up(l.entries * 4 + 4), ox = align_up(l.entries * 8 + 8);
        const uint32_t* const rptr = lists_.as<uint32_t>(off_ptr[n] * 4);
        const uint32_t* const cptr = rptr + l.x + 1;
        char* const e = lists_.as<char>(ptr_bytes + off_ent[n]);
        uint32_t* const ridx = reinterpret_cast<uint32_t*>(e);
        uint32_t* const cidx = reinterpret_cast<uint32_t*>(e + oi);
        double* const rxv = reinterpret_cast<double*>(e + 2 * oi);
        double* const cxv = reinterpret_cast<double*>(e + 2 * oi + ox);
        BNMF_HIP(launch_appr_fill(arena_.as<double>(l.off_X), l.x, l.y, rptr, ridx, rxv, cptr, cidx, cxv, nullptr));
        ApprInst& a = ai[n];
        a.rptr = rptr;
        a.ridx = ridx;
        a.rxv = rxv;
        a.cptr = cptr;
        a.cidx = cidx;
        a.cxv = cxv;
        // the dense passes' second partials are free: y*z and x*z at least
        a.muT = base + l.off_pjk2;
        a.partA = base + l.off_ipk2;
        a.nA = ceil_div(l.x, 4u / list_waves(l.entries, l.x, l.z));
        zmax_live_ = std::max(zmax_live_, l.z);
        // left out of the dense instances' psi(A)
        bi[n].x = 0;
    }
    BNMF_HIP(hipStreamSynchronize(nullptr));
}

ApprBatch::ApprBatch(int dtype, double eps, const std::vector<ApprSpec>& specs)
    : dtype_(dtype), psi_(dtype == BNMF_F32 ? PSIM_F32 : PSIM_F64_APPR), es_(dtype == BNMF_F32 ? 4 : 8) {
    ensure_runtime();
    for (const ApprSpec& s : specs) BNMF_REQUIRE(s.z >= 1, "bld_appr needs z >= 1");
    // where memory runs out, without the lists: the dense passes, which sum
    // in another order (last digits)
    for (bool lists : {true, false}) {
        try {
            plan(specs, eps, lists);
            return;
        } catch (const Error& e) {
            release();
            if (e.status != BNMF_ERR_OUT_OF_MEMORY || !lists) throw;
            (void)hipGetLastError();
        } catch (...) {
            release();
            throw;
        }
    }
}

void ApprBatch::plan(const std::vector<ApprSpec>& specs, double eps, bool lists) {
    const int dtype = dtype_;
    // layouts
    size_t total = 0, n_counts = 0;
    for (const ApprSpec& s : specs) {
        L_ l{};
        l.x = s.x;
        l.y = s.y;
        l.z = s.z;
        // fibers deeper than 64 take the wavefront-per-fiber pass on
        // kWideRows x kWideCols tiles
        const bool deep = s.z > kFusedZ;
        l.n_tj = ceil_div(s.y, deep ? kWideCols : kTileCols);
        l.ti_rows = deep ? kWideRows : appr_ti_rows(s.x, s.y, l.n_tj);
        l.n_ti = ceil_div(s.x, l.ti_rows);
        l.nA = ceil_div(s.x, kPrepRows);
        l.n_cj = ceil_div(s.y, kPrepCols);
        size_t off = total;
        auto take = [&](size_t n) {
            const size_t o = off;
            off = align_up(off + std::max<size_t>(n, 1));
            return o;
        };
        const size_t x = s.x, y = s.y, z = s.z;
        l.off_X = take(x * y * es_);
        l.off_nu = take(x * z * es_);
        l.off_mu = take(z * y * es_);
        l.off_nu0 = take(x * z * es_);
        l.off_mu0 = take(z * y * es_);
        l.off_alpha = take(x * 8);
        l.off_beta = take(z * 8);
        l.off_psib = take(y * z * es_);
        l.off_psia = take(x * z * es_);
        l.off_partA = take((size_t)l.nA * z * es_);
        l.off_psiA = take(z * es_);
        l.off_pjk = take((size_t)l.n_ti * y * z * es_);
        l.off_pjk2 = take((size_t)l.n_ti * y * z * es_);
        l.off_ipk = take((size_t)l.n_tj * x * z * es_);
        l.off_ipk2 = take((size_t)l.n_tj * x * z * es_);
        l.off_S = take(x * y * z * es_);
        l.live = lists && live_candidate(s, eps);
        if (l.live) n_counts += x + y;
        total = off;
        lay_.push_back(l);
    }
    arena_ = DeviceBuffer(std::max<size_t>(total + n_counts * 4, kAlign));

    // uploads; nu0 / mu0 drawn when not given: rows of nu and columns of mu
    // are Dirichlet(1_z) (bld_appr.hpp:302-318), from the init_S stream of
    // `seed` over x + y unit fibers (rows of nu first, then columns of mu)
    std::vector<ApprInst> ai;
    std::vector<BldInst> bi;
    std::vector<char> tmp;
    for (size_t n = 0; n < specs.size(); ++n) {
        const ApprSpec& s = specs[n];
        const L_& l = lay_[n];
        char* b = arena_.as<char>();
        const size_t x = s.x, y = s.y, z = s.z;
        if (x * y) BNMF_HIP(hipMemcpy(b + l.off_X, s.X, x * y * es_, hipMemcpyHostToDevice));
        if (x) BNMF_HIP(hipMemcpy(b + l.off_alpha, s.alpha, x * 8, hipMemcpyHostToDevice));
        BNMF_HIP(hipMemcpy(b + l.off_beta, s.beta, z * 8, hipMemcpyHostToDevice));
        const void* nu0 = s.nu0;
        const void* mu0 = s.mu0;
        std::vector<char> dn, dm;
        if ((!nu0 || !mu0) && x + y > 0) {
            tmp.resize((x + y) * z * es_);
            if (dtype == BNMF_F32) {
                std::vector<float> ones(x + y, 1.0f);
                init_S<float>(s.seed, ones.data(), x + y, 1, z, reinterpret_cast<float*>(tmp.data()));
            } else {
                std::vector<double> ones(x + y, 1.0);
                init_S<double>(s.seed, ones.data(), x + y, 1, z, reinterpret_cast<double*>(tmp.data()));
            }
            if (!nu0) {
                dn.assign(tmp.data(), tmp.data() + x * z * es_);
                nu0 = dn.data();
            }
            if (!mu0) {
                // columns of mu: transpose the y rows drawn after nu's
                dm.resize(z * y * es_);
                for (size_t j = 0; j < y; ++j)
                    for (size_t k = 0; k < z; ++k)
                        std::memcpy(dm.data() + (k * y + j) * es_, tmp.data() + ((x + j) * z + k) * es_, es_);
                mu0 = dm.data();
            }
        }
        if (x * z) BNMF_HIP(hipMemcpy(b + l.off_nu0, nu0, x * z * es_, hipMemcpyHostToDevice));
        if (z * y) BNMF_HIP(hipMemcpy(b + l.off_mu0, mu0, z * y * es_, hipMemcpyHostToDevice));

        ApprInst a{};
        a.X = b + l.off_X;
        a.nu = b + l.off_nu;
        a.mu = b + l.off_mu;
        a.psib = b + l.off_psib;
        a.psia = b + l.off_psia;
        a.psiA = b + l.off_psiA;
        a.part_pjk = b + l.off_pjk;
        a.part_ipk = b + l.off_ipk;
        a.part_pjk2 = b + l.off_pjk2;
        a.part_ipk2 = b + l.off_ipk2;
        a.S = b + l.off_S;
        a.eps = eps;
        a.x = s.x;
        a.y = s.y;
        a.z = s.z;
        a.ti_rows = l.ti_rows;
        a.n_ti = l.n_ti;
        a.n_tj = l.n_tj;
        uint32_t zq = 1, lg = 0;
        while (zq < s.z) {
            zq <<= 1;
            ++lg;
        }
        a.zq = zq;
        a.zq_log2 = lg;
        a.alpha = reinterpret_cast<const double*>(b + l.off_alpha);
        a.beta = reinterpret_cast<const double*>(b + l.off_beta);
        ai.push_back(a);

        // the prep view of the same buffers
        BldInst d{};
        d.alpha = reinterpret_cast<const double*>(b + l.off_alpha);
        d.beta = reinterpret_cast<const double*>(b + l.off_beta);
        d.psib = b + l.off_psib;
        d.psia = b + l.off_psia;
        d.partA = b + l.off_partA;
        d.psiA = b + l.off_psiA;
        d.part_pjk = b + l.off_pjk;
        d.part_ipk = b + l.off_ipk;
        d.eps = eps;
        d.inv_z = 1.0f / (float)s.z;
        d.x = s.x;
        d.y = s.y;
        d.z = s.z;
        d.n_ti = l.n_ti;
        d.n_tj = l.n_tj;
        d.nA = l.nA;
        d.n_cj = l.n_cj;
        d.zq = zq;
        d.zq_log2 = lg;
        bi.push_back(d);
    }
    plan_live(arena_.as<uint32_t>(total), ai, bi);

    // work lists: pass items by z bucket, prep items, factor items
    std::map<uint32_t, std::vector<PassItem>> by_zb;
    std::map<uint32_t, uint32_t> zmax;
    std::vector<PrepItem> prep;
    std::vector<PassItem> fnu, fmu, lrow, lcol, lall;
    for (size_t n = 0; n < specs.size(); ++n) {
        const L_& l = lay_[n];
        if ((size_t)l.x * l.y == 0) continue;
        if (l.live) {
            const uint32_t wr = list_waves(l.entries, l.x, l.z), wc = list_waves(l.entries, l.y, l.z);
            for (uint32_t i = 0; i < l.x; i += 4u / wr) lrow.push_back(PassItem{(uint32_t)n, i, 0, wr});
            for (uint32_t j = 0; j < l.y; j += 4u / wc) lcol.push_back(PassItem{(uint32_t)n, j, 1, wc});
            continue;
        }
        const uint32_t zb = z_bucket(l.z);
        auto& v = by_zb[zb];
        for (uint32_t ti = 0; ti < l.n_ti; ++ti)
            for (uint32_t tj = 0; tj < l.n_tj; ++tj) v.push_back(PassItem{(uint32_t)n, ti, tj, 0});
        zmax[zb] = std::max(zmax[zb], l.z);
        zmax_dense_ = std::max(zmax_dense_, l.z);
        for (uint32_t c = 0; c < l.n_cj; ++c) prep.push_back(PrepItem{(uint32_t)n, 0, c, 0});
        for (uint32_t c = 0; c < l.nA; ++c) prep.push_back(PrepItem{(uint32_t)n, 1, c, 0});
        // factor updates: four rows (columns) per item, one per wavefront
        for (uint32_t c = 0; c < ceil_div(l.x, 4); ++c) fnu.push_back(PassItem{(uint32_t)n, c, 0, 0});
        for (uint32_t c = 0; c < ceil_div(l.y, 4); ++c) fmu.push_back(PassItem{(uint32_t)n, c, 0, 0});
    }
    lall = lrow;
    lall.insert(lall.end(), lcol.begin(), lcol.end());
    n_live_ = (uint32_t)lall.size();
    n_lrow_ = (uint32_t)lrow.size();
    n_lcol_ = (uint32_t)lcol.size();
    size_t moff = 0;
    auto mtake = [&](size_t nbytes) {
        const size_t o = moff;
        moff = align_up(moff + std::max<size_t>(nbytes, 4));
        return o;
    };
    off_live_ = mtake(lall.size() * sizeof(PassItem));
    off_lrow_ = mtake(lrow.size() * sizeof(PassItem));
    off_lcol_ = mtake(lcol.size() * sizeof(PassItem));
    off_ai_ = mtake(ai.size() * sizeof(ApprInst));
    off_bi_ = mtake(bi.size() * sizeof(BldInst));
    for (auto& kv : by_zb) {
        Group g;
        g.zb = kv.first;
        g.zmax = zmax[kv.first];
        g.n_items = (uint32_t)kv.second.size();
        g.off_items = mtake(kv.second.size() * sizeof(PassItem));
        g.off_count = mtake(4);
        groups_.push_back(g);
    }
    n_prep_ = (uint32_t)prep.size();
    off_prep_ = mtake(prep.size() * sizeof(PrepItem));
    off_prep_count_ = mtake(4);
    n_fnu_ = (uint32_t)fnu.size();
    n_fmu_ = (uint32_t)fmu.size();
    off_fnu_ = mtake(fnu.size() * sizeof(PassItem));
    off_fnu_count_ = mtake(4);
    off_fmu_ = mtake(fmu.size() * sizeof(PassItem));
    off_fmu_count_ = mtake(4);
    meta_ = DeviceBuffer(std::max<size_t>(moff, kAlign));
    char* m = meta_.as<char>();
    auto put = [&](size_t off, const void* src, size_t nbytes) {
        if (nbytes) BNMF_HIP(hipMemcpy(m + off, src, nbytes, hipMemcpyHostToDevice));
    };
    put(off_ai_, ai.data(), ai.size() * sizeof(ApprInst));
    put(off_bi_, bi.data(), bi.size() * sizeof(BldInst));
    {
        size_t gi = 0;
        for (auto& kv : by_zb) {
            const Group& g = groups_[gi++];
            put(g.off_items, kv.second.data(), kv.second.size() * sizeof(PassItem));
            put(g.off_count, &g.n_items, 4);
        }
    }
    put(off_live_, lall.data(), lall.size() * sizeof(PassItem));
    put(off_lrow_, lrow.data(), lrow.size() * sizeof(PassItem));
    put(off_lcol_, lcol.data(), lcol.size() * sizeof(PassItem));
    put(off_prep_, prep.data(), prep.size() * sizeof(PrepItem));
    put(off_prep_count_, &n_prep_, 4);
    put(off_fnu_, fnu.data(), fnu.size() * sizeof(PassItem));
    put(off_fnu_count_, &n_fnu_, 4);
    put(off_fmu_, fmu.data(), fmu.size() * sizeof(PassItem));
    put(off_fmu_count_, &n_fmu_, 4);
    BNMF_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
}

ApprBatch::~ApprBatch() { release(); }

void ApprBatch::release() {
    if (stream_) (void)hipStreamSynchronize(stream_);
    for (hipGraphExec_t& g : graphs_) {
        if (g) (void)hipGraphExecDestroy(g);
        g = nullptr;
    }
    if (stream_) (void)hipStreamDestroy(stream_);
    if (side_) (void)hipStreamDestroy(side_);
    if (fork_) (void)hipEventDestroy(fork_);
    if (join_) (void)hipEventDestroy(join_);
    stream_ = side_ = nullptr;
    fork_ = join_ = nullptr;
    lists_ = DeviceBuffer();
    meta_ = DeviceBuffer();
    arena_ = DeviceBuffer();
    lay_.clear();
    groups_.clear();
    zmax_dense_ = zmax_live_ = 0;
}

void ApprBatch::enqueue_dense() {
    char* m = meta_.as<char>();
    const ApprInst* ai = reinterpret_cast<const ApprInst*>(m + off_ai_);
    const int dt = dtype_ == BNMF_F32 ? 0 : 1;
    auto passes = [&](int mode) {
        for (const Group& g : groups_)
            BNMF_HIP(launch_appr_pass(dt, mode, (int)g.zb, dim3(g.n_items), stream_, ai,
                                      reinterpret_cast<const PassItem*>(m + g.off_items),
                                      reinterpret_cast<const uint32_t*>(m + g.off_count), g.zmax));
    };
    for (int half = 0; half < 2; ++half) {
        passes(0);
        BNMF_HIP(launch_prep(dtype_, psi_, false, dim3(n_prep_), stream_, reinterpret_cast<const BldInst*>(m + off_bi_),
                             reinterpret_cast<const PrepItem*>(m + off_prep_),
                             reinterpret_cast<const uint32_t*>(m + off_prep_count_), (uint32_t)lay_.size(), zmax_dense_));
        passes(1 + half);
        BNMF_HIP(launch_appr_factor(dt, half, dim3(half == 0 ? n_fnu_ : n_fmu_), stream_, ai,
                                    reinterpret_cast<const PassItem*>(m + (half == 0 ? off_fnu_ : off_fmu_)),
                                    reinterpret_cast<const uint32_t*>(m + (half == 0 ? off_fnu_count_ : off_fmu_count_))));
    }
}

void ApprBatch::enqueue_live(hipStream_t st) {
    char* m = meta_.as<char>();
    const ApprInst* ai = reinterpret_cast<const ApprInst*>(m + off_ai_);
    for (int half = 0; half < 2; ++half) {
        BNMF_HIP(launch_appr_live(0, n_live_, st, ai, reinterpret_cast<const PassItem*>(m + off_live_)));
        BNMF_HIP(launch_appr_psiA((uint32_t)lay_.size(), zmax_live_, st, ai));
        BNMF_HIP(launch_appr_live(1, half == 0 ? n_lrow_ : n_lcol_, st, ai,
                                  reinterpret_cast<const PassItem*>(m + (half == 0 ? off_lrow_ : off_lcol_))));
    }
}

// 1 << level iterations. Dense and listed instances have nothing in common, so
// a batch with both runs them side by side, as two branches of the graph.
hipGraphExec_t ApprBatch::graph_of(int level) {
    if (graphs_[level]) return graphs_[level];
    hipGraph_t g = nullptr;
    const bool both = n_prep_ > 0 && n_live_ > 0;
    if (both && !side_) {
        BNMF_HIP(hipStreamCreateWithFlags(&side_, hipStreamNonBlocking));
        BNMF_HIP(hipEventCreateWithFlags(&fork_, hipEventDisableTiming));
        BNMF_HIP(hipEventCreateWithFlags(&join_, hipEventDisableTiming));
    }
    BNMF_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
    try {
        if (both) {
            BNMF_HIP(hipEventRecord(fork_, stream_));
            BNMF_HIP(hipStreamWaitEvent(side_, fork_, 0));
        }
        for (int t = 0; t < 1 << level; ++t) {
            if (n_live_ > 0) enqueue_live(both ? side_ : stream_);
            if (n_prep_ > 0) enqueue_dense();
        }
        if (both) {
            BNMF_HIP(hipEventRecord(join_, side_));
            BNMF_HIP(hipStreamWaitEvent(stream_, join_, 0));
        }
    } catch (...) {
        (void)hipStreamEndCapture(stream_, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
    }
    BNMF_HIP(hipStreamEndCapture(stream_, &g));
    hipError_t e = hipGraphInstantiate(&graphs_[level], g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    BNMF_HIP(e);
    return graphs_[level];
}

// iterations from the largest graphs down
void ApprBatch::replay(size_t iters) {
    for (int l = kGraphLevels - 1; l >= 0; --l)
        for (; iters >= (size_t)1 << l; iters -= (size_t)1 << l) BNMF_HIP(hipGraphLaunch(graph_of(l), stream_));
}

void ApprBatch::solve_async(size_t iters) {
    char* b = arena_.as<char>();
    for (const L_& l : lay_) {
        const size_t xz = (size_t)l.x * l.z, zy = (size_t)l.z * l.y;
        if (xz) BNMF_HIP(hipMemcpyAsync(b + l.off_nu, b + l.off_nu0, xz * es_, hipMemcpyDeviceToDevice, stream_));
        if (zy) BNMF_HIP(hipMemcpyAsync(b + l.off_mu, b + l.off_mu0, zy * es_, hipMemcpyDeviceToDevice, stream_));
    }
    if (n_prep_ + n_live_ == 0 || iters == 0) return;
    load_factors();
    replay(iters);
    store_factors();
}

// mu of the instances that run over lists is transposed during a solve.
void ApprBatch::load_factors() {
    for (const L_& l : lay_)
        if (l.live)
            BNMF_HIP(launch_appr_transpose(arena_.as<double>(l.off_pjk2), arena_.as<double>(l.off_mu), l.y, l.z, stream_));
}

void ApprBatch::store_factors() {
    for (const L_& l : lay_)
        if (l.live)
            BNMF_HIP(launch_appr_transpose(arena_.as<double>(l.off_mu), arena_.as<double>(l.off_pjk2), l.z, l.y, stream_));
}

void ApprBatch::synchronize() { BNMF_HIP(hipStreamSynchronize(stream_)); }

void ApprBatch::get(size_t idx, void* S, void* nu, void* mu) {
    BNMF_REQUIRE(idx < lay_.size(), "instance index out of range");
    const L_& l = lay_[idx];
    char* b = arena_.as<char>();
    const size_t xy = (size_t)l.x * l.y;
    if (S && xy) {
        const ApprInst* ai = reinterpret_cast<const ApprInst*>(meta_.as<char>() + off_ai_) + idx;
        BNMF_HIP(launch_appr_S(dtype_ == BNMF_F32 ? 0 : 1, ai, xy, stream_));
    }
    BNMF_HIP(hipStreamSynchronize(stream_));
    if (S && xy) stage_.copy(S, b + l.off_S, xy * l.z * es_, stream_);
    if (nu && l.x) BNMF_HIP(hipMemcpy(nu, b + l.off_nu, (size_t)l.x * l.z * es_, hipMemcpyDeviceToHost));
    if (mu && l.y) BNMF_HIP(hipMemcpy(mu, b + l.off_mu, (size_t)l.z * l.y * es_, hipMemcpyDeviceToHost));
}

double ApprBatch::time_iteration(int reps) {
    BNMF_REQUIRE(reps > 0, "reps must be positive");
    if (n_prep_ + n_live_ == 0) return 0.0;
    load_factors();
    hipGraphExec_t graph = graph_of(0);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    BNMF_HIP(hipEventCreate(&e0));
    hipError_t err = hipEventCreate(&e1);
    if (err != hipSuccess) {
        (void)hipEventDestroy(e0);
        BNMF_HIP(err);
    }
    float ms = 0.f;
    err = hipGraphLaunch(graph, stream_);
    if (err == hipSuccess) err = hipEventRecord(e0, stream_);
    for (int r = 0; r < reps && err == hipSuccess; ++r) err = hipGraphLaunch(graph, stream_);
    if (err == hipSuccess) err = hipEventRecord(e1, stream_);
    if (err == hipSuccess) err = hipEventSynchronize(e1);
    if (err == hipSuccess) err = hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    BNMF_HIP(err);
    store_factors();
    return (double)ms / reps;
}

size_t ApprBatch::device_bytes() const { return arena_.bytes + meta_.bytes + lists_.bytes; }

}  // namespace bnmf
