// live.cpp — host side of the packed nonempty fibers (bld_live.hip): which
// instances take them, and the layout of their lists and packed S.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <numeric>
#include <vector>

#include "bnmf_internal.hpp"

namespace bnmf {

namespace {
constexpr size_t kAlign = 256;
size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

// LDS a block takes when its tile needs it, so that two share a CU; a tile
// with more fibers does its partial sums over k in parts, and may take up to
// kLdsMost.
constexpr size_t kLdsWant = 80 * 1024;
constexpr size_t kLdsMost = 150 * 1024;
}  // namespace

size_t LivePlan::scratch_bytes(const std::vector<InstLayout>& lay) {
    size_t tiles = 0;
    for (const InstLayout& L : lay) tiles += (size_t)L.n_ti * L.n_tj;
    return align_up(lay.size() * sizeof(BldInst)) + align_up(tiles * sizeof(PassItem)) + align_up(tiles * 4);
}

// A matrix (rows of y entries) whose sampled entries (some 4096, evenly spaced)
// are mostly nonzero is not worth the count on the device. The spacing has no
// factor in common with y, so that the samples go through all columns: a busy
// column, or a few, must not stand for the matrix.
template <typename T>
static bool mostly_full(const T* X, size_t n, size_t y, double most) {
    size_t step = std::max<size_t>(1, n / 4096);
    while (std::gcd(step, y) != 1) ++step;
    size_t seen = 0, full = 0;
    for (size_t t = 0; t < n; t += step) {
        ++seen;
        full += X[t] != T(0);
    }
    return (double)full > 1.2 * most * (double)seen;
}

// The count on the device, the allocation and the lists take 0.15 ms, and for
// large instances as long as clearing the packed buffers. Plain calls, packed
// and dense: 100x100x17 FP32 at 3 % nonempty 0.80 and 0.82 ms for 8 iterations,
// 1.23 and 1.70 for 32; 64x64x8 at 25 % 0.91 and 0.87 for 16, 1.20 and 1.23 for
// 32; 512x512x32 at 25 % 5.8 and 6.0 for 16, FP64 8.95 and 8.20 for 32, 10.05 and
// 10.11 for 64; 2048x2048x32 at 25 % 51 and 47 for 64, 51 and 56 for 128.
size_t LivePlan::least_iterations(size_t elements) {
    return elements < (1u << 22) ? 24 : elements < (1u << 24) ? 40 : 80;
}

bool LivePlan::worth(int dtype, const void* X, size_t x, size_t y, double most) {
    return !(dtype == BNMF_F32 ? mostly_full(static_cast<const float*>(X), x * y, y, most)
                               : mostly_full(static_cast<const double*>(X), x * y, y, most));
}

// The packed step's cost grows with the share, the dense step's does not. Where
// they meet, from iterations (packed / dense, us) of one or n instances:
//   FP32  z <= 4, where a dense step is as fast as its launches: 128x128x4
//         16.5/15.9 at a share of 0.03, 64 of them 18/19; 8 of 512x512x4 18/30
//         and 31/31 at 0.49
//         z <= 24: 513x861x24 44/44 at 0.49, 64 of 100x100x17 41/39
//         z <= 32: 64 of 40x40x32 24/30 at 0.45; 100x100x32 37/38 at 0.40;
//         256x256x32 39/44 at 0.35, 44/44 at 0.40; 32 of them 107/116, 123/116;
//         16 of 400x400x28 126/140 at 0.40; 1448x1448x32 173/176 at 0.45;
//         2048x2048x32 267/263 at 0.45, 432/265 at 0.49
//         z <= 64: 64 of 32x32x64 50/64 at 0.45; 16 of 128x128x64 115/129 at
//         0.30, 141/130 at 0.35; 16 of 200x200x40 77/83 at 0.35; 512x512x48 59/63
//         at 0.40; 8 of 512x512x64 259/282 at 0.45; 2048x2048x64 439/484 at 0.30,
//         515/485 at 0.35, 911/484 at 0.49
//   FP64  z <= 24: 100x100x17 26/31 at 0.49, 8 of 384x384x24 175/175
//         z <= 32: 256x256x32 30/31 at 0.35, 33/31 at 0.40; 16 of them 183/188,
//         4 of 512x512x32 178/186 and 384x384x32 51/52 at 0.45; 1024x1024x32 159/167 at 0.30, 173/171 at 0.35;
//         2048x2048x32 339/529 at 0.20, 483/546 at 0.25, 565/533 at 0.30
//         z <= 64: 8 of 200x200x64 129/138 at 0.49; 4 of 512x512x64 263/323 at
//         0.35, 334/327 at 0.40; 1024x1024x64 280/305 at 0.30, 335/307 at 0.35
//         additive step: 4 of 512x512x64 571/724 at 0.49, 256x256x32 41/51
// Large deep instances lose soonest: their tiles have more fibers than the LDS
// holds, and the partial sums read S again in parts.
double LivePlan::most_share(int dtype, bool add, size_t x, size_t y, uint32_t z, size_t elements) {
    const size_t xy = x * y;
    if (dtype == BNMF_F32) {
        if (z <= 4) return elements >= 6000000 ? 0.5 : 0.0;
        if (z <= 24) return 0.5;
        if (z <= 32) return xy < (1u << 11) ? 0.5 : xy >= (1u << 20) ? 0.45 : z <= 28 ? 0.42 : 0.37;
        if (xy >= (1u << 17)) return xy < (1u << 21) ? 0.43 : 0.32;
        return xy < (1u << 11) ? 0.5 : z <= 48 ? 0.38 : 0.34;
    }
    if (add || z <= 24) return 0.5;
    if (xy >= (1u << 20)) return xy < (1u << 21) ? 0.32 : 0.26;
    if (z <= 32) return elements < (1u << 22) ? 0.38 : 0.45;
    return xy < (1u << 17) ? 0.5 : 0.38;
}

LivePlan::LivePlan(int dtype, bool add, const std::vector<BldInst>& descs, const std::vector<InstLayout>& lay,
                   const std::vector<bool>& candidate, char* scratch, hipStream_t st,
                   const std::function<void*(size_t, size_t)>& mem)
    : dtype_(dtype), offs_(descs.size()), fibers_(descs.size(), 0), lds_(descs.size(), 0) {
    const size_t es = dtype == BNMF_F32 ? 4 : 8;
    size_t elements = 0;
    for (const InstLayout& L : lay) elements += L.elements();
    // nonempty fibers of every candidate's tiles
    std::vector<PassItem> items;
    for (size_t n = 0; n < descs.size(); ++n) {
        const InstLayout& L = lay[n];
        if (!candidate[n] || L.elements() == 0 || L.z > kFusedZ || L.ti_rows > kLiveRows) continue;
        for (uint32_t ti = 0; ti < L.n_ti; ++ti)
            for (uint32_t tj = 0; tj < L.n_tj; ++tj) items.push_back(PassItem{(uint32_t)n, ti, tj, 0});
    }
    if (items.empty() || items.size() > 0x7fffffffu) return;
    std::vector<uint32_t> counts(items.size());
    {
        char* const it = scratch + align_up(descs.size() * sizeof(BldInst));
        char* const ct = it + align_up(items.size() * sizeof(PassItem));
        BNMF_HIP(hipMemcpyAsync(scratch, descs.data(), descs.size() * sizeof(BldInst), hipMemcpyHostToDevice, st));
        BNMF_HIP(hipMemcpyAsync(it, items.data(), items.size() * sizeof(PassItem), hipMemcpyHostToDevice, st));
        BNMF_HIP(launch_live_count(dtype, reinterpret_cast<const BldInst*>(scratch), reinterpret_cast<const PassItem*>(it),
                                   (uint32_t)items.size(), reinterpret_cast<uint32_t*>(ct), st));
        BNMF_HIP(hipMemcpyAsync(counts.data(), ct, items.size() * 4, hipMemcpyDeviceToHost, st));
        BNMF_HIP(hipStreamSynchronize(st));
    }

    // Which instances pay, alone or among their like; work of those that do and
    // those that do not, for each of the two launches (z <= 32, z <= 64). An
    // instance past its own limit joins the others' launch all the same where
    // they are the larger part of it: that costs an iteration less than a dense
    // launch of its own (19 instances of up to 248x292x32, three of them past
    // their limits: 133 iterations 9.0 against 12.1 ms).
    std::vector<size_t> pays(descs.size(), 0);
    size_t work[2][2] = {};
    for (size_t at = 0; at < items.size();) {
        const size_t n = items[at].inst;
        const InstLayout& L = lay[n];
        const size_t nt = (size_t)L.n_ti * L.n_tj;
        size_t total = 0;
        for (size_t t = 0; t < nt; ++t) total += counts[at + t];
        const double xy = (double)L.x * (double)L.y;
        if ((double)total <= kMostShare * xy) {
            pays[n] = (double)total <= most_share(dtype, add, L.x, L.y, L.z, elements) * xy;
            work[L.z > 32][pays[n]] += total * L.z;
        }
        at += nt;
    }

    // the packed form is extra memory: an instance without room for it runs the
    // dense passes, with the same results
    size_t all = 0;
    for (size_t at = 0; at < items.size();) {
        const size_t n = items[at].inst;
        const InstLayout& L = lay[n];
        const size_t nt = (size_t)L.n_ti * L.n_tj;
        uint32_t ge = 0, gf = 0;
        live_group(dtype, L.z, &ge, &gf);
        uint64_t total = 0, slots = 0;
        uint32_t most = 0;
        bool ok = true;
        std::vector<uint32_t> slot(nt);
        for (size_t t = 0; t < nt && ok; ++t) {
            const uint32_t c = counts[at + t];
            ok = c < 65536u;
            slot[t] = (uint32_t)slots;
            total += c;
            slots += (c + gf - 1) / gf * gf;
            most = std::max(most, c);
        }
        ok = ok && total > 0 && (double)total <= kMostShare * (double)L.x * (double)L.y && slots < (1ull << 31);
        ok = ok && (pays[n] || work[L.z > 32][0] <= work[L.z > 32][1]);
        if (ok) {
            const size_t least = live_lds_need(dtype, L.z, L.tile_cols, L.ti_rows, most, 4);
            const size_t all = live_lds_need(dtype, L.z, L.tile_cols, L.ti_rows, most, (L.z + 3) / 4 * 4);
            ok = least <= kLdsMost;
            if (ok) lds_[n] = (uint32_t)std::max(least, std::min(all, kLdsWant));
        }
        if (ok) {
            size_t off = 0;
            auto take = [&](size_t bytes) {
                const size_t o = off;
                off = align_up(off + bytes);
                return o;
            };
            fibers_[n] = (size_t)total;
            Off& o = offs_[n];
            o.Sc = take((size_t)(slots / gf) * ge * es);
            o.fib = take((size_t)slots * 2);
            o.xv = take((size_t)slots * es);
            o.rdesc = take(nt * L.ti_rows * sizeof(LiveRow));
            o.cdesc = take(nt * L.tile_cols * sizeof(LiveCol));
            o.map = take(nt * L.ti_rows * L.tile_cols * 2);
            o.smap = take(nt * L.ti_rows * L.tile_cols * 2);
            o.base = reinterpret_cast<char*>(all);  // without mem: an offset so far
            if (mem)
                o.base = static_cast<char*>(mem(n, off));
            else
                all += off;
            if (mem && !o.base) {
                lds_[n] = 0;
                at += nt;
                continue;
            }
            o.tile0 = slot_.size();
            slot_.insert(slot_.end(), slot.begin(), slot.end());
            count_.insert(count_.end(), counts.begin() + at, counts.begin() + at + nt);
        }
        at += nt;
    }
    if (mem || slot_.empty()) return;
    const size_t off_tab = all;
    all = align_up(all + slot_.size() * sizeof(LiveTile));
    void* p = nullptr;
    if (hipMalloc(&p, all) != hipSuccess) {
        (void)hipGetLastError();
        std::fill(lds_.begin(), lds_.end(), 0u);
        return;
    }
    buf_.ptr = p;
    buf_.bytes = bytes_ = all;
    for (Off& o : offs_) o.base = buf_.as<char>((size_t)o.base);
    tab_ = buf_.as<LiveTile>(off_tab);
}

uint32_t LivePlan::add_launch(std::vector<PassItem>& items, const std::vector<BldInst>& descs) {
    // fullest tiles first: the launch's tail is then made of its short blocks
    std::stable_sort(items.begin(), items.end(), [&](const PassItem& a, const PassItem& b) {
        auto cost = [&](const PassItem& it) {
            const BldInst& d = descs[it.inst];
            return (uint64_t)count_[offs_[it.inst].tile0 + (size_t)it.ti * d.n_tj + it.tj] * d.z;
        };
        return cost(a) > cost(b);
    });
    const uint32_t first = (uint32_t)tiles_.size();
    const size_t es = dtype_ == BNMF_F32 ? 4 : 8;
    for (const PassItem& it : items) {
        const BldInst& d = descs[it.inst];
        const Off& o = offs_[it.inst];
        const size_t tile = (size_t)it.ti * d.n_tj + it.tj, slot = slot_[o.tile0 + tile];
        const size_t i0 = (size_t)it.ti * d.ti_rows, j0 = (size_t)it.tj * d.tile_cols, z = d.z;
        uint32_t ge = 0, gf = 0;
        live_group(dtype_, d.z, &ge, &gf);
        LiveTile t{};
        t.Sc = o.base + o.Sc + slot / gf * ge * es;
        t.fib = reinterpret_cast<uint16_t*>(o.base + o.fib) + slot;
        t.xv = o.base + o.xv + slot * es;
        t.rdesc = reinterpret_cast<LiveRow*>(o.base + o.rdesc) + tile * d.ti_rows;
        t.cdesc = reinterpret_cast<LiveCol*>(o.base + o.cdesc) + tile * d.tile_cols;
        t.map = reinterpret_cast<uint16_t*>(o.base + o.map) + tile * d.ti_rows * d.tile_cols;
        t.smap = reinterpret_cast<uint16_t*>(o.base + o.smap) + tile * d.ti_rows * d.tile_cols;
        t.psib = static_cast<const char*>(d.psib) + j0 * z * es;
        t.psia = static_cast<const char*>(d.psia) + i0 * z * es;
        t.psiA = d.psiA;
        t.part_ipk = static_cast<char*>(d.part_ipk) + ((size_t)it.tj * d.x + i0) * z * es;
        t.part_pjk = static_cast<char*>(d.part_pjk) + ((size_t)it.ti * d.y + j0) * z * es;
        t.eps = d.eps;
        t.inst = it.inst;
        t.ti = it.ti;
        t.tj = it.tj;
        t.z = d.z;
        t.n = count_[o.tile0 + tile];
        t.trows = (uint16_t)std::min<size_t>(d.ti_rows, d.x - i0);
        t.tcols = (uint16_t)std::min<size_t>(d.tile_cols, d.y - j0);
        t.xs = (uint8_t)(d.rw == 4 ? d.hs : 0);
        t.xm = (uint8_t)(d.rw == 4 ? d.hm : 0);
        t.zq_log2 = d.zq_log2;
        t.inv_z = d.inv_z;
        tiles_.push_back(t);
    }
    return first;
}

void LivePlan::build(const std::vector<BldInst>& descs, const BldInst* insts, hipStream_t st, LiveTile* tab) {
    if (!any()) return;
    const size_t bytes = tiles_.size() * sizeof(LiveTile);
    for (LiveTile& t : tiles_) t.iter = descs[t.inst].iter;
    LiveTile* const dev = tab ? tab : tab_;
    BNMF_HIP(hipMemcpyAsync(dev, tiles_.data(), bytes, hipMemcpyHostToDevice, st));
    BNMF_HIP(launch_live_build(dtype_, insts, dev, (uint32_t)tiles_.size(), st));
    if (tab) BNMF_HIP(hipMemcpyAsync(tiles_.data(), dev, bytes, hipMemcpyDeviceToHost, st));
}

void LivePlan::gather(const BldInst* insts, hipStream_t st) const {
    if (any()) BNMF_HIP(launch_live_gather(dtype_, insts, tiles(), (uint32_t)tiles_.size(), st));
}

void LivePlan::scatter(const BldInst* insts, hipStream_t st) const {
    if (any()) BNMF_HIP(launch_live_scatter(dtype_, insts, tiles(), (uint32_t)tiles_.size(), st));
}

}  // namespace bnmf
