// bnmf_internal.hpp — host-side internals shared by the library sources.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <mutex>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/bnmf_hip.h"
#include "bld_types.hpp"

namespace bnmf {

// ------------------------------------------------------------------ errors
struct Error : std::runtime_error {
    bnmf_status status;
    Error(bnmf_status s, const std::string& m) : std::runtime_error(m), status(s) {}
};
void set_last_error(const std::string& msg);
void clear_last_error();

#define BNMF_HIP(call)                                                                  \
    do {                                                                                \
        hipError_t bnmf_e_ = (call);                                                    \
        if (bnmf_e_ != hipSuccess)                                                      \
            throw ::bnmf::Error(bnmf_e_ == hipErrorOutOfMemory ? BNMF_ERR_OUT_OF_MEMORY \
                                                               : BNMF_ERR_DEVICE,       \
                                std::string(#call) + ": " + hipGetErrorString(bnmf_e_)); \
    } while (0)

#define BNMF_REQUIRE(cond, msg)                                               \
    do {                                                                      \
        if (!(cond)) throw ::bnmf::Error(BNMF_ERR_INVALID_ARGUMENT, (msg)); \
    } while (0)

// ----------------------------------------------------------------- kernels
enum : int { MODE_UPDATE = 0, MODE_SUMS = 1, MODE_SCORE = 2, MODE_ADD = 3 };
enum : int { PSIM_F32 = 0, PSIM_F64_EXACT = 1, PSIM_F64_APPR = 2 };
hipError_t launch_pass(int dtype, int psi, int mode, int zb, int rw, dim3 grid, hipStream_t st,
                       const BldInst* insts, const PassItem* items, const uint32_t* n_items,
                       uint32_t zmax);
void read_layout(int dtype, uint32_t z, uint32_t* rw, uint32_t* hs, uint32_t* hm);
// raw = false: also the per-instance psi(sum_i alpha_eph) kernel over n_inst
// descriptors
hipError_t launch_prep(int dtype, int psi, bool raw, dim3 grid, hipStream_t st,
                       const BldInst* insts, const PrepItem* items, const uint32_t* n_items,
                       uint32_t n_inst, uint32_t zmax);
hipError_t launch_score(dim3 grid, hipStream_t st, const BldInst* insts, const PrepItem* items,
                        const uint32_t* n_items, uint32_t n_inst);
hipError_t launch_psi_eval(int kind, const double* xin, double* out, size_t n, hipStream_t st);
hipError_t launch_init_s(int dtype, void* S, const void* X, size_t n_fibers, uint32_t z,
                         uint64_t seed, hipStream_t st);
hipError_t init_kernel_attributes();
hipError_t launch_fact(int dtype, const BldInst* inst, uint32_t y, uint32_t z, double eps, double* W,
                       double* H, double* L, hipStream_t st);
// FP64 step pass (MODE_UPDATE or MODE_ADD), two lanes per fiber, z bucket
// zb <= 64 and LDS read width rw (bld_pass_f64.hip)
hipError_t launch_pass_f64(int psi, int mode, int zb, int rw, dim3 grid, hipStream_t st, const BldInst* insts,
                           const PassItem* items, const uint32_t* n_items);
hipError_t init_f64_attributes();
// any mode and dtype for instances deeper than kFusedZ (bld_wide.hip)
int wide_regs_nk(uint32_t z);  // wavefront-lengths of a fiber the wide pass holds in registers; 0: too deep
hipError_t launch_pass_wide(int dtype, int psi, int mode, int nk, dim3 grid, hipStream_t st, const BldInst* insts,
                            const PassItem* items, const uint32_t* n_items);
// FP32 step pass (MODE_UPDATE or MODE_ADD) specialised on the exact fiber
// depth z (bld_pass_f32z.hip)
hipError_t launch_pass_f32z(int z, int mode, dim3 grid, hipStream_t st, const BldInst* insts,
                            const PassItem* items, const uint32_t* n_items);
hipError_t init_f32z_attributes();
// step passes over the packed nonempty fibers of n tiles (bld_live.hip) of
// instances with z <= 32 or (big) 33 <= z <= 64; lds: dynamic LDS bytes
hipError_t launch_pass_live(int dtype, int psi, int mode, bool big, uint32_t n, hipStream_t st, const LiveTile* tiles,
                            uint32_t lds);
hipError_t init_live_attributes();
// LDS of a block whose tile has n fibers, with kc elements of k at once
size_t live_lds_need(int dtype, uint32_t z, uint32_t tile_cols, uint32_t rows, uint32_t n, uint32_t kc);
void live_group(int dtype, uint32_t z, uint32_t* elems, uint32_t* fibers);
hipError_t launch_live_count(int dtype, const BldInst* insts, const PassItem* items, uint32_t n, uint32_t* counts,
                             hipStream_t st);
hipError_t launch_live_build(int dtype, const BldInst* insts, LiveTile* tiles, uint32_t n, hipStream_t st);
hipError_t launch_live_gather(int dtype, const BldInst* insts, const LiveTile* tiles, uint32_t n, hipStream_t st);
hipError_t launch_live_scatter(int dtype, const BldInst* insts, const LiveTile* tiles, uint32_t n, hipStream_t st);
// iters iterations of n_inst FP64 instances of one tile each, a block per
// instance with everything in LDS (bld_tiny.hip): S from S_src, S and its
// partial sums out
constexpr uint32_t kTinyElems = 4096;
constexpr size_t kTinyLds = 156 * 1024;
size_t tiny_lds(uint32_t x, uint32_t y, uint32_t z);
uint32_t tiny_threads(uint32_t x, uint32_t y, uint32_t z);
hipError_t launch_tiny(int psi, uint32_t n_inst, uint32_t threads, size_t lds, hipStream_t st, const BldInst* insts,
                       uint32_t iters);
hipError_t init_tiny_attributes();
// approximate solver (bld_appr.hip): mode 0 sums, 1 nu step, 2 mu step
hipError_t launch_appr_pass(int dtype, int mode, int zb, dim3 grid, hipStream_t st, const ApprInst* insts,
                            const PassItem* items, const uint32_t* n_items, uint32_t zmax);
hipError_t launch_appr_factor(int dtype, int half, dim3 grid, hipStream_t st, const ApprInst* insts,
                              const PassItem* items, const uint32_t* n_items);
// the FP64 iteration over the nonempty entries of X (bld_appr_live.hip): step
// 0 sums (row and column items), 1 step
hipError_t launch_appr_live(int step, uint32_t n, hipStream_t st, const ApprInst* insts, const PassItem* items);
hipError_t launch_appr_psiA(uint32_t n_inst, uint32_t zmax, hipStream_t st, const ApprInst* insts);
hipError_t launch_appr_count(const double* X, uint32_t x, uint32_t y, uint32_t* counts, hipStream_t st);
hipError_t launch_appr_fill(const double* X, uint32_t x, uint32_t y, const uint32_t* rptr, uint32_t* ridx, double* rxv,
                            const uint32_t* cptr, uint32_t* cidx, double* cxv, hipStream_t st);
// dst (n x m) = src (m x n) transposed
hipError_t launch_appr_transpose(double* dst, const double* src, uint32_t n, uint32_t m, hipStream_t st);
hipError_t launch_appr_S(int dtype, const ApprInst* inst, size_t n_fibers, hipStream_t st);
hipError_t init_appr_attributes();
void ensure_runtime();  // per-process kernel attributes, once

// ----------------------------------------------------------------- sampler
int sample_X(uint64_t seed, size_t x, size_t y, size_t z, const double* alpha,
             const double* beta, double a, double b, double* X);
int sample_S(uint64_t seed, size_t x, size_t y, size_t z, const double* alpha,
             const double* beta, double a, double b, double* S);
template <typename T>
int init_S(uint64_t seed, const T* X, size_t x, size_t y, size_t z, T* S);
// the priors of bnmf_priors: W (x*z), H (z*y), L (y)
void sample_priors(uint64_t seed, size_t x, size_t y, size_t z, const double* alpha,
                   const double* beta, double a, double b, std::vector<double>& W,
                   std::vector<double>& H, std::vector<double>& L);
// device draws of X (mode 0, n = x*y) or S (mode 1, n = x*y*z) from the priors
hipError_t launch_sample(double* out, const double* W, const double* H, const double* L, size_t y,
                         uint32_t z, uint64_t seed, int mode, size_t n, hipStream_t st);

// ----------------------------------------------------------- tile planner
// z bucket of the fused generic pass (z <= kFusedZ); 0 for the wide pass
uint32_t z_bucket(uint32_t z);
// tall: without the short tiles of small FP64 instances
uint32_t choose_ti_rows(int dtype, uint32_t x, uint32_t y, uint32_t z, bool tall = false);
// Lays the items of one pass launch out XCD by XCD (L2 sharing of the
// per-column psi staging); results do not depend on item order.
void xcd_order(std::vector<PassItem>& items);

// ------------------------------------------------------ no-allocation solve
// bld_mult's FP32 solve on caller-owned device buffers, workspace in the
// library's fixed device scratch (noalloc.hip); enqueued on st
void bld_mult_f32_noalloc(const float* X, uint32_t x, uint32_t y, uint32_t z, const double* alpha,
                          const double* beta, size_t max_iter, double eps, const float* S0, uint64_t seed,
                          float* S, hipStream_t st);

// ------------------------------------------------------------- tile table
// Rows per pass tile by shape class (tune.cpp); 0 = built-in rule.
int tune_zclass(uint32_t z);
int tune_sclass(uint64_t fibers);
uint32_t tune_ti_cap(int dtype, uint32_t z, uint64_t fibers);
void tune_set(int dtype, uint32_t z, uint64_t fibers, uint32_t cap);
void tune_load(const std::string& path);
void tune_save(const std::string& path);
std::string tune_source();

// --------------------------------------------------------- device buffers
struct DeviceBuffer {
    void* ptr = nullptr;
    size_t bytes = 0;
    DeviceBuffer() = default;
    explicit DeviceBuffer(size_t n);
    ~DeviceBuffer();
    DeviceBuffer(const DeviceBuffer&) = delete;
    DeviceBuffer& operator=(const DeviceBuffer&) = delete;
    DeviceBuffer(DeviceBuffer&& o) noexcept : ptr(o.ptr), bytes(o.bytes) {
        o.ptr = nullptr;
        o.bytes = 0;
    }
    DeviceBuffer& operator=(DeviceBuffer&& o) noexcept;
    template <typename T>
    T* as(size_t byte_off = 0) const {
        return reinterpret_cast<T*>(static_cast<char*>(ptr) + byte_off);
    }
};

// Results to (pageable) host memory, large or many ones through a pinned buffer
// of its own (hostcopy.cpp). Safe with several threads: one copy through the
// buffer at a time.
struct HostStage {
    void* pinned = nullptr;
    size_t fetched = 0;  // bytes of results large enough for the buffer
    std::mutex mu;
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage();
    // bytes from device memory, after the work on st; returns when they are there
    void copy(void* dst, const void* src, size_t bytes, hipStream_t st);
};

// ----------------------------------------------------------------- batches
struct InstSpec {
    uint32_t x = 0, y = 0, z = 0;
    const void* X = nullptr;       // host
    const double* alpha = nullptr; // host
    const double* beta = nullptr;  // host
    double a = 1.0, b = 1.0;
    const void* S0 = nullptr;      // host or null
    uint64_t seed = 0;
};

// Byte layout of one instance inside an arena.
struct InstLayout {
    uint32_t x, y, z, zb, rw, hs, hm, ti_rows, n_ti, n_tj, nA, n_cj;
    uint32_t tile_cols;  // fibers per tile row: kTileCols, or kWideCols (z > kFusedZ)
    size_t off_S, off_S0, off_X, off_alpha, off_beta, off_psib, off_psia, off_partA, off_psiA, off_pjk,
        off_ipk, off_score, off_result;
    size_t bytes;  // total, 256-byte aligned
    size_t elements() const { return (size_t)x * y * z; }
};
// with_S0: reserve a separate buffer for the initial tensor (batches keep S0
// to restart solves; the server solves in place).
InstLayout plan_instance(int dtype, uint32_t x, uint32_t y, uint32_t z, bool with_S0 = true, bool tall = false);
BldInst make_desc(const InstLayout& L, void* base, double eps, double a, double b, bool first,
                  bool nonneg = false);

// Kernel of one pass launch: the exact-z FP32 step kernel (zexact > 0), the
// FP64 step kernel (f64, z bucket zb, LDS read width rw), the generic
// z-bucket kernel (zb, rw) or, for z > kFusedZ, the wide kernel (zb = 0).
// Instances with equal keys share a launch. The key follows from the instance's
// shape, S0 and parameters, so an instance runs the same kernel alone, batched or
// served, and from whether its nonempty fibers are packed (the same bits).
struct PassKey {
    int zexact = 0, zb = 0, rw = 0, f64 = 0;  // wide: rw as wide_regs_nk
    int live = 0;  // step over packed nonempty fibers: 1 for z <= 32, 2 for 33 <= z <= 64
    bool operator<(const PassKey& o) const {
        return std::tie(zexact, zb, rw, f64, live) < std::tie(o.zexact, o.zb, o.rw, o.f64, o.live);
    }
    bool wide() const { return zexact == 0 && zb == 0; }
};
// fibers per tile row of an instance: kWideCols for z > kFusedZ, else
// kTileColsF64 (FP64, z <= 32), half that (FP64, z <= 64) or kTileCols (FP32)
uint32_t tile_cols_of(int dtype, uint32_t z);
// nonneg: the instance's S stays >= 0 (S0 >= 0 and beta >= 1); live: its
// nonempty fibers are packed (LivePlan)
PassKey pass_key(int dtype, int mode, const InstLayout& L, bool nonneg, bool live = false);
hipError_t launch_pass_key(const PassKey& k, int dtype, int psi, int mode, dim3 grid,
                           hipStream_t st, const BldInst* insts, const PassItem* items,
                           const uint32_t* n_items, uint32_t zmax);

// nonneg: S stays >= 0 (S0 >= 0 and beta >= 1). packable: additionally every
// gradient of its solve is finite, so that a fiber with X_ij = 0 stays exactly
// zero, and X looks sparse enough (LivePlan).
void classify(int dtype, const InstSpec& s, double eps, bool* nonneg, bool* packable);

// Which instances of a batch keep their nonempty fibers packed, and where
// (live.cpp). Results do not depend on it.
class LivePlan {
   public:
    // Counts the nonempty fibers of the candidates' tiles (X and the tile
    // plan from the descriptors) and lays the packed buffers out.
    // scratch: device memory of scratch_bytes, used until the call returns; it
    // starts with the descriptors. st: where X is ready; the counts run there (a
    // server's own stream, never the null stream, on which results are copied to
    // callers). mem(n, bytes): where the packed buffers of instance n come from and
    // are given back to (null for none left); without it they are the plan's own.
    LivePlan(int dtype, bool add, const std::vector<BldInst>& descs, const std::vector<InstLayout>& lay,
             const std::vector<bool>& candidate, char* scratch, hipStream_t st,
             const std::function<void*(size_t, size_t)>& mem = nullptr);
    LivePlan() = default;
    static size_t scratch_bytes(const std::vector<InstLayout>& lay);
    // Largest share of nonempty fibers at which packing an instance pays, alone or
    // among its like; elements: those of its batch. add: the additive solver's
    // step. None is packed above kMostShare.
    static constexpr double kMostShare = 0.5;
    static double most_share(int dtype, bool add, size_t x, size_t y, uint32_t z, size_t elements);
    // Iterations from which packing an instance of so many elements pays.
    static size_t least_iterations(size_t elements);
    // false where X (host, x*y entries) is plainly fuller than `most`
    static bool worth(int dtype, const void* X, size_t x, size_t y, double most);
    bool any() const { return !tiles_.empty(); }
    bool live(size_t n) const { return n < lds_.size() && lds_[n] > 0; }
    uint32_t lds(size_t n) const { return lds_[n]; }
    size_t fibers(size_t n) const { return fibers_[n]; }  // its nonempty fibers
    size_t bytes() const { return bytes_; }
    // Appends the tiles of one launch (items: batch instance numbers) to the
    // tile table and returns the first one's index.
    uint32_t add_launch(std::vector<PassItem>& items, const std::vector<BldInst>& descs);
    // Uploads the tile table and builds the lists; insts: the descriptors on
    // the device. A plan whose buffers are not its own keeps its table on the
    // host (host_tiles, complete once st is done) and only builds in tab.
    void build(const std::vector<BldInst>& descs, const BldInst* insts, hipStream_t st, LiveTile* tab = nullptr);
    const LiveTile* tiles() const { return tab_; }
    const std::vector<LiveTile>& host_tiles() const { return tiles_; }
    // packed S from S_src, and S from its packed form
    void gather(const BldInst* insts, hipStream_t st) const;
    void scatter(const BldInst* insts, hipStream_t st) const;

   private:
    struct Off {
        char* base;  // of the instance's buffers
        size_t Sc, fib, xv, rdesc, cdesc, map, smap, tile0;
    };
    int dtype_ = 0;
    LiveTile* tab_ = nullptr;
    size_t bytes_ = 0;
    DeviceBuffer buf_;
    std::vector<Off> offs_;
    std::vector<size_t> fibers_;
    std::vector<uint32_t> lds_;  // 0: the instance runs the dense passes
    std::vector<uint32_t> slot_, count_;  // per tile of the live instances: first slot, fibers
    std::vector<LiveTile> tiles_;
};

// A fixed set of instances sharing one arena, one stream and one set of
// captured per-iteration graphs.
class Batch {
   public:
    // algo: BNMF_ALGO_MULT (bld_mult) or BNMF_ALGO_ADD (bld_add); iters: the
    // iterations of the batch's only solve, where that is known
    Batch(int dtype, int psi_mode, double eps, const std::vector<InstSpec>& specs, int algo = BNMF_ALGO_MULT,
          size_t iters = SIZE_MAX);
    ~Batch();
    void solve_async(size_t iters);
    // Restarts from S0 and runs at most max_iter iterations; every
    // check_every iterations the FP64 log_marginal_S of every instance is
    // evaluated, and the solve stops once each relative change is <= tol.
    // Returns the iterations run; lm_out (n values, may be null) receives the
    // final log-marginals. Synchronous.
    size_t solve_tol(size_t max_iter, double tol, size_t check_every, double* lm_out);
    void synchronize();
    void get_S(size_t idx, void* host) const;
    void log_marginal(double* out);
    void time_pass(int reps, double* pass_ms, double* iter_ms);
    void tensor_sums(void* S_pjk, void* S_ipk, void* S_ijp);
    // bld_fact of instance idx's current S: W (x*z), H (z*y), L (y), host
    void fact(size_t idx, double eps, double* W, double* H, double* L);
    bnmf_batch_info info() const;
    size_t size() const { return layouts_.size(); }

   private:
    struct Bucket {
        PassKey key;
        int lane;          // side stream the bucket's pass runs on
        size_t work;       // elements
        uint32_t zmax;
        uint32_t n_items;
        size_t off_items;  // in meta_
        size_t off_count;
        uint32_t tile0 = 0, lds = 0;  // live groups: first tile, dynamic LDS
    };
    // What a batch takes beyond what it cannot do without: short tiles and
    // packed fibers, short tiles, nothing.
    enum class Extras { kPacked, kShortTiles, kNone };
    // Everything on the device for specs; release() undoes it.
    void plan(const std::vector<InstSpec>& specs, Extras extras);
    void release();
    // iterations of a batch of tiny instances; first: from S0
    void run_tiny(size_t iters, bool first);
    // S of the packed instances from their packed form, and back
    void unpack_S();
    void pack_S(bool first);
    void enqueue_iteration(bool first) { enqueue_iterations(1, first); }
    // first iteration of a solve (step counters reset, S0's partials, the
    // step reading S0), then `rem` more iterations from the captured graphs
    void start_solve();
    void replay_iterations(size_t rem);
    // `iters` iterations; each update group runs prep, psi(A) and its pass
    // on its own stream, iteration after iteration, with one fork and join
    // (with_prep = false: the update passes alone, for timing)
    void enqueue_iterations(int iters, bool first, bool with_prep = true);
    void enqueue_pass(int mode, bool first);
    // pass launches of the update pass (groups_[0]) and of the sums-only and
    // scoring passes (groups_[1])
    std::vector<Bucket>& groups_of(int mode) {
        return groups_[(mode == MODE_UPDATE || mode == MODE_ADD) ? 0 : 1];
    }
    hipGraphExec_t graph_of(int level);

    int dtype_, psi_;
    int algo_ = BNMF_ALGO_MULT;
    int step_mode_ = MODE_UPDATE;  // pass mode of an iteration's step
    int dev_ = 0;
    double eps_;
    size_t es_;
    size_t iters_known_;  // iterations of the only solve, or SIZE_MAX
    std::vector<InstLayout> layouts_;
    std::vector<InstSpec> specs_;
    DeviceBuffer arena_;
    DeviceBuffer meta_;  // descriptors, work lists, counts
    LivePlan live_;
    // every instance is tiny: threads and LDS of a block (0: run the passes),
    // iterations of a launch
    uint32_t tiny_threads_ = 0, tiny_iters_ = 1;
    size_t tiny_lds_ = 0;
    mutable HostStage stage_;
    size_t off_desc_first_ = 0, off_desc_ = 0, off_prep_items_ = 0, off_prep_count_ = 0;
    size_t off_iter_ = 0;  // additive solver: uint32 iteration counters, one per instance
    uint32_t n_prep_items_ = 0, zmax_ = 0;
    std::vector<Bucket> groups_[2];
    // per stream: descriptor arrays of the instances of its update groups
    // (the groups' pass items index them), its prep work list
    struct Lane {
        size_t off_desc = 0, off_desc_first = 0, off_prep = 0, off_prep_count = 0;
        uint32_t n_prep = 0, n_inst = 0, zmax = 0;
    };
    std::vector<Lane> lanes_;
    hipStream_t stream_ = nullptr;
    // z-bucket passes of one iteration are independent: they run on up to
    // four streams forked from and joined back to stream_ (graph branches
    // when captured)
    std::vector<hipStream_t> side_;
    std::vector<hipEvent_t> fork_ev_, join_ev_;
    // captured iteration graphs of 1, 2, 4, ... unroll_ iterations (level l
    // holds 2^l), each instantiated on first use
    static constexpr int kGraphLevels = 7;
    hipGraphExec_t graphs_[kGraphLevels] = {};
    int unroll_ = 32;
    // the partial axis sums in the workspace belong to the current S (true
    // after a solve: its last pass accumulates them)
    bool partials_valid_ = false;
    int cus_ = 256;
    size_t device_bytes_ = 0;
};

// ------------------------------------------------- approximate solver
struct ApprSpec {
    uint32_t x = 0, y = 0, z = 0;
    const void* X = nullptr;        // host, x*y
    const double* alpha = nullptr;  // host, x
    const double* beta = nullptr;   // host, z
    const void* nu0 = nullptr;      // host x*z, or null (drawn from seed)
    const void* mu0 = nullptr;      // host z*y, or null (drawn from seed)
    uint64_t seed = 0;
};

// Instances of bld::bld_appr solved together: the factors stay resident,
// one captured graph per iteration.
class ApprBatch {
   public:
    ApprBatch(int dtype, double eps, const std::vector<ApprSpec>& specs);
    ~ApprBatch();
    // restarts from nu0 / mu0 and runs iters iterations
    void solve_async(size_t iters);
    void synchronize();
    // S (x*y*z, formed from the current factors), nu (x*z), mu (z*y); any null
    void get(size_t idx, void* S, void* nu, void* mu);
    // mean ms of one iteration (graph replays, HIP events); advances the factors
    double time_iteration(int reps);
    size_t device_bytes() const;
    size_t size() const { return lay_.size(); }

   private:
    struct L_ {
        uint32_t x, y, z, ti_rows, n_ti, n_tj, nA, n_cj;
        size_t off_X, off_nu, off_mu, off_nu0, off_mu0, off_alpha, off_beta, off_psib, off_psia, off_partA,
            off_psiA, off_pjk, off_pjk2, off_ipk, off_ipk2, off_S;
        bool live = false;  // over the nonempty entries of X
        size_t entries = 0;
    };
    struct Group {
        uint32_t zb, zmax, n_items;
        size_t off_items, off_count;
    };
    // everything on the device for specs, with the lists of nonempty entries
    // or without; release() undoes it
    void plan(const std::vector<ApprSpec>& specs, double eps, bool lists);
    void release();
    void enqueue_dense();
    void enqueue_live(hipStream_t st);
    hipGraphExec_t graph_of(int level);
    void replay(size_t iters);
    void load_factors();
    void store_factors();
    bool live_candidate(const ApprSpec& s, double eps) const;
    void plan_live(uint32_t* counts, std::vector<ApprInst>& ai, std::vector<BldInst>& bi);

    int dtype_, psi_ = 0;
    size_t es_;
    std::vector<L_> lay_;
    std::vector<Group> groups_;
    DeviceBuffer arena_, meta_;
    size_t off_ai_ = 0, off_bi_ = 0, off_prep_ = 0, off_prep_count_ = 0, off_fnu_ = 0, off_fnu_count_ = 0,
           off_fmu_ = 0, off_fmu_count_ = 0;
    uint32_t n_prep_ = 0, n_fnu_ = 0, n_fmu_ = 0;
    // work lists over the nonempty entries: both sides (sums), rows, columns
    DeviceBuffer lists_;
    size_t off_live_ = 0, off_lrow_ = 0, off_lcol_ = 0;
    uint32_t zmax_dense_ = 0, zmax_live_ = 0, n_live_ = 0, n_lrow_ = 0, n_lcol_ = 0;
    hipStream_t stream_ = nullptr;
    hipStream_t side_ = nullptr;  // the listed instances' branch of a graph
    hipEvent_t fork_ = nullptr, join_ = nullptr;
    // captured graphs of 1, 2, 4, ... iterations, each instantiated on first use
    static constexpr int kGraphLevels = 5;
    hipGraphExec_t graphs_[kGraphLevels] = {};
    HostStage stage_;
};

}  // namespace bnmf
