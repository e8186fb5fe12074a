// fake_hip.cpp — a HIP runtime on host memory for tests of the host sources
// (planning, allocation, scheduling): device memory is malloc'ed, copies are
// memcpy, streams and events do nothing, and kernels are empty except those
// whose output the host reads to make its plan. Linked in place of the runtime
// and of the kernels' launchers.
#include "fake_hip.hpp"

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../bnmf-algs_amd/csrc/bnmf_internal.hpp"

namespace fake {
std::mutex mu;
std::map<void*, size_t> blocks;
size_t used = 0, capacity = ~(size_t)0, fail_at = 0, mallocs = 0, pins = 0;
bool tiny = false;
std::vector<uint32_t> tiny_iters;
std::atomic<size_t> copies{0}, launches{0}, packs{0}, on_null{0};

void reset(size_t cap, size_t fail) {
    std::lock_guard<std::mutex> lk(mu);
    capacity = cap;
    fail_at = fail;
    mallocs = pins = 0;
    copies = launches = packs = on_null = 0;
}
size_t in_use() {
    std::lock_guard<std::mutex> lk(mu);
    return used;
}
size_t n_mallocs() {
    std::lock_guard<std::mutex> lk(mu);
    return mallocs;
}
size_t n_pins() {
    std::lock_guard<std::mutex> lk(mu);
    return pins;
}
}  // namespace fake

extern "C" {
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lk(fake::mu);
    ++fake::mallocs;
    *p = nullptr;
    if (fake::mallocs == fake::fail_at || fake::used + n > fake::capacity) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    std::memset(*p, 0xff, n);  // NaN in every type: nothing may count on fresh memory
    fake::blocks[*p] = n;
    fake::used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lk(fake::mu);
    auto it = fake::blocks.find(p);
    if (it == fake::blocks.end()) std::abort();
    fake::used -= it->second;
    fake::blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::mutex> lk(fake::mu);
    ++fake::pins;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    ++fake::copies;
    ++fake::on_null;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    ++fake::copies;
    fake::on_null += st == nullptr;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
static void* const kHandle = &fake::used;
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = static_cast<hipStream_t>(kHandle);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = static_cast<hipGraph_t>(kHandle);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* g, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *g = static_cast<hipGraphExec_t>(kHandle);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = static_cast<hipEvent_t>(kHandle);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
}

namespace bnmf {

static hipError_t launched() {
    ++fake::launches;
    return hipSuccess;
}

hipError_t init_kernel_attributes() { return hipSuccess; }
hipError_t init_f32z_attributes() { return hipSuccess; }
hipError_t init_f64_attributes() { return hipSuccess; }
hipError_t init_appr_attributes() { return hipSuccess; }
hipError_t init_live_attributes() { return hipSuccess; }
hipError_t init_tiny_attributes() { return hipSuccess; }

void read_layout(int, uint32_t z, uint32_t* rw, uint32_t* hs, uint32_t* hm) {
    *rw = z % 4 == 0 ? 4 : z % 2 == 0 ? 2 : 1;
    *hs = *hm = 0;
}
int wide_regs_nk(uint32_t z) { return z <= 256 ? (int)((z + 63) / 64) : 0; }
size_t tiny_lds(uint32_t x, uint32_t y, uint32_t z) { return fake::tiny ? (size_t)2 * x * y * z * 8 : kTinyLds + 1; }
uint32_t tiny_threads(uint32_t, uint32_t, uint32_t) { return 64; }
size_t live_lds_need(int, uint32_t, uint32_t, uint32_t, uint32_t n, uint32_t) { return 4096 + n; }
void live_group(int dtype, uint32_t z, uint32_t* elems, uint32_t* fibers) {
    *elems = dtype == 0 ? (z + 3) / 4 * 256 : z;
    *fibers = dtype == 0 ? 64 : 1;
}

hipError_t launch_pass(int, int, int, int, int, dim3, hipStream_t, const BldInst*, const PassItem*, const uint32_t*, uint32_t) { return launched(); }
hipError_t launch_pass_f64(int, int, int, int, dim3, hipStream_t, const BldInst*, const PassItem*, const uint32_t*) { return launched(); }
hipError_t launch_pass_f32z(int, int, dim3, hipStream_t, const BldInst*, const PassItem*, const uint32_t*) { return launched(); }
hipError_t launch_pass_wide(int, int, int, int, dim3, hipStream_t, const BldInst*, const PassItem*, const uint32_t*) { return launched(); }
hipError_t launch_pass_live(int, int, int, bool, uint32_t, hipStream_t, const LiveTile*, uint32_t) { return launched(); }
hipError_t launch_prep(int, int, bool, dim3, hipStream_t, const BldInst*, const PrepItem*, const uint32_t*, uint32_t, uint32_t) { return launched(); }
hipError_t launch_score(dim3, hipStream_t, const BldInst*, const PrepItem*, const uint32_t*, uint32_t) { return launched(); }
hipError_t launch_fact(int, const BldInst*, uint32_t, uint32_t, double, double*, double*, double*, hipStream_t) { return launched(); }
hipError_t launch_tiny(int, uint32_t, uint32_t, size_t, hipStream_t, const BldInst*, uint32_t iters) {
    fake::tiny_iters.push_back(iters);
    return launched();
}
hipError_t launch_live_build(int, const BldInst*, LiveTile*, uint32_t, hipStream_t) {
    ++fake::packs;
    return launched();
}
hipError_t launch_psi_eval(int, const double*, double*, size_t, hipStream_t) { return launched(); }
hipError_t launch_sample(double*, const double*, const double*, const double*, size_t, uint32_t, uint64_t, int, size_t, hipStream_t) { return launched(); }
void bld_mult_f32_noalloc(const float*, uint32_t, uint32_t, uint32_t, const double*, const double*, size_t, double, const float*, uint64_t, float*, hipStream_t) {}
hipError_t launch_live_gather(int, const BldInst*, const LiveTile*, uint32_t, hipStream_t) { return launched(); }
hipError_t launch_live_scatter(int, const BldInst*, const LiveTile*, uint32_t, hipStream_t) { return launched(); }
hipError_t launch_appr_pass(int, int, int, dim3, hipStream_t, const ApprInst*, const PassItem*, const uint32_t*, uint32_t) { return launched(); }
hipError_t launch_appr_factor(int, int, dim3, hipStream_t, const ApprInst*, const PassItem*, const uint32_t*) { return launched(); }
hipError_t launch_appr_live(int, uint32_t, hipStream_t, const ApprInst*, const PassItem*) { return launched(); }
hipError_t launch_appr_psiA(uint32_t, uint32_t, hipStream_t, const ApprInst*) { return launched(); }
hipError_t launch_appr_fill(const double*, uint32_t, uint32_t, const uint32_t*, uint32_t*, double*, const uint32_t*, uint32_t*, double*, hipStream_t) { return launched(); }
hipError_t launch_appr_transpose(double*, const double*, uint32_t, uint32_t, hipStream_t) { return launched(); }
hipError_t launch_appr_S(int, const ApprInst*, size_t, hipStream_t) { return launched(); }

hipError_t launch_init_s(int dtype, void* S, const void*, size_t n_fibers, uint32_t z, uint64_t, hipStream_t) {
    std::memset(S, 0, n_fibers * z * (dtype == 0 ? 4 : 8));
    return launched();
}

// nonempty entries of the tiles and of the rows and columns: the host's plan
// follows from them
template <typename T>
static uint32_t count_tile(const BldInst& I, const PassItem& it) {
    uint32_t n = 0;
    for (uint32_t i = it.ti * I.ti_rows; i < std::min(I.x, (it.ti + 1) * I.ti_rows); ++i)
        for (uint32_t j = it.tj * I.tile_cols; j < std::min(I.y, (it.tj + 1) * I.tile_cols); ++j)
            n += static_cast<const T*>(I.X)[(size_t)i * I.y + j] != T(0);
    return n;
}
hipError_t launch_live_count(int dtype, const BldInst* insts, const PassItem* items, uint32_t n, uint32_t* counts, hipStream_t st) {
    fake::on_null += st == nullptr;
    for (uint32_t t = 0; t < n; ++t) {
        const BldInst& I = insts[items[t].inst];
        counts[t] = dtype == 0 ? count_tile<float>(I, items[t]) : count_tile<double>(I, items[t]);
    }
    return launched();
}
hipError_t launch_appr_count(const double* X, uint32_t x, uint32_t y, uint32_t* counts, hipStream_t) {
    std::memset(counts, 0, ((size_t)x + y) * 4);
    for (uint32_t i = 0; i < x; ++i)
        for (uint32_t j = 0; j < y; ++j)
            if (X[(size_t)i * y + j] != 0.0) ++counts[i], ++counts[x + j];
    return launched();
}

}  // namespace bnmf
