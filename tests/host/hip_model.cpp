// See hip_model.h.
#include "hip_model.h"

#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <unordered_map>

#include "../../ckks-train_amd/csrc/runtime.h"

struct EventState {
    uint64_t recorded = 0, done = 0;  // the latest record queued, and the latest that has run
    hipStream_t stream = nullptr;
};
struct ihipEvent_t {
    std::shared_ptr<EventState> st = std::make_shared<EventState>();
};
struct StreamOp {
    std::function<bool()> ready;
    std::function<void()> run;
};
struct ihipStream_t {
    std::deque<StreamOp> q;
    bool capturing = false;
};

namespace {
std::recursive_mutex mu;
thread_local hipError_t last_error = hipSuccess;
std::unordered_map<void*, size_t> blocks;
size_t held = 0;

#define LOCKED std::lock_guard<std::recursive_mutex> lk(mu)

bool step_one(hipStream_t s) {
    if (s->q.empty()) return false;
    if (s->q.front().ready && !s->q.front().ready()) return false;
    StreamOp op = std::move(s->q.front());
    s->q.pop_front();
    if (op.run) op.run();
    return true;
}
void finish_event(const std::shared_ptr<EventState>& e, uint64_t upto);
// Runs s until it is empty (or e has reached upto), the streams that it waits for before it.
void drain(hipStream_t s, const std::function<bool()>& enough) {
    while (!s->q.empty() && !enough())
        if (!step_one(s)) {
            std::fprintf(stderr, "MODEL: a stream waits for an event that cannot complete\n");
            std::abort();
        }
}
void finish_event(const std::shared_ptr<EventState>& e, uint64_t upto) {
    if (e->done < upto) drain(e->stream, [&] { return e->done >= upto; });
}
hipError_t fail_with(hipError_t e) {
    last_error = e;
    return e;
}
void* reserve(size_t bytes) {
    void* p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (p == MAP_FAILED) return nullptr;
    blocks[p] = bytes;
    held += bytes;
    return p;
}
void release(void* p) {
    auto it = blocks.find(p);
    if (it == blocks.end()) return;
    held -= it->second;
    munmap(p, it->second);
    blocks.erase(it);
}
}  // namespace

namespace model {
std::vector<Copy> uploads;
uint64_t launches = 0;
bool refuse_launch = false;
float elapsed_ms = 1.0f;
uint64_t records_while_capturing = 0;
uint64_t destroyed_graphs = 0;
uint64_t ip_launches = 0, ip_finish_launches = 0;
size_t free_bytes = (size_t)1 << 40;

std::function<void()> on_launch;
std::function<void(size_t)> on_malloc;

void kernel() {
    LOCKED;
    if (on_launch) on_launch();
    if (refuse_launch) {
        refuse_launch = false;
        last_error = hipErrorLaunchFailure;
        return;
    }
    ++launches;
}
void queue_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
    LOCKED;
    if (s->capturing) return;  // a node of the caller's graph
    s->q.push_back({nullptr, [=] { std::memcpy(dst, src, bytes); }});
}
void set_capturing(hipStream_t s, bool on) {
    LOCKED;
    s->capturing = on;
}
size_t pending(hipStream_t s) {
    LOCKED;
    return s->q.size();
}
bool step(hipStream_t s) {
    LOCKED;
    return step_one(s);
}
size_t mapped() {
    LOCKED;
    return held;
}
}  // namespace model

// ------------------------------------------------------------------ the runtime's calls
#define OK return hipSuccess
extern "C" {
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    OK;
}
hipError_t hipSetDevice(int) { OK; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "error"; }
hipError_t hipDeviceSynchronize() { OK; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    OK;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) {
    *p = nullptr;
    OK;
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { OK; }
hipError_t hipMemPoolGetAttribute(hipMemPool_t, hipMemPoolAttr, void* v) {
    *(uint64_t*)v = 0;
    OK;
}
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { OK; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = model::free_bytes;
    *t = (size_t)1 << 40;
    OK;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = new ihipStream_t;
    OK;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    delete s;
    OK;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    LOCKED;
    if (s->capturing) return fail_with(hipErrorStreamCaptureUnsupported);
    drain(s, [] { return false; });
    OK;
}
hipError_t hipStreamQuery(hipStream_t s) {
    LOCKED;
    if (s->capturing) return fail_with(hipErrorStreamCaptureUnsupported);
    return s->q.empty() ? hipSuccess : hipErrorNotReady;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    LOCKED;
    *st = s->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    OK;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    LOCKED;
    auto st = e->st;
    const uint64_t upto = st->recorded;
    s->q.push_back({nullptr, [st, upto] { finish_event(st, upto); }});
    OK;
}

hipError_t hipEventCreate(hipEvent_t* e) {
    *e = new ihipEvent_t;
    OK;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    OK;
}
// On a stream being captured the record joins the caller's graph: the event itself then reads as
// complete, as one that was never recorded.
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    LOCKED;
    if (s->capturing) {
        ++model::records_while_capturing;
        e->st = std::make_shared<EventState>();
        OK;
    }
    auto st = e->st;
    st->stream = s;
    const uint64_t id = ++st->recorded;
    s->q.push_back({nullptr, [st, id] { st->done = id; }});
    OK;
}
hipError_t hipEventQuery(hipEvent_t e) {
    LOCKED;
    return e->st->done >= e->st->recorded ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    LOCKED;
    finish_event(e->st, e->st->recorded);
    OK;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = model::elapsed_ms;
    OK;
}

hipError_t hipMalloc(void** p, size_t bytes) {
    LOCKED;
    if (model::on_malloc) model::on_malloc(bytes);
    *p = reserve(bytes);
    return *p ? hipSuccess : fail_with(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) {
    LOCKED;
    release(p);
    OK;
}
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t) { return hipMalloc(p, bytes); }
hipError_t hipFreeAsync(void* p, hipStream_t s) {
    LOCKED;
    s->q.push_back({nullptr, [p] { release(p); }});
    OK;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = std::malloc(bytes);
    OK;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    OK;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    OK;
}
hipError_t hipMemset(void*, int, size_t) { OK; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { OK; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    OK;
}
hipError_t hipMemcpyAsync(void* d, const void* src, size_t n, hipMemcpyKind k, hipStream_t s) {
    LOCKED;
    if (k == hipMemcpyHostToDevice) model::uploads.push_back({n, false});
    model::queue_copy(d, src, n, s);
    OK;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { OK; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = nullptr;
    OK;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = (hipGraphExec_t)(uintptr_t)1;
    OK;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { OK; }
hipError_t hipGraphDestroy(hipGraph_t) { OK; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) {
    ++model::destroyed_graphs;
    OK;
}
}

// ------------------------------------------------------------------ the library's kernels
namespace ckh {
hipError_t upload_launch(const void* pinned, void* out, u64 bytes, hipStream_t s) {
    const uint64_t before = model::launches;
    model::kernel();
    if (model::launches == before) return last_error;
    std::lock_guard<std::recursive_mutex> lk(mu);
    model::uploads.push_back({bytes, true});
    model::queue_copy(out, pinned, bytes, s);
    return hipSuccess;
}
uint8_t* static_scratch_address(int) {
    static uint8_t* p = (uint8_t*)mmap(nullptr, CKH_STATIC_SCRATCH_BYTES, PROT_READ | PROT_WRITE,
                                       MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p;
}
u32 xcc_layout_check(hipStream_t) { return 0; }
u32 fused_occupancy() { return 1; }
bool ntt_fast_supported(u32 log_n) { return log_n >= 12 && log_n <= 16; }

#define K model::kernel()
void ntt_forward(const NttTables&, const LimbRef*, u32, hipStream_t) { K; }
void ntt_inverse(const NttTables&, const LimbRef*, u32, hipStream_t) { K; }
void ntt_fast_inverse(const NttTables&, const LimbRef*, u32, hipStream_t, const YForm*) { K; }
void ntt_fast_forward_finish(const NttTables&, const LimbRef*, const FinishJob*, u32, hipStream_t) { K; }
void ntt_fast_forward_cols(const NttTables&, const LimbRef*, u32, hipStream_t) { K; }
void ntt_fast_forward_rows(const NttTables&, const LimbRef*, u32, hipStream_t) { K; }
void ntt_fast_forward_rows_finish(const NttTables&, const LimbRef*, const FinishJob*, u32, hipStream_t) { K; }
void ntt_fast_forward_fused(const NttTables&, const LimbRef*, u32, const FinishJob*, u32*, const FusedCfg&, hipStream_t) { K; }
void ntt_fast_inverse_fused(const NttTables&, const LimbRef*, u32, u32*, const FusedCfg&, hipStream_t) { K; }
void narrow_ip_inverse(const NttTables&, const IpInvJob*, const LimbRef*, u32, const YForm*, hipStream_t) { K; }
void narrow_ip_finish(const NttTables&, const IpFinJob*, u32, hipStream_t) {
    ++model::ip_finish_launches;
    K;
}
void rows_ip_launch(const NttTables&, const RowIpJob*, u32, hipStream_t) { K; }
void rows_ip_fin_launch(const NttTables&, const RowIpFinJob*, u32, hipStream_t) { K; }
void conv_cols_launch(const ConvTables&, const NttTables&, const ConvColRef*, u32, u32, hipStream_t) { K; }
void conv_launch(const ConvTables&, const ConvJob*, u32, u32, u32, u32, u32, bool, hipStream_t) { K; }
void finish_launch(const FinishJob*, u32, const PrimeConst*, u32, hipStream_t) { K; }
void mul_sum_launch(const MulSumJob*, const MulSumTerm*, u32, const PrimeConst*, u32, hipStream_t) { K; }
void tensor_sum_launch(const TensorJob*, const TensorTerm*, u32, const PrimeConst*, u32, hipStream_t) { K; }
void tensor_launch(const TensorTerm&, u64*, u32, const PrimeConst*, u32, hipStream_t) { K; }
void add_sum_launch(const AddSumJob*, const u64* const*, u32, const PrimeConst*, u32, hipStream_t) { K; }
void inner_product_launch(const IpJob*, u32, const PrimeConst*, u32, bool, hipStream_t) {
    ++model::ip_launches;
    K;
}
void stream_copy_launch(const void*, void*, u64, hipStream_t) { K; }
void copy_launch(const LimbRef*, u32, u32, hipStream_t) { K; }
void pointwise_launch(PwOp, const u64*, const u64*, u64*, u32, u32, const PrimeConst*, u32, hipStream_t) { K; }
void scalar_mul_launch(const u64*, u64*, u32, const u64*, bool, const PrimeConst*, u32, hipStream_t) { K; }
void automorphism_ntt_launch(const u64*, u64*, u32, u64, u32, hipStream_t) { K; }
void automorphism_coeff_launch(const u64*, u64*, u32, u32, u32, u64, const PrimeConst*, u32, hipStream_t) { K; }
void automorphism_batch_launch(const AutJob*, u32, u32, hipStream_t) { K; }
void fill_uniform_launch(u64*, u32, u32, u32, u64, u64, const PrimeConst*, u32, hipStream_t) { K; }
void digest_launch(const u64*, u64, u64*, hipStream_t) { K; }
}  // namespace ckh
