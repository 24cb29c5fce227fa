// HIPBackend against a stand-in for libspy_hip.so that queues what the real one queues and carries it out at the next synchronisation of the
// stream: pinned memory that is written again too early shows as wrong bytes, calls can be made to fail, and allocations are counted.
// argv[1]: the scenario.  Prints "ok", or what went wrong (exit status 1).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "../../spy_amd/backend/hip_backend.h"
#include "../../include/spy_hip.h"

using namespace spy;

static std::vector<std::function<void()>> g_queue;
static int g_fail_download = 0, g_fail_sync = 0, g_fail_host_alloc = 0, g_host_allocs = 0, g_overwritten = 0, g_syncs = 0;

extern "C" {
int roctxRangePushA(const char *) { return 0; }
int roctxRangePop() { return 0; }
int spy_hip_init(int) { return 0; }
int spy_hip_device_info(char *, int, int *, size_t *, size_t *) { return 0; }
int spy_hip_stream_create(void **s) { *s = reinterpret_cast<void *>(1); return 0; }
int spy_hip_stream_destroy(void *) { return 0; }
int spy_hip_alloc(void **p, size_t n) { *p = std::malloc(n); return 0; }
int spy_hip_free(void *p) { std::free(p); return 0; }
int spy_hip_host_alloc(void **p, size_t n) { ++g_host_allocs; *p = nullptr; if (g_fail_host_alloc) return 2; *p = std::malloc(n); return 0; }
int spy_hip_host_free(void *p) { std::free(p); return 0; }
int spy_hip_sync(void *s) {
    if (s && g_fail_sync > 0) { --g_fail_sync; return 999; }
    ++g_syncs;
    for (auto &f : g_queue) f();
    g_queue.clear();
    return 0;
}
int spy_hip_upload(void *dst, const void *src, size_t n, void *s) { const int rc = spy_hip_sync(s); if (rc == 0) std::memcpy(dst, src, n); return rc; }
int spy_hip_download(void *dst, const void *src, size_t n, void *s) {
    if (g_fail_download > 0) { --g_fail_download; return 998; }
    const int rc = spy_hip_sync(s);
    if (rc == 0) std::memcpy(dst, src, n);
    return rc;
}
int spy_hip_take_error(int *f) { *f = 0; return spy_hip_sync(nullptr); }
int spy_hip_upload_pinned(void *dst, const void *src, size_t n, void *) {
    const std::vector<uint8_t> at_queue_time(static_cast<const uint8_t *>(src), static_cast<const uint8_t *>(src) + n);
    g_queue.push_back([=] { if (std::memcmp(src, at_queue_time.data(), n) != 0) ++g_overwritten; std::memcpy(dst, src, n); });
    return 0;
}
int spy_hip_download_pinned(void *dst, const void *src, size_t n, int *flag, void *) {
    if (g_fail_download > 0) { --g_fail_download; return 998; }
    g_queue.push_back([=] { std::memcpy(dst, src, n); *flag = 0; });
    return 0;
}
int spy_hip_op_relu(void *, const spy_hip_tensor *x, const spy_hip_tensor *y) {
    const spy_hip_tensor a = *x, b = *y;
    g_queue.push_back([=] {
        for (int64_t i = 0; i < a.ne[0] * a.ne[1]; ++i) { const float v = static_cast<const float *>(a.data)[i]; static_cast<float *>(b.data)[i] = v < 0 ? 0 : v; }
    });
    return 0;
}
#define UNUSED_OP(NAME, ...) int NAME(__VA_ARGS__) { return SPY_HIP_EUNSUPPORTED; }
typedef const spy_hip_tensor *T;
UNUSED_OP(spy_hip_op_silu, void *, T, T)
UNUSED_OP(spy_hip_op_quantize, void *, T, T)
UNUSED_OP(spy_hip_op_dup, void *, T, T)
UNUSED_OP(spy_hip_op_contiguous, void *, T, T)
UNUSED_OP(spy_hip_op_norm_rms, void *, T, T, float)
UNUSED_OP(spy_hip_op_binary, void *, int, T, T, T)
UNUSED_OP(spy_hip_op_softmax, void *, T, T, T, float)
UNUSED_OP(spy_hip_op_rope, void *, T, T, T, const spy_hip_rope_param *)
UNUSED_OP(spy_hip_op_get_row, void *, T, T, T)
UNUSED_OP(spy_hip_op_matmul, void *, T, T, T, void *, size_t)
size_t spy_hip_op_matmul_scratch_size(T, T) { return 0; }
}
void OperatorDefinition<OperatorType::Relu>::propagate() { output_data(0)->tensor.shape = input_data(0)->tensor.shape; }

// one Relu node between two host vectors
struct Pass {
    std::vector<float> x, y;
    DataNode in, out;
    OperatorDefinition<OperatorType::Relu> op;
    explicit Pass(int64_t n) : x(static_cast<size_t>(n)), y(static_cast<size_t>(n)) {
        in.node_prop.node_type = out.node_prop.node_type = DataNodeType::IO;
        in.tensor = Tensor(Shape({n, 1}, NumberType::FP32), x.data());
        op.add_input(&in);
        op.add_output(&out);
        op.propagate();
        out.tensor.set_data_ptr(y.data());
    }
    void run(Backend &be, float value) {
        for (float &v : x) v = value;
        for (float &v : y) v = -1;
        be.submit(&op);
    }
    bool holds(float value) const { for (float v : y) if (v != value) return false; return true; }
};

#define NEED(cond) do { if (!(cond)) { std::printf("line %d: %s\n", __LINE__, #cond); return 1; } } while (0)

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    const int64_t n = argc > 2 ? std::atoll(argv[2]) : 1000;
    ConfigTable config;
    hip::HIPBackend be(config);
    Pass p(n);
    if (what == "failed-download") {                 // the result's copy is not queued and nothing waits for the stream: the input's upload is still on its way
        g_fail_download = 1;
        p.run(be, 1.0f);
        NEED(be.last_status() == OperatorStatus::Fail);
        p.run(be, 2.0f);
        NEED(p.holds(2.0f));
    } else if (what == "failed-sync") {              // the wait for the result fails, and so does the one before the input's next upload
        g_fail_sync = 2;
        p.run(be, 1.0f);
        NEED(be.last_status() == OperatorStatus::Fail);
        const int before = g_syncs;
        p.run(be, 2.0f);
        NEED(g_syncs == before && p.holds(-1.0f));   // not run: its input could not be brought over
        p.run(be, 3.0f);
        NEED(p.holds(3.0f));
    } else if (what == "repeated") {
        for (int i = 0; i < 5; ++i) { p.run(be, static_cast<float>(i / 2)); NEED(p.holds(static_cast<float>(i / 2))); }
        NEED(be.last_status() == OperatorStatus::Success);
    } else if (what == "first-pass") {               // a single token's pass: ids, positions and a mask row in, logits out
        Pass ids(1), pos(1), mask(4352), logits(32000);
        const int before = g_host_allocs;
        for (Pass *q : {&ids, &pos, &mask}) { q->run(be, 5.0f); NEED(q->holds(5.0f)); }
        NEED(g_host_allocs == before);
        logits.run(be, 7.0f);                        // a large input has memory of its own
        NEED(logits.holds(7.0f) && g_host_allocs == before + 1);
    } else if (what == "many-inputs") {              // more than the block of the small ones holds, and one that grows
        std::vector<std::unique_ptr<Pass>> ps;
        for (int i = 0; i < 100; ++i) ps.push_back(std::make_unique<Pass>(n + i));
        for (int r = 0; r < 3; ++r)
            for (size_t i = 0; i < ps.size(); ++i) { ps[i]->run(be, static_cast<float>(i + 1000 * r)); NEED(ps[i]->holds(static_cast<float>(i + 1000 * r))); }
        ps[0]->in.tensor.shape = Shape({n / 2 + 1, 1}, NumberType::FP32);
        ps[0]->op.propagate();
        ps[0]->run(be, 1.0f);
        ps[0]->in.tensor.shape = Shape({n, 1}, NumberType::FP32);
        ps[0]->op.propagate();
        ps[0]->run(be, 3.0f);
        NEED(ps[0]->holds(3.0f) && be.last_status() == OperatorStatus::Success);
    } else if (what == "nothing-to-pin") {
        g_fail_host_alloc = 1;
        hip::HIPBackend other(config);
        for (int i = 0; i < 4; ++i) { p.run(other, static_cast<float>(i)); NEED(p.holds(static_cast<float>(i))); }
        NEED(other.last_status() == OperatorStatus::Success && other.last_error() == 0);
    } else { std::printf("no such scenario\n"); return 1; }
    NEED(g_overwritten == 0);
    std::printf("ok\n");
    return 0;
}
