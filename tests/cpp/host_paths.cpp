// Host paths of the library on a stand-in for the HIP runtime: device memory is
// host memory, kernels are counted and not run, and allocations fail when the
// scenario says so.  The definitions here come before the runtime's own in the
// program's symbol lookup, so the library as built is what runs.
//   host_paths <scenario>      prints what went wrong and exits 1, or "ok"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "sfhip.h"

struct dim3 {
    unsigned x, y, z;
};

namespace {
std::set<void*> live;           // device allocations
long mallocs_left = -1;         // allocations until they fail (-1: never)
std::vector<std::string> launched;
int graph_launches = 0;
int null_stream_ops = 0;        // copies and clears outside any stream
int copies = 0;
struct Config {
    dim3 g, b;
    size_t lds;
    void* stream;
} config;
std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> m;  // filled before main
    return m;
}

int failures = 0;
#define EXPECT(c, ...)                    \
    do {                                  \
        if (!(c)) {                       \
            ++failures;                   \
            std::printf("FAILED: %s: ", #c); \
            std::printf(__VA_ARGS__);     \
            std::printf("\n");            \
        }                                 \
    } while (0)
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) {
    config = {g, b, lds, s};
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
    *g = config.g;
    *b = config.b;
    *lds = config.lds;
    *s = config.stream;
    return 0;
}
int hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, void*) {
    launched.push_back(kernels()[f]);
    return 0;
}
int hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (mallocs_left == 0) return 2;  // out of memory
    if (mallocs_left > 0) --mallocs_left;
    *p = std::calloc(n, 1);
    live.insert(*p);
    return 0;
}
int hipFree(void* p) {
    if (p && !live.erase(p)) EXPECT(false, "free of %p, which is no allocation", p);
    std::free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return 0;
}
int hipHostFree(void* p) {
    std::free(p);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* stream) {
    null_stream_ops += stream == nullptr;
    ++copies;
    std::memmove(d, s, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* stream) {
    null_stream_ops += stream == nullptr;
    std::memset(d, v, n);
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
int hipMemset(void* d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = std::malloc(1);
    return 0;
}
int hipStreamDestroy(void* s) {
    std::free(s);
    return 0;
}
int hipStreamSynchronize(void*) { return 0; }
int hipEventCreate(void** e) {
    *e = std::malloc(1);
    return 0;
}
int hipEventDestroy(void* e) {
    std::free(e);
    return 0;
}
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.0f;
    return 0;
}
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
    *g = std::malloc(1);
    return 0;
}
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) {
    *e = std::malloc(1);
    return 0;
}
int hipGraphDestroy(void* g) {
    std::free(g);
    return 0;
}
int hipGraphExecDestroy(void* e) {
    std::free(e);
    return 0;
}
int hipGraphLaunch(void*, void*) {
    ++graph_launches;
    return 0;
}
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256;
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 4;
    return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetSymbolAddress(void** p, const void*) {
    static double scratch[1024];
    *p = scratch;
    return 0;
}
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "stand-in error"; }
}

static sf_ctx* context(int N1, int N2, int N3, int precision) {
    const sf_grid g = {N1, N2, N3, N2 > 1 ? SF_THREE_D : SF_TWO_D};
    const sf_flow f = {14.28, 7.14, 10.0, 1000.0, 0.1, 1.0, 0};
    sf_ctx* c = nullptr;
    const int rc = sf_ctx_create(&g, &f, precision, &c);
    EXPECT(rc == SF_OK, "context: %s", sf_last_error(nullptr));
    if (rc != SF_OK) std::exit(1);
    return c;
}

// An adjoint step whose n-th allocation fails reports it, and so does the next
// one while memory is short, without a launch; with memory back it runs on the
// buffers of a context that never failed.
static void adjoint_memory() {
    size_t whole = 0;
    for (int fail = -1; fail < 24; ++fail) {
        sf_ctx* c = context(24, 12, 16, 8);
        sf_field* f[4];
        for (int i = 0; i < 4; ++i) sf_field_alloc(c, SF_MODAL, i == 2 ? SF_DIRICHLET : SF_NEUMANN, &f[i]);
        launched.clear();
        if (fail >= 0) {
            mallocs_left = fail;
            for (int again = 0; again < 2; ++again) {
                const int rc = sf_step_adjoint(c, f, f);
                EXPECT(rc != SF_OK && launched.empty(), "allocation %d, attempt %d: rc %d, %zu launches", fail, again, rc,
                       launched.size());
            }
            mallocs_left = -1;
        }
        const int rc = sf_step_adjoint(c, f, f);
        EXPECT(rc == SF_OK && !launched.empty(), "allocation %d, memory back: rc %d", fail, rc);
        if (fail < 0) whole = live.size();
        EXPECT(live.size() == whole, "allocation %d: %zu buffers, %zu without a failure", fail, live.size(), whole);
        for (sf_field* x : f) sf_field_free(x);
        sf_ctx_destroy(c);
        EXPECT(live.empty(), "allocation %d: %zu buffers left", fail, live.size());
    }
}

// No kernel runs, so no inner product may return: every call says that its result
// did not arrive, whatever its number (numbers wrap, and no word of the results
// may be taken for one of a call that it does not belong to).
static void inner_product_results() {
    sf_ctx* c = context(24, 1, 16, 8);
    for (int i = 0; i < 1000; ++i) {
        double ke = -1, pe = -1;
        const int rc = sf_energy(c, &ke, &pe);
        EXPECT(rc == SF_ERR_STATE, "call %d: rc %d, energies %g %g", i, rc, ke, pe);
    }
    sf_ctx_destroy(c);
}

// A plan whose tables cannot be allocated is reported, and so is every step until
// they can be: no launch goes without its tables.
static void batch_memory() {
    for (int fail = 0; fail < 8; ++fail) {
        sf_ctx* c[2] = {context(24, 1, 16, 8), context(32, 1, 16, 8)};
        sf_batch* b = nullptr;
        EXPECT(sf_batch_create(c, 2, &b) == SF_OK, "batch: %s", sf_batch_last_error(nullptr));
        if (!b) std::exit(1);
        EXPECT(sf_batch_step(b, 1) == SF_OK, "first step");
        mallocs_left = fail;
        EXPECT(sf_batch_select(b, SF_BATCH_MIXED, SF_BATCH_MIXED) != SF_OK, "allocation %d: select succeeded", fail);
        mallocs_left = 0;
        launched.clear();
        graph_launches = 0;
        for (int again = 0; again < 2; ++again) {
            const int rc = sf_batch_step(b, 1);
            EXPECT(rc != SF_OK && launched.empty() && graph_launches == 0, "allocation %d, step %d: rc %d, %zu launches", fail,
                   again, rc, launched.size());
        }
        mallocs_left = -1;
        EXPECT(sf_batch_step(b, 1) == SF_OK && graph_launches == 1, "allocation %d, memory back", fail);
        sf_batch_destroy(b);
        for (sf_ctx* x : c) sf_ctx_destroy(x);
        EXPECT(live.empty(), "allocation %d: %zu buffers left", fail, live.size());
    }
}

// A network's copies and clears take their turn on its context's stream: what is
// still queued there reads the weights, activations and training pairs that were
// there when it was queued.
static void net_stream() {
    sf_ctx* c = context(24, 1, 16, 4);
    sf_field* f[4];
    for (int i = 0; i < 4; ++i) sf_field_alloc(c, SF_MODAL, i == 2 ? SF_DIRICHLET : SF_NEUMANN, &f[i]);
    null_stream_ops = 0;
    const size_t before = live.size();
    sf_net* n = nullptr;
    EXPECT(sf_net_create(c, 32, 3, 1, &n) == SF_OK, "%s", sf_net_last_error(nullptr));
    if (!n) std::exit(1);
    // parameters, gradient, two moments and mask, two layouts of three layers, partial sums
    EXPECT(live.size() - before == 12, "%zu buffers", live.size() - before);
    auto expect = [&](const char* call) {
        EXPECT(null_stream_ops == 0, "%s: %d outside the stream", call, null_stream_ops);
        null_stream_ops = 0;
    };
    expect("create");
    size_t count = 0;
    sf_net_param_count(n, &count);
    std::vector<float> p(count, 0.5f), q(count);
    sf_net_set_params(n, p.data());
    expect("set_params");
    sf_net_get_params(n, q.data());
    expect("get_params");
    EXPECT(p == q, "parameters");
    sf_net_apply(n, f, f);
    expect("apply");
    std::vector<float> x(2 * 16 * 32), y(2 * 16 * 32);
    sf_net_forward_raw(n, x.data(), 2, y.data());
    expect("forward_raw");
    double loss = 0;
    sf_net_grad_raw(n, x.data(), y.data(), 2, q.data(), &loss);
    expect("grad_raw");
    sf_net_destroy(n);
    for (sf_field* g : f) sf_field_free(g);
    sf_ctx_destroy(c);
}

// A raw forward pass whose n-th allocation of twelve fails reports it, and so does
// the next one while memory is short, without a launch; with memory back it runs.
static void net_memory() {
    for (int fail = 0; fail < 12; ++fail) {
        sf_ctx* c = context(24, 1, 16, 4);
        sf_net* n = nullptr;
        EXPECT(sf_net_create(c, 32, 3, 1, &n) == SF_OK, "%s", sf_net_last_error(nullptr));
        if (!n) std::exit(1);
        std::vector<float> x(4 * 16 * 32), y(4 * 16 * 32);
        EXPECT(sf_net_forward_raw(n, x.data(), 2, y.data()) == SF_OK, "two profiles");
        launched.clear();
        mallocs_left = fail;
        for (int again = 0; again < 2; ++again) {
            const int rc = sf_net_forward_raw(n, x.data(), 4, y.data());
            EXPECT(rc != SF_OK && launched.empty(), "allocation %d, attempt %d: rc %d, %zu launches", fail, again, rc,
                   launched.size());
        }
        mallocs_left = -1;
        EXPECT(sf_net_forward_raw(n, x.data(), 4, y.data()) == SF_OK, "allocation %d, memory back", fail);
        sf_net_destroy(n);
        sf_ctx_destroy(c);
        EXPECT(live.empty(), "allocation %d: %zu buffers left", fail, live.size());
    }
}

// A new background or new flow parameters reach the device in one copy, and the
// background is read back from there.
static void table_copies() {
    for (int precision = 4; precision <= 8; precision += 4) {
        sf_ctx* c = context(24, 12, 100, precision);
        std::vector<double> u(100), s(100), back(100);
        for (int j = 0; j < 100; ++j) {
            u[j] = j / 64.0;  // exact in either precision
            s[j] = 1 + j / 128.0;
        }
        copies = 0;
        EXPECT(sf_set_background(c, u.data(), s.data()) == SF_OK && copies == 1, "set_background: %d copies", copies);
        const sf_flow f = {14.28, 7.14, 12.0, 500.0, 0.2, 2.0, 1};
        copies = 0;
        EXPECT(sf_set_flow(c, &f) == SF_OK && copies == 1, "set_flow: %d copies", copies);
        EXPECT(sf_get_background(c, back.data()) == SF_OK && back == u, "the background that was set");
        EXPECT(sf_set_flow(c, &f) == SF_OK && sf_get_background(c, back.data()) == SF_OK && back == u,
               "the background after set_flow");
        sf_ctx_destroy(c);
    }
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> scenarios = {{"adjoint_memory", adjoint_memory},
                                                         {"inner_product_results", inner_product_results},
                                                         {"batch_memory", batch_memory},
                                                         {"net_stream", net_stream},
                                                         {"net_memory", net_memory},
                                                         {"table_copies", table_copies}};
    const auto s = argc == 2 ? scenarios.find(argv[1]) : scenarios.end();
    if (s == scenarios.end()) {
        std::printf("unknown scenario\n");
        return 2;
    }
    s->second();
    if (failures) return 1;
    std::printf("ok\n");
    return 0;
}
