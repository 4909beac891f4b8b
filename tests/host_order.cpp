// A HIP runtime of promises for the host code (tests/test_host_order.py): work is done as late as HIP allows it -- a stream's when somebody waits for that stream, the null stream's when a
// blocking copy follows it -- so that whatever relies on an order that nothing establishes is seen.  The kernels are stand-ins that leave a mark.  A blocking copy of rows (hipMemcpy2D)
// does not wait for the null stream's fills here, although it should: under rocprofv3's kernel trace the runtime's has overtaken a hipMemset of the same memory.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <vector>

#include "decoder.hpp"
#include "stack_model.hpp"

namespace {
typedef std::deque<std::function<void()>> Queue;
Queue g_null;
std::vector<Queue *> g_streams;
Queue &queue(void *s) { return s ? *static_cast<Queue *>(s) : g_null; }
void run(Queue &q) {
    while (!q.empty()) {
        auto f = std::move(q.front());
        q.pop_front();
        f();
    }
}
void run_all() {
    run(g_null);
    for (Queue *q : g_streams) run(*q);
}
std::vector<std::pair<const uint8_t *, size_t>> g_memory;
uint32_t g_clamped = 0, g_taken = 0;  // the device's count, and what of it f16_saturations_dev has given out
int g_clamping = 0;                   // the next product clamps, and somebody else takes the count at once
uint32_t take() {
    const uint32_t n = g_clamped - g_taken;
    g_taken = g_clamped;
    return n;
}
void product(void *s) {
    if (g_clamping == 0) return;
    --g_clamping;
    queue(s).push_back([] { ++g_clamped, take(); });
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    *p = malloc(n + 64), memset(*p, 0x5a, n + 64);
    return g_memory.push_back({(const uint8_t *)*p, n}), hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void *p) {
    run_all();
    for (auto &m : g_memory)
        if (m.first == p) m = {nullptr, 0};
    return free(p), hipSuccess;
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipDeviceSynchronize() { return run_all(), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    g_streams.push_back(new Queue);
    return *s = reinterpret_cast<hipStream_t>(g_streams.back()), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return run(queue(s)), hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return g_null.push_back([=] { memset(p, v, n); }), hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) { return queue(s).push_back([=] { memset(p, v, n); }), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return run(g_null), memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpy2D(void *d, size_t ldd, const void *s, size_t lds, size_t n, size_t rows, hipMemcpyKind) {
    for (size_t r = 0; r < rows; ++r) memcpy((char *)d + r * ldd, (const char *)s + r * lds, n);
    return hipSuccess;
}

size_t bitnet_hip_qact_bytes(size_t) { return 64; }
size_t bitnet_hip_qact_stats_bytes(size_t) { return 64; }
size_t bitnet_hip_attention_scratch_bytes(size_t, size_t) { return 64; }
size_t bitnet_hip_attention_prefill_workspace_bytes(size_t, size_t, size_t) { return 64; }
size_t bitnet_hip_matmul_workspace_bytes(size_t, size_t, int) { return 64; }
int bitnet_hip_matmul_f16_supported(bitnet_hip_weights_t) { return 1; }
int bitnet_hip_weights_info(bitnet_hip_weights_t, size_t *rows, size_t *cols, size_t *bytes) {
    if (rows) *rows = 512;
    if (cols) *cols = 512;
    if (bytes) *bytes = 512 * 128;
    return 0;
}
int bitnet_hip_weights_upload_qk256(const uint8_t *, size_t, size_t, size_t, size_t, bitnet_hip_weights_t *h) { return *h = 1, 0; }
int bitnet_hip_weights_concat(const bitnet_hip_weights_t *, size_t, int, bitnet_hip_weights_t *h) { return *h = 1, 0; }
int bitnet_hip_sequence_update_dev(int32_t *history, size_t first, size_t n, const int32_t *tokens, int32_t *n_forced, int32_t forced, int32_t *pos, int32_t position, const float *row,
                                   float *x, size_t width, void *s) {
    queue(s).push_back([=] {
        if (history)
            for (size_t i = 0; i < n; ++i) history[first + i] = tokens ? tokens[i] : 0;
        if (n_forced) *n_forced = forced;
        if (pos) *pos = position;
        if (x) memcpy(x, row, width * 4);
    });
    return 0;
}
int bitnet_hip_attention_prefill_flags_dev(const float *, const float *, const float *, void *k, void *v, size_t, size_t, size_t, size_t, size_t, void *, size_t, void *, int, void *s) {
    queue(s).push_back([=] { *(float *)k = 7.f, *(float *)v = 8.f; });
    return 0;
}
int bitnet_hip_attention_prefill_dev(const float *, const float *, const float *, float *k, float *v, size_t, size_t, size_t, size_t, size_t, void *, size_t, float *, void *s) {
    queue(s).push_back([=] { *k = 7.f, *v = 8.f; });
    return 0;
}
int bitnet_hip_matmul_f16_dev(bitnet_hip_weights_t, const void *, size_t, const float *, size_t, const float *, float, float *, const float *, int, void *, const float *, float *, void *s) {
    return product(s), 0;
}
int bitnet_hip_advance_pos_dev(int32_t *pos, void *s) { return queue(s).push_back([=] { ++*pos; }), 0; }
int bitnet_hip_f16_saturations_dev(uint32_t *count, void *s) {
    queue(s).push_back([=] {
        const uint32_t n = take();
        if (count) *count = n;
    });
    return 0;
}
int bitnet_hip_f16_saturations_total_dev(uint32_t *total, void *s) { return queue(s).push_back([=] { *total = g_clamped; }), 0; }
}

using bitnet_host::Decoder;

#define CHECK(x) \
    if (!(x)) return printf("%s:%d: %s\n", __FILE__, __LINE__, #x), 1

// a matrix of 6 rows lies on the device, with zeros behind its columns
bool arrived(const std::vector<uint16_t> &w, size_t cols, size_t ld) {
    std::vector<uint16_t> want(6 * ld, 0);
    for (size_t r = 0; r < 6; ++r) memcpy(&want[r * ld], &w[r * cols], cols * 2);
    for (const auto &m : g_memory)
        if (m.second == 6 * ld * 2 && !memcmp(m.first, want.data(), m.second)) return true;
    return false;
}

int matrices() {
    for (int width : {40, 64, 200}) {
        bitnet_host::StackSpec spec;
        spec.width = width, spec.vocab = 6, spec.layers.resize(1);
        auto &layer = spec.layers[0];
        layer.mixer = bitnet_host::LayerSpec::Linear;
        layer.linear.heads = 1, layer.linear.dim = layer.linear.vdim = 6, layer.linear.decay = {0.5};
        bitnet_host::StackModel m(spec, false, 16);
        CHECK(!m.dead());
        std::vector<uint16_t> w(6 * width), head(6 * width);
        for (size_t i = 0; i < w.size(); ++i) w[i] = (uint16_t)(i + 1), head[i] = (uint16_t)(i + 2000);
        bitnet_host::StackGlobalWeights g;
        g.embed = w.data(), g.head = head.data(), g.final_norm.resize(width);
        CHECK(m.set_globals(g) == 0);
        hipDeviceSynchronize();
        CHECK(arrived(w, width, (width + 63) / 64 * 64) && arrived(head, width, (width + 63) / 64 * 64));
    }
    return 0;
}

int main(int argc, char **argv) {
    if (argc > 1 && !strcmp(argv[1], "matrices")) return matrices();
    bitnet_host::Config c;
    c.hidden = 512, c.n_layers = 2, c.n_heads = 4, c.n_kv_heads = 1, c.head_dim = 128, c.ffn = 512, c.vocab = 64, c.max_pos = 128, c.eps = 1e-5f, c.rope_theta = 1e4f;
    std::vector<uint8_t> zeros(1 << 20);
    const float *f = reinterpret_cast<const float *>(zeros.data());
    const int32_t tokens[3] = {11, 12, 13};
    Decoder d(c);
    CHECK(!d.dead());
    for (int l = 0; l < c.n_layers; ++l) {
        const uint8_t *z = zeros.data();
        CHECK(d.set_layer_qk256(l, bitnet_host::LayerWeightsQk256{f, f, z, z, z, z, z, z, z}) == 0);
    }
    CHECK(d.set_globals(reinterpret_cast<const uint16_t *>(zeros.data()), f) == 0);
    const char *what = argc > 1 ? argv[1] : "";
    auto prompt = [&] { return d.feed(tokens, 3) || d.prefill(3, false, 2, nullptr); };
    if (!strcmp(what, "cache_type")) {  // the caches are clear ahead of the prompt that fills them, whichever stream did it
        for (bool f16 : {true, false, true}) {
            CHECK(d.reset() == 0 && d.set_kv_f16(f16) == 0 && prompt() == 0);
            hipDeviceSynchronize();
            for (int l = 0; l < c.n_layers; ++l) {
                uint64_t h[4];
                void *p[4];
                d.layer_objects(l, h, p);
                CHECK(*(float *)p[2] == 7.f && *(float *)p[3] == 8.f && ((float *)p[2])[1] == 0.f && ((float *)p[3])[1] == 0.f);
            }
        }
    } else if (!strcmp(what, "objects")) {  // what is handed out holds what the calls before have put there, and so it stays
        uint64_t h[4];
        void *g[7], *p[4];
        CHECK(d.reset() == 0 && d.feed(tokens, 2) == 0);
        d.global_objects(g);
        const int32_t *history = (int32_t *)g[4];
        int32_t *pos = (int32_t *)g[5];
        CHECK(history[0] == 11 && history[1] == 12 && *pos == 0);
        CHECK(d.feed(tokens + 2, 1) == 0 && history[2] == 13);
        CHECK(d.prefill(3, false, 2, nullptr) == 0 && *pos == 3 && d.position() == 3);
        *pos = 2;
        CHECK(d.position() == 2);
        CHECK(d.reset() == 0 && *pos == 0 && history[0] == 0 && d.set_kv_f16(true) == 0);
        d.layer_objects(1, h, p);
        CHECK(*(float *)p[2] == 0.f && *(float *)p[3] == 0.f);
    } else if (!strcmp(what, "clamps")) {  // a clamp is not lost to a sequence beside this one that takes the count meanwhile
        for (int n : {0, 1, 0, 2}) {
            const int before = d.saturation_fallbacks();
            g_clamping = n;
            CHECK(d.reset() == 0 && prompt() == 0 && d.position() == 3);
            CHECK(d.saturation_fallbacks() == before + (n > 0));
            bitnet_hip_f16_saturations_dev(nullptr, d.stream());
        }
    } else {
        CHECK(!"a case of this name");
    }
    return 0;
}
