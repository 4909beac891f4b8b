// Steps, graphs and portions of a stack model on a HIP runtime that does everything at once and keeps count (tests/test_host_steps.py): a captured graph is the list of its launches, launches
// are stand-ins that move tokens and positions as the kernels do.  A row's first number is the token that it was embedded from, all the way to the end of the stack.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "stack_model.hpp"

namespace {
struct Launch {
    std::string name;
    std::function<void()> f;
};
typedef std::vector<Launch> Graph;
Graph *g_capture = nullptr;
std::vector<size_t> g_made;          // launches of every graph that was instantiated, or should have been
std::vector<size_t> g_replayed;      // and of every one that was launched
std::vector<std::string> g_done;     // what ran, in order; "malloc" and "free" among it
size_t g_largest_graph = ~size_t(0); // launches of the largest graph that instantiates
size_t g_largest_block = ~size_t(0); // bytes
hipError_t g_last_error = hipSuccess;
bool g_follows = true, g_narrow = true;

void launch(const char *name, std::function<void()> f) {
    if (g_capture) return g_capture->push_back({name, f});
    g_done.push_back(name), f();
}
size_t count(const char *name) {
    size_t n = 0;
    for (const std::string &s : g_done) n += s == name;
    return n;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    *p = nullptr;
    g_done.push_back("malloc");
    if (n > g_largest_block) return g_last_error = hipErrorOutOfMemory;
    *p = malloc(n + 64), memset(*p, 0, n + 64);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void *p) { return g_done.push_back("free"), free(p), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = g_last_error;
    return g_last_error = hipSuccess, e;
}
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return g_capture = new Graph, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = reinterpret_cast<hipGraph_t>(g_capture);
    return g_capture = nullptr, hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t g, hipGraphNode_t *, size_t *n) { return *n = reinterpret_cast<Graph *>(g)->size(), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    const Graph &of = *reinterpret_cast<Graph *>(g);
    g_made.push_back(of.size());
    if (of.size() > g_largest_graph) return g_last_error = hipErrorOutOfMemory;
    return *e = reinterpret_cast<hipGraphExec_t>(new Graph(of)), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    const Graph &of = *reinterpret_cast<Graph *>(e);
    g_replayed.push_back(of.size());
    for (const Launch &l : of) launch(l.name.c_str(), l.f);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return delete reinterpret_cast<Graph *>(e), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return delete reinterpret_cast<Graph *>(g), hipSuccess; }

size_t bitnet_hip_gqa_scratch_bytes(size_t, size_t, size_t, size_t) { return 256; }
size_t bitnet_hip_gqa_prefill_scratch_bytes(const bitnet_hip_gqa *, size_t n_ctx, size_t nq) { return n_ctx > nq ? n_ctx * 16384 : 0; }
int bitnet_hip_gqa_supported(size_t, size_t) { return g_narrow; }
size_t bitnet_hip_gqa_out_records(const bitnet_hip_gqa *, size_t) { return 4; }
size_t bitnet_hip_gqa_project_records(const bitnet_hip_gqa *, size_t) { return 12; }
int bitnet_hip_embedding_follows(const bitnet_hip_embedding *) { return g_follows; }
int bitnet_hip_sequence_update_dev(int32_t *history, size_t first, size_t n, const int32_t *tokens, int32_t *n_forced, int32_t forced, int32_t *pos, int32_t position, const float *, float *,
                                   size_t, void *) {
    launch("update", [=] {
        if (history)
            for (size_t i = 0; i < n; ++i) history[first + i] = tokens ? tokens[i] : 0;
        if (n_forced) *n_forced = forced;
        if (pos) *pos = position;
    });
    return 0;
}
int bitnet_hip_embed_bf16_dev(const uint16_t *, size_t, const int32_t *tokens, const int32_t *pos, size_t n, size_t width, size_t, float, float *out, void *) {
    launch("embed", [=] {
        for (size_t i = 0; i < n; ++i) out[i * width] = (float)tokens[*pos + i];
    });
    return 0;
}
int bitnet_hip_advance_pos_dev(int32_t *pos, void *) { return launch("advance", [=] { ++*pos; }), 0; }
int bitnet_hip_dense_gemv_dev(const bitnet_hip_vector_input *in, const uint16_t *, size_t, size_t, size_t, const float *, int, int, size_t, float *, size_t, size_t, size_t, size_t,
                              const bitnet_hip_latent_rows *, int, const bitnet_hip_epilogue *, void *) {
    const float *x = in->x;
    float *out = in->x_out;
    launch("gemv", [=] {
        if (out) *out = *x;
    });
    return 0;
}
static void logits(const bitnet_hip_vector_input *in, int32_t *pos, int32_t *history, const int32_t *n_forced, float *next) {
    const float *x = in->x;
    float *out = in->x_out;
    launch(next ? "logits and embed" : "logits", [=] {
        if (out) *out = *x;
        if (++*pos >= *n_forced) history[*pos] = 1000 + *pos;
        if (next) *next = (float)history[*pos];
    });
}
int bitnet_hip_dense_logits_dev(const bitnet_hip_vector_input *in, const uint16_t *, size_t, size_t, size_t, float *, void *, int32_t *, int32_t *pos, int32_t *history, const int32_t *n_forced,
                                void *) {
    return logits(in, pos, history, n_forced, nullptr), 0;
}
int bitnet_hip_dense_logits_embed_dev(const bitnet_hip_vector_input *in, const uint16_t *, size_t, size_t, size_t, float *, void *, int32_t *, int32_t *pos, int32_t *history,
                                      const int32_t *n_forced, const bitnet_hip_embedding *next, void *) {
    return logits(in, pos, history, n_forced, next->out), 0;
}
int bitnet_hip_gqa_step_dev(const bitnet_hip_gqa *, const float *, const int32_t *, float *, void *) { return launch("step", [] {}), 0; }
int bitnet_hip_gqa_rows_dev(const bitnet_hip_gqa *, void *, size_t, int, int, const int32_t *, size_t, void *, size_t, void *) { return launch("rows", [] {}), 0; }
int bitnet_hip_gqa_any_dev(const bitnet_hip_gqa *, const void *, size_t, int, int, const int32_t *, size_t, size_t, float *, void *) { return launch("any", [] {}), 0; }
int bitnet_hip_gqa_merge_dev(const bitnet_hip_gqa *, const int32_t *, size_t, size_t, const float *, void *, size_t, int, void *) { return launch("merge", [] {}), 0; }
int bitnet_hip_gqa_project_dev(const bitnet_hip_gqa *, const int32_t *, size_t, const float *, const uint16_t *, size_t, size_t, size_t, const float *, float *, void *) {
    return launch("project", [] {}), 0;
}
int bitnet_hip_gqa_prefill_scratch_dev(const bitnet_hip_gqa *, const uint16_t *, size_t, size_t, size_t, uint16_t *, size_t, float *, size_t, void *) { return launch("prefill", [] {}), 0; }
}

using bitnet_host::LayerSpec;

#define CHECK(x) \
    if (!(x)) return printf("%s:%d: %s\n", __FILE__, __LINE__, #x), 1

struct Model : bitnet_host::StackModel {
    static bitnet_host::StackSpec spec(int dim, int heads) {
        bitnet_host::StackSpec s;
        s.width = 64, s.vocab = 100, s.layers.resize(2);
        for (LayerSpec &l : s.layers) l.mixer = LayerSpec::Attention, l.attention.heads = heads, l.attention.kv_heads = 1, l.attention.dim = l.attention.vdim = dim;
        return s;
    }
    int rc = 0;
    std::vector<int32_t> tokens;
    Model(int max_pos, int dim = 32, int heads = 2) : StackModel(spec(dim, heads), false, max_pos) {
        std::vector<uint16_t> zeros(64 * 64 * 64);
        for (int i = 0; i < 2; ++i) {
            bitnet_host::StackLayerWeights w;
            w.norm1.resize(64);
            w.q = w.k = w.v = w.o = zeros.data();
            rc |= set_layer(i, w);
        }
        bitnet_host::StackGlobalWeights g;
        g.embed = g.head = zeros.data(), g.final_norm.resize(64);
        rc |= dead() ? 1 : set_globals(g);
        for (int i = 0; i + 2 < max_pos; ++i) tokens.push_back(10 + i % 90);
        g_made.clear(), g_replayed.clear(), g_done.clear();
    }
    // a new sequence of n fed tokens, the first of them as a prompt
    int start(int n, int prompt) { return reset() || feed(tokens.data(), n) || (prompt > 0 && prefill(prompt, false, 0, nullptr)); }
    // the token whose row last_hidden gives; -1: none
    int last() {
        std::vector<float> row(64);
        return last_hidden(row.data()) == 0 ? (int)row[0] : -1;
    }
};
#define START(m) CHECK(!(m).dead() && (m).rc == 0)

// last_hidden gives the row of the position that ran last: whatever ran it, and however often its graph was captured before
int last_row() {
    for (bool follows : {true, false}) {
        g_follows = follows;
        Model m(600);
        START(m);
        for (int again = 0; again < 3; ++again) {
            CHECK(m.start(40, 4) == 0 && m.last() == m.tokens[3]);
            CHECK(m.prepare_graphs(true) == 0 && m.prepare_graphs(false) == 0 && m.last() == m.tokens[3]);
            CHECK(m.run(1, true, true, nullptr) == 0 && m.last() == m.tokens[4]);
            CHECK(m.run(9, true, true, nullptr) == 0 && m.last() == m.tokens[13]);
            CHECK(m.run(2, false, true, nullptr) == 0 && m.last() == -1);
            CHECK(m.run(1, true, false, nullptr) == 0 && m.last() == m.tokens[16]);
            CHECK(m.run(0, true, true, nullptr) == 0 && m.last() == m.tokens[16]);
            CHECK(m.prefill(3, true, 0, nullptr) == 0 && m.last() == m.tokens[19]);
            CHECK(m.run(8, true, true, nullptr) == 0 && m.last() == m.tokens[27]);
            CHECK(m.reset() == 0 && m.last() == -1 && m.feed(m.tokens.data(), 9) == 0 && m.run(5, true, true, nullptr) == 0 && m.last() == m.tokens[4]);
        }
    }
    return 0;
}

// several steps make one graph where as many are asked for and all of one form; nothing is captured that is not launched
int chain_use() {
    Model m(600);
    START(m);
    CHECK(m.start(590, 4) == 0);
    for (int n : {1, 2, 3}) CHECK(m.run(n, true, true, nullptr) == 0 && g_made.size() == 1);
    const size_t one = g_made[0], four = 4 * one - 3;  // (three embeddings go with the logits ahead of them)
    g_replayed.clear();
    CHECK(m.run(9, true, true, nullptr) == 0 && g_made.size() == 2 && g_made[1] == four && g_replayed == (std::vector<size_t>{four, four, one}) && m.last_graph_steps() == 4);
    CHECK(m.start(590, 254) == 0);  // behind two steps the next form
    g_made.clear(), g_replayed.clear();
    CHECK(m.run(5, true, true, nullptr) == 0 && g_made == std::vector<size_t>{one} && g_replayed == std::vector<size_t>(5, one));
    CHECK(m.run(4, false, true, nullptr) == 0 && g_replayed.size() == 9);
    g_follows = false;
    Model alone(600);
    START(alone);
    CHECK(alone.start(590, 4) == 0 && alone.run(20, true, true, nullptr) == 0 && g_made.size() == 1 && g_replayed == std::vector<size_t>(20, g_made[0]) && alone.last_graph_steps() == 1);
    return 0;
}

// a chain that cannot be made is tried once, its error is nobody's, and the steps run one by one
int chain_refused() {
    Model m(600);
    START(m);
    g_largest_graph = 8;
    for (int again = 0; again < 3; ++again) {
        CHECK(m.start(200, 4) == 0 && m.run(20, true, true, nullptr) == 0 && m.position() == 24 && m.last() == m.tokens[23]);
        CHECK(g_made.size() == 2 && g_made[0] <= 8 && g_made[1] > 8 && m.error().empty() && g_last_error == hipSuccess);
        for (size_t n : g_replayed) CHECK(n == g_made[0]);
    }
    return 0;
}

// behind prepare_graphs no run captures anything, wherever it starts and however long it is
int prepared() {
    for (int max_pos : {3, 40, 130, 600}) {
        Model m(max_pos);
        START(m);
        CHECK(m.prepare_graphs(true) == 0 && m.prepare_graphs(false) == 0);
        const size_t made = g_made.size();
        for (int from = 0; from < max_pos - 1; from += 7)
            for (int n : {1, 2, 4, 9, max_pos - 1 - from}) {
                if (from + n > max_pos - 2) continue;
                CHECK(m.start(max_pos - 2, from) == 0 && m.run(n, true, true, nullptr) == 0 && m.last() == m.tokens[(size_t)(from + n - 1)]);
                CHECK(m.start(max_pos - 2, from) == 0 && m.run(n, false, true, nullptr) == 0);
            }
        CHECK(g_made.size() == made);
        for (size_t a : g_made) CHECK(max_pos > 4 || a <= g_made[0]);  // no chain where no sequence has room for one
    }
    return 0;
}

// the output product merges the records, whichever kernel has left them
int wide_heads() {
    for (bool narrow : {true, false}) {
        g_narrow = narrow;
        Model m(2000, narrow ? 32 : 288);
        START(m);
        for (int at : {0, 127, 128, 500, 900, 1500, 1600}) {
            CHECK(m.reset() == 0 && m.feed(m.tokens.data(), at + 2) == 0 && (at == 0 || m.prefill(at, false, 0, nullptr) == 0));
            g_done.clear();
            CHECK(m.run(1, true, true, nullptr) == 0 && count(narrow ? "step" : "any") == 2 && count(narrow ? "any" : "step") == 0);
            CHECK(count("project") == (at < 1536 ? 2 : 0) && count("merge") == (at < 1536 ? 0 : 2));
        }
    }
    return 0;
}

// everything that a portion needs is there ahead of its first launch; where it cannot be had, nothing has run
int portion_room() {
    Model m(4000);
    START(m);
    for (int n : {100, 300, 64, 700, 20, 1000}) {
        const int p = m.position();
        CHECK(m.feed(m.tokens.data() + p, n) == 0);
        g_done.clear();
        CHECK(m.prefill(n, false, 0, nullptr) == 0 && count("prefill") == 2);
        bool launched = false;
        for (const std::string &s : g_done) {
            launched = launched || (s != "malloc" && s != "free");
            CHECK(!launched || (s != "malloc" && s != "free"));
        }
    }
    g_largest_block = 45 << 20;  // (the records of 2184 + 900 positions take more)
    const int p = m.position();
    CHECK(m.feed(m.tokens.data() + p, 900) == 0);
    g_done.clear();
    CHECK(m.prefill(900, false, 0, nullptr) != 0 && m.position() == p && g_last_error == hipSuccess);
    for (const std::string &s : g_done) CHECK(s == "malloc" || s == "free");
    g_largest_block = ~size_t(0);
    CHECK(m.prefill(900, false, 0, nullptr) == 0 && m.position() == p + 900 && m.last() == m.tokens[(size_t)p + 899]);
    return 0;
}

// nine to twelve records of many columns are merged by a launch of their own, fewer by the product, and no form of a step is made that is another's twin
int many_columns() {
    Model m(2000, 128, 28);
    START(m);
    CHECK(m.prepare_graphs(true) == 0 && g_made.size() == 8);  // forms of 2, 4 and 8 records and of a launch, one step and several
    for (int at : {0, 500, 1023, 1024, 1500, 1600}) {
        CHECK(m.reset() == 0 && m.feed(m.tokens.data(), at + 2) == 0 && (at == 0 || m.prefill(at, false, 0, nullptr) == 0));
        g_done.clear();
        CHECK(m.run(1, true, true, nullptr) == 0 && count("step") == 2 && count("project") == (at < 1024 ? 2 : 0) && count("merge") == (at < 1024 ? 0 : 2));
    }
    return 0;
}

int main(int argc, char **argv) {
    const std::map<std::string, int (*)()> cases = {
        {"last_row", last_row},
        {"chain_use", chain_use},
        {"chain_refused", chain_refused},
        {"prepared", prepared},
        {"wide_heads", wide_heads},
        {"portion_room", portion_room},
        {"many_columns", many_columns},
    };
    const auto it = cases.find(argc > 1 ? argv[1] : "");
    CHECK(it != cases.end());
    return it->second();
}
