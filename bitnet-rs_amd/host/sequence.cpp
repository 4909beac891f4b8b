// sequence.cpp -- see sequence.hpp.
#include "sequence.hpp"

#include <cstdio>
#include <cstring>

namespace bitnet_host {

int Sequence::fail_arg(const char *what) {
    err_ = what;
    return BITNET_HIP_ERR_INVALID_ARGUMENT;
}

int Sequence::fail(const char *what) {
    const char *e = bitnet_hip_get_last_error();
    err_ = std::string(what) + ": " + (e ? e : "error");
    return BITNET_HIP_ERR_EXECUTION;
}

int Sequence::init_sequence(int vocab, int width, int max_pos) {
    vocab_ = vocab, width_ = width, max_pos_ = max_pos;
    BCHK(bitnet_hip_init(-1));
    hipStream_t s;
    HCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    stream_ = s;
    HCHK(hipMalloc((void **)&logits_, (size_t)vocab * 4));
    HCHK(hipMalloc((void **)&pos_, 4));
    HCHK(hipMalloc((void **)&n_forced_, 4));
    HCHK(hipMalloc((void **)&token_, 4));
    HCHK(hipMalloc((void **)&history_, ((size_t)max_pos + 2) * 4));
    HCHK(hipHostMalloc((void **)&pinned_, ((size_t)kCounts + kStaged) * 4, hipHostMallocCoherent));
    HCHK(hipEventCreate(&begin_.e));
    HCHK(hipEventCreate(&end_.e));
    return 0;
}

Sequence::~Sequence() {
    drop_graphs();
    for (void *p : {(void *)logits_, (void *)pos_, (void *)n_forced_, (void *)history_, (void *)token_})
        if (p) hipFree(p);
    if (pinned_) hipHostFree(pinned_);
    if (stream_) hipStreamDestroy((hipStream_t)stream_);
}

void Sequence::drop_graphs() {
    for (int i = 0; i < 2 * kForms; ++i) {
        if (graph_exec_[i]) hipGraphExecDestroy((hipGraphExec_t)graph_exec_[i]);
        if (graph_[i]) hipGraphDestroy((hipGraph_t)graph_[i]);
        graph_exec_[i] = graph_[i] = nullptr;
    }
    for (int i = 0; i < kForms; ++i) {
        if (chain_exec_[i]) hipGraphExecDestroy((hipGraphExec_t)chain_exec_[i]);
        if (chain_graph_[i]) hipGraphDestroy((hipGraph_t)chain_graph_[i]);
        chain_exec_[i] = chain_graph_[i] = nullptr, chain_refused_[i] = false;
    }
    chain_steps_ = 0;
}

int Sequence::settle() {
    HCHK(hipStreamSynchronize((hipStream_t)stream_));
    staged_ = false;
    return 0;
}

// the tokens, position and row a step reads, in stream order: nothing here waits for the device
int Sequence::update(int first, int n, const int32_t *tokens, bool forced, int pos, const float *row, float *x) {
    host_pos_ = pos >= 0 ? -1 : host_pos_;
    BCHK(bitnet_hip_sequence_update_dev(n > 0 ? history_ : nullptr, (size_t)first, (size_t)n, n > 0 ? tokens : nullptr, forced ? n_forced_ : nullptr, host_forced_, pos >= 0 ? pos_ : nullptr, pos, row, x,
                                        x ? (size_t)width_ : 0, stream_));
    if (pos >= 0) moved_to(pos);
    return 0;
}

int Sequence::reset() {
    host_forced_ = 0;
    if (int rc = update(0, max_pos_ + 2, nullptr, true, 0)) return rc;
    if (int rc = clear_state()) return rc;
    return exposed_ ? settle() : 0;
}

int Sequence::feed(const int32_t *tokens, int n) {
    const int p = position();
    if (p < 0) return BITNET_HIP_ERR_GPU;
    const int base = p > host_forced_ ? p : host_forced_;
    if (n < 0 || (n > 0 && !tokens)) return fail_arg("feed: null tokens");
    for (int i = 0; i < n; ++i)
        if (tokens[i] < 0 || tokens[i] >= vocab_) {  // TransformerModel::embed's index_select fails on it (T:1390-1426)
            char b[96];
            snprintf(b, sizeof(b), "token id %d out of range [0, %d)", tokens[i], vocab_);
            return fail_arg(b);
        }
    if (base + n > max_pos_) return fail_arg("KV cache overflow");  // T:1190-1194
    if (staged_)
        if (int rc = settle()) return rc;
    for (int i = 0; i == 0 || i < n; i += kStaged) {
        const int part = n - i < kStaged ? n - i : kStaged;
        if (i > 0)
            if (int rc = settle()) return rc;
        if (part > 0) memcpy(pinned_ + kCounts, tokens + i, (size_t)part * 4);
        host_forced_ = base + i + part;
        if (int rc = update(base + i, part, pinned_ + kCounts, true, -1)) return rc;
        staged_ = true;
    }
    return exposed_ ? settle() : 0;
}

int Sequence::position() {
    if (host_pos_ >= 0) return host_pos_;
    int p = -1;
    if (settle() != 0 || hipMemcpy(&p, pos_, 4, hipMemcpyDeviceToHost) != hipSuccess) {
        err_ = "position readback failed";
        return -1;
    }
    moved_to(p);
    return p;
}

int Sequence::history(int32_t *out, int n) {
    if (!out || n < 0 || n > max_pos_ + 2) return fail_arg("history: n out of range");
    if (int rc = settle()) return rc;
    HCHK(hipMemcpy(out, history_, (size_t)n * 4, hipMemcpyDeviceToHost));
    return 0;
}

int Sequence::last_logits(float *out) {
    HCHK(hipMemcpy(out, logits_, (size_t)vocab_ * 4, hipMemcpyDeviceToHost));
    return 0;
}

int Sequence::prepare_graphs(bool with_logits) {
    if (!ready()) return fail_arg("model globals not set");
    std::vector<int> forms;
    for (int pos = 0; pos + 1 < max_pos_; ++pos) forms.push_back(form_at(pos));
    return make_graphs(forms, with_logits, true);
}

// what steps of these forms, one behind the other, are launched with; any: from wherever a run may start among them, and however far it may go
int Sequence::make_graphs(const std::vector<int> &forms, bool with_logits, bool any) {
    const int n = (int)forms.size();
    for (int i = 0, k; i < n; i += k) {
        if (int rc = ensure_graph(with_logits, forms[(size_t)i])) return rc;
        k = with_logits ? steps_together(&forms[(size_t)i], n - i) : 1;
        if (any) k = 1;
    }
    return 0;
}

int Sequence::ensure_graph(bool with_logits, int form) {
    const int gi = 2 * form + (with_logits ? 1 : 0);
    if (graph_exec_[gi]) return 0;
    hipStream_t s = (hipStream_t)stream_;
    hipGraph_t g = nullptr;
    HCHK(hipStreamBeginCapture(s, hipStreamCaptureModeGlobal));
    const int rc = step(with_logits, form);
    const hipError_t e = hipStreamEndCapture(s, &g);
    if (rc != 0) {
        if (g) hipGraphDestroy(g);
        return rc;
    }
    HCHK(e);
    hipGraphExec_t ex = nullptr;
    HCHK(hipGraphInstantiate(&ex, g, nullptr, nullptr, 0));
    graph_[gi] = g;
    graph_exec_[gi] = ex;
    if (with_logits && !chain_steps_) {
        size_t nodes = 0;
        HCHK(hipGraphGetNodes(g, nullptr, &nodes));
        const int fit = nodes ? (int)(kChainNodes / nodes) : 1;
        chain_steps_ = !chains() || fit < 1 ? 1 : fit < kChainMost ? fit : kChainMost;
    }
    return 0;
}

int Sequence::steps_together(const int *forms, int n) {
    if (chain_steps_ < 2 || chain_steps_ > n) return 1;
    for (int k = 1; k < chain_steps_; ++k)
        if (forms[k] != forms[0]) return 1;
    if (chain_refused_[forms[0]]) return 1;
    const std::string err = err_;
    if (ensure_chain(forms[0]) == 0) return chain_steps_;
    chain_refused_[forms[0]] = true;  // (steps one by one do the same: nobody's error)
    (void)hipGetLastError();
    err_ = err;
    return 1;
}

int Sequence::ensure_chain(int form) {
    if (chain_exec_[form]) return 0;
    hipStream_t s = (hipStream_t)stream_;
    hipGraph_t g = nullptr;
    HCHK(hipStreamBeginCapture(s, hipStreamCaptureModeGlobal));
    int rc = 0;
    for (int i = 0; i < chain_steps_ && rc == 0; ++i) {
        follows_ = i > 0, followed_ = i + 1 < chain_steps_;
        rc = step(true, form);
    }
    follows_ = followed_ = false;
    const hipError_t e = hipStreamEndCapture(s, &g);
    if (rc != 0) {
        if (g) hipGraphDestroy(g);
        return rc;
    }
    HCHK(e);
    hipGraphExec_t ex = nullptr;
    const hipError_t made = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    if (made != hipSuccess) hipGraphDestroy(g);
    HCHK(made);
    chain_graph_[form] = g;
    chain_exec_[form] = ex;
    return 0;
}

int Sequence::check_run(int n, bool with_logits) {
    if (!ready()) return fail_arg("model globals not set");
    const int p = position();
    if (p < 0) return BITNET_HIP_ERR_GPU;
    if (n < 0 || p + n > max_pos_ - 1) return fail_arg("KV cache overflow");  // T:1190-1194
    // a step without logits samples nothing: the NEXT position's token must already be in the history
    if (!with_logits && p + n > host_forced_) return fail_arg("run(with_logits = false) past the fed tokens: nothing would choose the next token");
    return 0;
}

int Sequence::run(int n, bool with_logits, bool use_graph, float *elapsed_ms) {
    if (int rc = check_run(n, with_logits)) return rc;
    const int p = position();
    hipStream_t s = (hipStream_t)stream_;
    std::vector<int> forms((size_t)n);
    for (int i = 0; i < n; ++i) forms[(size_t)i] = form_at(p + i);
    auto together = [&](int i) { return with_logits ? steps_together(&forms[(size_t)i], n - i) : 1; };
    if (use_graph)
        if (int rc = make_graphs(forms, with_logits, false)) return rc;
    host_pos_ = -1;
    graph_steps_ = 0;
    HCHK(hipEventRecord(begin_.e, s));
    for (int i = 0; i < n;) {
        if (use_graph) {
            const int form = forms[(size_t)i], k = together(i);
            HCHK(hipGraphLaunch((hipGraphExec_t)(k > 1 ? chain_exec_[form] : graph_exec_[2 * form + (with_logits ? 1 : 0)]), s));
            i += k;
            if (k > graph_steps_) graph_steps_ = k;
        } else {
            int rc = step(with_logits, forms[(size_t)i]);
            if (rc) return rc;
            ++i;
        }
    }
    if (n > 0) ran(with_logits);
    HCHK(hipEventRecord(end_.e, s));
    if (int rc = settle()) return rc;
    moved_to(p + n);
    if (elapsed_ms) HCHK(hipEventElapsedTime(elapsed_ms, begin_.e, end_.e));
    return 0;
}

int Sequence::forward(const int32_t *tokens, int n, const int32_t *want, int n_want, float *logits) {
    if (n_want < 0 || (n_want > 0 && (!want || !logits))) return fail_arg("forward: null pointer");
    for (int w = 0; w < n_want; ++w)
        if (want[w] < 0 || want[w] >= n) return fail_arg("forward: a wanted place is not among the tokens");
    if (int rc = feed(tokens, n)) return rc;
    for (int i = 0; i < n; ++i) {
        bool wanted = false;
        for (int w = 0; w < n_want; ++w) wanted = wanted || want[w] == i;
        if (int rc = run(1, wanted, true, nullptr)) return rc;
        for (int w = 0; w < n_want; ++w)
            if (want[w] == i)
                if (int rc = last_logits(logits + (size_t)w * vocab_)) return rc;
    }
    return 0;
}

}  // namespace bitnet_host
