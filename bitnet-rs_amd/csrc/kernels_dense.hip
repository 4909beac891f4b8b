// kernels_dense.hip -- operators on bf16 weight matrices (gfx950): embedding rows, residual + norm rows, the many-row matmul
// and the matrix-vector product of the decode step with its input transform folded in.
//
// Precision: residual stream, norms and accumulation are f32 everywhere.  The matmul multiplies bf16 activations on the matrix
// cores, or -- a_f32 -- f32 activations with f32 multiply-adds; the matrix-vector product always multiplies f32 activations.
#include <algorithm>
#include <cmath>
#include <iterator>
#include <type_traits>

#include "dense.hpp"

namespace bitnet_hip {

// ---- embedding rows ---------------------------------------------------------------------------------------------------
__global__ void k_embed_bf16(const uint16_t *__restrict__ table, size_t ld, const int *__restrict__ tokens, const int *__restrict__ offset,
                             int width, int vocab, float scale, const float *__restrict__ norm_w, float eps, TokenPairs pairs, float *__restrict__ out) {
    __shared__ float slot[4];
    const int at = (offset ? *offset : 0) + blockIdx.x;
    auto token = [&](int i) { return min(max(tokens[i], 0), vocab - 1); };
    const int tok = token(at);
    if (pairs.table) {
        const uint64_t sum = (uint64_t)token(max(at - 1, 0)) * pairs.mul_prev + (uint64_t)tok * pairs.mul_cur;
        const uint64_t pair = at == 0 ? pairs.buckets : (sum | pairs.buckets) >> 32 ? sum % pairs.buckets : (uint32_t)sum % (uint32_t)pairs.buckets;
        const uint16_t *a = table + (size_t)tok * ld, *b = pairs.table + (size_t)pair * pairs.ld;
        float *o = out + (size_t)blockIdx.x * width;
        if (width % 4 == 0) {
            for (int i = 4 * (threadIdx.x + 256 * blockIdx.y); i < width; i += 1024 * gridDim.y) {
                const u32x2 x = *reinterpret_cast<const u32x2 *>(a + i), y = *reinterpret_cast<const u32x2 *>(b + i);
                *reinterpret_cast<f32x4 *>(o + i) = scale * f32x4{bf2f(x.x & 0xffffu), bf2f(x.x >> 16), bf2f(x.y & 0xffffu), bf2f(x.y >> 16)} +
                                                    f32x4{bf2f(y.x & 0xffffu), bf2f(y.x >> 16), bf2f(y.y & 0xffffu), bf2f(y.y >> 16)};
            }
        } else {
            for (int i = threadIdx.x + 256 * blockIdx.y; i < width; i += 256 * gridDim.y) o[i] = scale * bf2f(a[i]) + bf2f(b[i]);
        }
        return;
    }
    // four columns at a time: a row of one token is a chain of three dependent loads (position, token, columns), and no loop of them
    const uint16_t *row = table + (size_t)tok * ld;
    const bool vec = width % 4 == 0 && ld % 4 == 0 && ((uintptr_t)table & 7) == 0 && (((uintptr_t)out | (uintptr_t)norm_w) & 15) == 0;
    auto four = [&](int i) {
        const u32x2 x = *reinterpret_cast<const u32x2 *>(row + i);
        return scale * f32x4{bf2f(x.x & 0xffffu), bf2f(x.x >> 16), bf2f(x.y & 0xffffu), bf2f(x.y >> 16)};
    };
    if (norm_w && vec && width <= 4096) {
        f32x4 v[4], w[4];
        const int n4 = width / 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = reinterpret_cast<const f32x4 *>(norm_w)[min((int)threadIdx.x + 256 * j, n4 - 1)];
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = four(4 * min((int)threadIdx.x + 256 * j, n4 - 1));
#pragma unroll
        for (int j = 0; j < 4; ++j) ss += (int)threadIdx.x + 256 * j < n4 ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.f;
        const float inv = 1.0f / sqrtf(group_total<4>(ss, slot) / (float)width + eps);
        f32x4 *o = reinterpret_cast<f32x4 *>(out + (size_t)blockIdx.x * width);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if ((int)threadIdx.x + 256 * j < n4) o[threadIdx.x + 256 * j] = v[j] * inv * w[j];
        return;
    }
    if (norm_w) {
        constexpr int NR = 16;  // rows of up to 4096 columns in registers, what lies behind is read again
        float ss = 0.f, v[NR], w[NR];
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const int i = threadIdx.x + 256 * j;
            v[j] = i < width ? scale * bf2f(row[i]) : 0.f;
            w[j] = i < width ? norm_w[i] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < NR; ++j) ss += v[j] * v[j];
        for (int i = threadIdx.x + 256 * NR; i < width; i += 256) ss += scale * bf2f(row[i]) * (scale * bf2f(row[i]));
        const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + eps);
        float *o = out + (size_t)blockIdx.x * width;
#pragma unroll
        for (int j = 0; j < NR; ++j)
            if ((int)threadIdx.x + 256 * j < width) o[threadIdx.x + 256 * j] = v[j] * inv * w[j];
        for (int i = threadIdx.x + 256 * NR; i < width; i += 256) o[i] = scale * bf2f(row[i]) * inv * norm_w[i];
        return;
    }
    if (vec) {
        for (int i = 4 * (threadIdx.x + 256 * blockIdx.y); i < width; i += 1024 * gridDim.y) *reinterpret_cast<f32x4 *>(out + (size_t)blockIdx.x * width + i) = four(i);
    } else {
        for (int i = threadIdx.x + 256 * blockIdx.y; i < width; i += 256 * gridDim.y) out[(size_t)blockIdx.x * width + i] = scale * bf2f(row[i]);
    }
}

// The greedy token out of a product's partial maxima (as k_argmax_final, position and history too) and the embedding row of the next position, which a step behind this one starts with: as
// k_embed_bf16 gives it, bit for bit.  A chain of latencies: position, token, columns; a token that is there already is on its way beside the maxima.  Two launches of 3.9 and 4.4 to 4.7 us
// become one of 4.5 to 5.2 us.
__global__ __launch_bounds__(256) void k_argmax_embed(const float *best_val, const int *best_idx, int n, int *token_out, int *pos_ptr, int *history, const int *n_forced, EmbedNext e) {
    __shared__ float sv[4], slot[4];
    __shared__ int si[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, at = *pos_ptr + 1;
    const bool forced = n_forced && at < *n_forced;
    const int there = history[at], prev = min(max(history[at - 1], 0), e.vocab - 1), n4 = e.width / 4;
    f32x4 v[4], w[4];
    u32x2 x[4], y[4];
    auto fetch = [&](int token) {
        const uint16_t *row = e.table + (size_t)token * e.ld, *two = nullptr;
        if (e.pairs.table) {
            const uint64_t sum = (uint64_t)prev * e.pairs.mul_prev + (uint64_t)token * e.pairs.mul_cur;
            two = e.pairs.table + (size_t)((sum | e.pairs.buckets) >> 32 ? sum % e.pairs.buckets : (uint32_t)sum % (uint32_t)e.pairs.buckets) * e.pairs.ld;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = 4 * min(tid + 256 * j, n4 - 1);
            x[j] = *reinterpret_cast<const u32x2 *>(row + i);
            y[j] = two ? *reinterpret_cast<const u32x2 *>(two + i) : u32x2{0u, 0u};
        }
    };
    if (forced) fetch(min(max(there, 0), e.vocab - 1));
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = e.norm_w ? reinterpret_cast<const f32x4 *>(e.norm_w)[min(tid + 256 * j, n4 - 1)] : f32x4{1.f, 1.f, 1.f, 1.f};
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    auto better = [&](float o, int i) {
        if (o > bv || (o == bv && i < bi)) bv = o, bi = i;
    };
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (tid + 256 * j < n) better(best_val[tid + 256 * j], best_idx[tid + 256 * j]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(bv, off, 64);
        const int i = __shfl_xor(bi, off, 64);
        better(o, i);
    }
    if (lane == 0) sv[wave] = bv, si[wave] = bi;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) better(sv[i], si[i]);
    const int token = bi == 0x7fffffff ? 0 : bi;
    if (!forced) fetch(min(token, e.vocab - 1));  // (there may be more logits than rows)
    if (tid == 0) {
        if (token_out) *token_out = token;
        if (!forced) history[at] = token;
        *pos_ptr = at;
    }
    auto four = [&](u32x2 u) { return f32x4{bf2f(u.x & 0xffffu), bf2f(u.x >> 16), bf2f(u.y & 0xffffu), bf2f(u.y >> 16)}; };
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = e.scale * four(x[j]);
    if (e.pairs.table)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = v[j] + four(y[j]);
    if (e.norm_w) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) ss += tid + 256 * j < n4 ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.f;
        const float inv = 1.0f / sqrtf(group_total<4>(ss, slot) / (float)e.width + e.eps);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = v[j] * inv * w[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (tid + 256 * j < n4) reinterpret_cast<f32x4 *>(e.out)[tid + 256 * j] = v[j];
}

bool embed_follows(const EmbedNext &e) {
    const uintptr_t rows = (uintptr_t)e.table | (uintptr_t)e.pairs.table, vectors = (uintptr_t)e.norm_w | (uintptr_t)e.out;
    return e.width > 0 && e.width % 4 == 0 && e.width <= 4096 && (e.ld | e.pairs.ld) % 4 == 0 && (rows & 7) == 0 && (vectors & 15) == 0 && !(e.norm_w && e.pairs.table);
}

hipError_t launch_argmax_embed(const float *best_val, const int *best_idx, int n, int *token, int *pos, int *history, const int *n_forced, const EmbedNext &e, hipStream_t s) {
    if (n > 1024 || !embed_follows(e)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_argmax_embed, dim3(1), dim3(256), 0, s, best_val, best_idx, n, token, pos, history, n_forced, e);
    return hipGetLastError();
}

hipError_t launch_embed_bf16(const uint16_t *table, size_t ld, const int *tokens, const int *offset, int n, int width, int vocab, float scale,
                             const float *norm_w, float eps, const TokenPairs &pairs, float *out, hipStream_t s) {
    const int parts = !norm_w && n == 1 ? (width + 1023) / 1024 : 1;  // (one token: its row at once)
    hipLaunchKernelGGL(k_embed_bf16, dim3(n, parts), dim3(256), 0, s, table, ld, tokens, offset, width, vocab, scale, norm_w, eps, pairs, out);
    return hipGetLastError();
}

__global__ void k_gather_rows(const float *__restrict__ x, const int *__restrict__ rows, int width, float *__restrict__ out) {
    const float *src = x + (size_t)rows[blockIdx.x] * width;
    for (int i = threadIdx.x; i < width; i += blockDim.x) out[(size_t)blockIdx.x * width + i] = src[i];
}

hipError_t launch_gather_rows(const float *x, const int *rows, int n, int width, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_gather_rows, dim3(n), dim3(256), 0, s, x, rows, width, out);
    return hipGetLastError();
}

// the last inputs of a portion into the ring of a causal convolution (position p in row p % taps)
template <class T>
__global__ __launch_bounds__(256) void k_conv_keep(const T *rows, size_t ld, int channels, int taps, float *ring, const int *pos_ptr, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x, pos0 = *pos_ptr;
    if (i >= channels) return;
    for (int t = max(0, n - (taps - 1)); t < n; ++t) ring[(size_t)((pos0 + t) % taps) * channels + i] = ld_act(rows + (size_t)t * ld, i);
}

hipError_t launch_conv_keep(const void *rows, size_t ld, int rows_f32, int channels, int taps, float *ring, const int *pos, int n, hipStream_t s) {
    const dim3 grid((channels + 255) / 256);
    if (rows_f32)
        hipLaunchKernelGGL(k_conv_keep<float>, grid, dim3(256), 0, s, (const float *)rows, ld, channels, taps, ring, pos, n);
    else
        hipLaunchKernelGGL(k_conv_keep<uint16_t>, grid, dim3(256), 0, s, (const uint16_t *)rows, ld, channels, taps, ring, pos, n);
    return hipGetLastError();
}

// ---- residual + norm rows ---------------------------------------------------------------------------------------------
// t = y + the chosen experts' rows (of a block whose sublayers add up), x += mult * t or scale * norm(t); h = norm(x), x or [x; x2].  One workgroup per row.
// Short prompts: a launch is its chain of loads and reductions, so whatever does not hang on a sum -- the weights too -- is requested ahead of the first one, four columns at a time
// and without branches around the loads.  Back to back, 8 rows of 3072 columns between two norms: 6.4 -> 3.3 us (single columns, weights behind the sums), of 1536 with eight
// experts' rows 5.3 -> 3.6.  Documents: bytes; 4096 rows of 3072 33.7 -> 27.6 us (5.5 TB/s), with eight experts' rows 65 -> 61.
__device__ __forceinline__ f32x4 ld4(const float *p, size_t i) { return *reinterpret_cast<const f32x4 *>(p + i); }
__device__ __forceinline__ f32x4 ld4(const uint16_t *p, size_t i) {
    const u32x2 v = *reinterpret_cast<const u32x2 *>(p + i);
    return f32x4{bf2f(v.x & 0xffffu), bf2f(v.x >> 16), bf2f(v.y & 0xffffu), bf2f(v.y >> 16)};
}
__device__ __forceinline__ void st4(float *p, size_t i, f32x4 v) { *reinterpret_cast<f32x4 *>(p + i) = v; }
__device__ __forceinline__ void st4(uint16_t *p, size_t i, f32x4 v) {
    *reinterpret_cast<bf16x4 *>(p + i) = bf16x4{(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
}
constexpr int kSumRegs = 4;

// NJ: a thread's groups of four columns, in registers (0: columns one by one, any width).  IDENTITY: slots may be negative.  GATED: with a number per row on y, a gate per column on
// what is added, or both.  AHEAD: the weights are requested ahead of the first sum.  Not with experts' rows of more than
// 2048 columns: the registers are the experts' loads' then; 300 rows of 4096 with eight experts' rows 6.9 us (ahead: 11.7), 8 of 2560 in f32 3.8 (5.4).
template <class T, int NJ, bool IDENTITY, bool GATED, bool AHEAD>
__global__ __launch_bounds__(256) void k_sum_norm_rows(SumRows p) {
    __shared__ float slot[4];
    const int tid = threadIdx.x, width = (int)p.width;
    float *x = p.x + (size_t)blockIdx.x * width;
    const float *y = p.y ? p.y + (size_t)blockIdx.x * p.ldy : nullptr;
    T *h = p.h ? (T *)p.h + (size_t)blockIdx.x * p.ldh : nullptr;
    const T *er = (const T *)p.expert_rows;
    const int *slots = p.slots + (size_t)blockIdx.x * p.top;
    const float *sw = p.slot_weights + (size_t)blockIdx.x * p.top;
    const float *x2 = p.x2 ? p.x2 + (size_t)blockIdx.x * width : nullptr;
    const T *gate = GATED && p.gate ? (const T *)p.gate + (size_t)blockIdx.x * p.ld_gate : nullptr;
    const float ys = GATED && p.y_scale ? p.y_scale[(size_t)blockIdx.x * p.ld_y_scale] : 1.0f;
    const T *input = p.input ? (const T *)p.input + (size_t)blockIdx.x * p.ld_input : nullptr;  // (may be h: a thread reads its columns ahead of writing them)
    const int top = (int)p.top;
    if constexpr (NJ > 0) {
        const int n4 = width >> 2;
        int at[NJ];  // (threads past the row read its last columns)
        bool mine[NJ];
        f32x4 v[NJ], a[NJ], gv[NJ], pw[NJ], sc[NJ], nw[NJ], nb[NJ];
        const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int i = tid + 256 * j;
            mine[j] = i < n4, at[j] = 4 * min(i, n4 - 1);
            v[j] = ld4(x, at[j]), a[j] = zero;
        }
        auto all = [&](auto f) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) f(j);
        };
        if (y) all([&](int j) { a[j] = ld4(y, at[j]); });
        auto post_weights = [&] {
            if (p.post_weight) all([&](int j) { pw[j] = ld4(p.post_weight, at[j]); });
            if (p.scale) all([&](int j) { sc[j] = ld4(p.scale, at[j]); });
            if (GATED && gate) all([&](int j) { gv[j] = ld4(gate, at[j]); });
        };
        auto weights = [&] {
            if (h && p.weight) all([&](int j) { nw[j] = ld4(p.weight, at[j]); });
            if (h && p.bias) all([&](int j) { nb[j] = ld4(p.bias, at[j]); });
        };
        if (AHEAD) post_weights(), weights();
        if (y || top) {
            if (GATED) all([&](int j) { a[j] *= ys; });
            float through = 0.f;
#pragma unroll 4
            for (int k = 0; k < top; ++k) {
                const int s = slots[k];
                const bool taken = !IDENTITY || s >= 0;  // (without a branch: an identity's place is taken by some row, which is not added)
                const float w = sw[k];
                const T *row = er + (size_t)(IDENTITY ? max(s, 0) : s) * p.ld_expert;
                if (IDENTITY) through += taken ? 0.f : w;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const f32x4 e = ld4(row, at[j]);
                    a[j] += taken ? w * e : zero;
                }
            }
            if (IDENTITY && through != 0.f) all([&](int j) { a[j] += through * (input ? ld4(input, at[j]) : v[j]); });
            if (!AHEAD) post_weights();
            float post = 0.f;
            if (p.post_weight) {
                float ss = 0.f;
                all([&](int j) { ss += mine[j] ? (a[j].x * a[j].x + a[j].y * a[j].y) + (a[j].z * a[j].z + a[j].w * a[j].w) : 0.f; });
                post = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + p.eps);
            }
            all([&](int j) {
                if (GATED && gate) a[j] *= gv[j];
                if (p.post_weight) {
                    f32x4 r = a[j] * post * (p.weight_offset + pw[j]);
                    if (p.scale) r *= sc[j];
                    v[j] += r;
                } else {
                    v[j] += p.mult * a[j];
                }
                if (mine[j]) st4(x, at[j], v[j]);
            });
        }
        if (!h) return;
        if (!AHEAD) weights();
        if (x2) {
            all([&](int j) {
                const f32x4 w = ld4(x2, at[j]);
                if (mine[j]) st4(h, at[j], v[j]), st4(h, width + at[j], w);
            });
        } else if (!p.weight) {
            all([&](int j) {
                if (mine[j]) st4(h, at[j], v[j]);
            });
        } else {
            float mean = 0.f, ss = 0.f;
            if (p.center) {
                float t = 0.f;
                all([&](int j) { t += mine[j] ? (v[j].x + v[j].y) + (v[j].z + v[j].w) : 0.f; });
                mean = group_sum<4>(t, slot) / (float)width;
            }
            all([&](int j) {
                v[j] -= mean;
                ss += mine[j] ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.f;
            });
            const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + p.eps);
            all([&](int j) {
                f32x4 r = v[j] * inv * (p.weight_offset + nw[j]);
                if (p.bias) r += nb[j];
                if (mine[j]) st4(h, at[j], r);
            });
        }
    } else {  // (a thread comes back to its own columns only)
        if (y || top) {
            auto sum = [&](int i) {
                float a = y ? ys * y[i] : 0.f;
                for (int k = 0; k < top; ++k) a += sw[k] * (!IDENTITY || slots[k] >= 0 ? ld_act(er + (size_t)slots[k] * p.ld_expert, i) : input ? ld_act(input, i) : x[i]);
                return a;
            };
            float post = 0.f;
            if (p.post_weight) {
                float ss = 0.f;
                for (int i = tid; i < width; i += 256) {
                    const float a = sum(i);
                    ss += a * a;
                }
                post = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + p.eps);
            }
            for (int i = tid; i < width; i += 256)
                x[i] += (gate ? ld_act(gate, i) : 1.0f) *
                        (p.post_weight ? (p.scale ? p.scale[i] : 1.0f) * (sum(i) * post * (p.weight_offset + p.post_weight[i])) : p.mult * sum(i));
        }
        if (!h) return;
        if (x2) {
            for (int i = tid; i < width; i += 256) {
                st_act(h, i, x[i]);
                st_act(h, width + i, x2[i]);
            }
        } else if (!p.weight) {
            for (int i = tid; i < width; i += 256) st_act(h, i, x[i]);
        } else {
            float mean = 0.f, ss = 0.f;
            if (p.center) {
                float t = 0.f;
                for (int i = tid; i < width; i += 256) t += x[i];
                mean = group_sum<4>(t, slot) / (float)width;
            }
            for (int i = tid; i < width; i += 256) ss += (x[i] - mean) * (x[i] - mean);
            const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + p.eps);
            for (int i = tid; i < width; i += 256) st_act(h, i, (x[i] - mean) * inv * (p.weight_offset + p.weight[i]) + (p.bias ? p.bias[i] : 0.f));
        }
    }
    for (int i = (x2 ? 2 : 1) * width + tid; i < (int)p.ldh; i += 256) st_act(h, i, 0.f);
}

// x += scale * norm(y), h = norm(x) or x, of rows that four columns at a time do not fit: an odd width, operands off their alignment, more than 4096 columns.  The kernel above goes over
// experts, gates and biases in every column there, with a load at a time in flight: 8 rows of 3073 columns 10.1 us, here 6.6; 4096 of 5121 89 and 85.  (Without y it is the faster one up to
// 2048 columns: 8 rows of 1022 2.6 and 2.9 us.)  REGS: up to 4096 columns in registers.
template <class T, bool REGS>
__global__ __launch_bounds__(256) void k_residual_norm_rows(SumRows p) {
    constexpr int NJ = REGS ? 16 : 1;
    __shared__ float slot[4];
    const int tid = threadIdx.x, width = (int)p.width;
    float *x = p.x + (size_t)blockIdx.x * width;
    const float *y = p.y ? p.y + (size_t)blockIdx.x * p.ldy : nullptr, *__restrict__ post = p.post_weight, *__restrict__ scale = p.scale, *__restrict__ weight = p.weight;
    T *h = p.h ? (T *)p.h + (size_t)blockIdx.x * p.ldh : nullptr;
    float xv[NJ], yv[NJ];
    auto columns = [&](auto f) {
        if constexpr (REGS) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) f(tid + 256 * j, j, tid + 256 * j < width);
        } else {
            for (int i = tid; i < width; i += 256) f(i, 0, true);
        }
    };
    auto x_at = [&](int i, int j) { return REGS ? xv[j] : x[i]; };
    if (y) {
        float ss = 0.f;
        columns([&](int i, int j, bool in) {
            yv[j] = in ? y[i] : 0.f;
            if (REGS) xv[j] = in ? x[i] : 0.f;
            ss += yv[j] * yv[j];
        });
        const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + p.eps);
        columns([&](int i, int j, bool in) {
            if (!in) return;
            const float v = x_at(i, j) + (scale ? scale[i] : 1.0f) * ((REGS ? yv[j] : y[i]) * inv * (p.weight_offset + post[i]));
            x[i] = v, xv[j] = v;
        });
    } else if (REGS) {
        columns([&](int i, int j, bool in) { xv[j] = in ? x[i] : 0.f; });
    }
    if (!h) return;
    if (weight) {
        float ss = 0.f;
        columns([&](int i, int j, bool) {
            const float v = x_at(i, j);
            ss += v * v;
        });
        const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)width + p.eps);
        columns([&](int i, int j, bool in) {
            if (in) st_act(h, i, x_at(i, j) * inv * (p.weight_offset + weight[i]));
        });
    } else {
        columns([&](int i, int j, bool in) {
            if (in) st_act(h, i, x_at(i, j));
        });
    }
    for (int i = width + tid; i < (int)p.ldh; i += 256) st_act(h, i, 0.f);
}

template <class T, int NJ, bool AHEAD>
static hipError_t sum_norm_go(const SumRows &a, hipStream_t s) {
    const bool g = a.gate || a.y_scale;
    auto fn = g ? k_sum_norm_rows<T, NJ, false, true, AHEAD> : k_sum_norm_rows<T, NJ, false, false, AHEAD>;
    if constexpr (NJ < 3 || !AHEAD)
        if (a.identity) fn = g ? k_sum_norm_rows<T, NJ, true, true, AHEAD> : k_sum_norm_rows<T, NJ, true, false, AHEAD>;
    hipLaunchKernelGGL(fn, dim3(a.m), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <class T>
static hipError_t sum_norm_type(const SumRows &a, hipStream_t s) {
    // four columns at a time: every row of every operand starts on its own alignment
    const uintptr_t wide = (uintptr_t)a.x | (uintptr_t)a.y | (uintptr_t)a.x2 | (uintptr_t)a.post_weight | (uintptr_t)a.scale | (uintptr_t)a.weight | (uintptr_t)a.bias,
                    own = (uintptr_t)a.h | (uintptr_t)a.expert_rows | (uintptr_t)a.input | (uintptr_t)a.gate;
    const bool vec = wide % 16 == 0 && own % (4 * sizeof(T)) == 0 && a.width % 4 == 0 && a.width <= 1024 * kSumRegs && a.ldy % 4 == 0 && a.ld_expert % 4 == 0 && a.ldh % 4 == 0 &&
                     a.ld_input % 4 == 0 && a.ld_gate % 4 == 0;
    if (!vec) {
        const bool plain = (a.y ? a.post_weight != nullptr : a.width > 2048) && a.top == 0 && !a.x2 && !a.center && !a.bias && !a.gate && !a.y_scale && !a.identity;
        if (!plain) return sum_norm_go<T, 0, true>(a, s);
        auto fn = a.width <= 4096 ? k_residual_norm_rows<T, true> : k_residual_norm_rows<T, false>;
        hipLaunchKernelGGL(fn, dim3(a.m), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    // (a group more than the row needs costs its registers and its share of the instructions: 4096 rows of 512 6.3 us with one, 8.1 with two)
    if (a.width <= 1024) return sum_norm_go<T, 1, true>(a, s);
    if (a.width <= 2048) return sum_norm_go<T, 2, true>(a, s);
    if (a.top > 0 || a.identity) return a.width <= 3072 ? sum_norm_go<T, 3, false>(a, s) : sum_norm_go<T, kSumRegs, false>(a, s);
    return a.width <= 3072 ? sum_norm_go<T, 3, true>(a, s) : sum_norm_go<T, kSumRegs, true>(a, s);
}

hipError_t launch_sum_norm_rows(const SumRows &a, hipStream_t s) { return a.h_f32 ? sum_norm_type<float>(a, s) : sum_norm_type<uint16_t>(a, s); }

// h = norm(o; w) * gate (gate: already through its sigmoid); the mean runs over mean_n elements, padding columns of o are zero.  Loads and NJ as above: 8 rows of 3072 columns
// 4.4 -> 2.2 us, 4096 rows 22.6 -> 15.7.
template <class TG, class TH, int NJ>
__global__ __launch_bounds__(256) void k_gated_norm_rows(const float *__restrict__ o, size_t ldo, const float *__restrict__ w, const TG *__restrict__ gate,
                                                         size_t ldg, float eps, int n, int mean_n, TH *__restrict__ h, size_t ldh) {
    __shared__ float slot[4];
    const int tid = threadIdx.x;
    const float *orow = o + (size_t)blockIdx.x * ldo;
    const TG *grow = gate + (size_t)blockIdx.x * ldg;
    TH *hr = h + (size_t)blockIdx.x * ldh;
    float ss = 0.f;
    if constexpr (NJ > 0) {
        f32x4 v[NJ], wv[NJ], gv[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int at = 4 * min(tid + 256 * j, (n >> 2) - 1);
            if (NJ > 1 || 4 * tid < n) v[j] = ld4(orow, at), wv[j] = ld4(w, at), gv[j] = ld4(grow, at);  // (narrow rows: most waves have none; 4096 rows of 64 3.0 us, 4.7 with two groups)
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) ss += 4 * (tid + 256 * j) < n ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.f;
        const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)mean_n + eps);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (4 * (tid + 256 * j) < n) st4(hr, 4 * (tid + 256 * j), v[j] * inv * wv[j] * gv[j]);
    } else {
        for (int i = tid; i < n; i += 256) ss += orow[i] * orow[i];
        const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)mean_n + eps);
        for (int i = tid; i < n; i += 256) st_act(hr, i, orow[i] * inv * w[i] * ld_act(grow, i));
    }
    for (int i = n + tid; i < (int)ldh; i += 256) st_act(hr, i, 0.f);
}

hipError_t launch_gated_norm_rows(const float *o, size_t ldo, const float *w, const void *gate, size_t ldg, int gate_f32, float eps, int m, int n,
                                  int mean_n, void *h, size_t ldh, int h_f32, hipStream_t s) {
    auto go = [&](auto *g, auto *out) {
        using TG = std::remove_const_t<std::remove_pointer_t<decltype(g)>>;
        using TH = std::remove_pointer_t<decltype(out)>;
        const bool vec = ((uintptr_t)o | (uintptr_t)w) % 16 == 0 && (uintptr_t)g % (4 * sizeof(TG)) == 0 && (uintptr_t)out % (4 * sizeof(TH)) == 0 && n % 4 == 0 && n <= 1024 * kSumRegs &&
                         ldo % 4 == 0 && ldg % 4 == 0 && ldh % 4 == 0;
        auto fn = !vec ? k_gated_norm_rows<TG, TH, 0> : n <= 512 ? k_gated_norm_rows<TG, TH, 1> : n <= 2048 ? k_gated_norm_rows<TG, TH, 2> : n <= 3072 ? k_gated_norm_rows<TG, TH, 3> : k_gated_norm_rows<TG, TH, kSumRegs>;
        hipLaunchKernelGGL(fn, dim3(m), dim3(256), 0, s, o, ldo, w, g, ldg, eps, n, mean_n, out, ldh);
    };
    if (gate_f32 && h_f32)
        go((const float *)gate, (float *)h);
    else if (gate_f32)
        go((const float *)gate, (uint16_t *)h);
    else if (!h_f32)
        go((const uint16_t *)gate, (uint16_t *)h);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---- latent rows ------------------------------------------------------------------------------------------------------
// A row's keys, in the cache: norm of the latent part, rotated part.  What does not hang on the sum is requested ahead of it.
template <class T>
__device__ void latent_row(const LatentRows &p, int row, float *slot) {
    if (p.kv_rank == 0) return;
    constexpr int REGS = 4;  // of kv_rank <= 1024
    const int tid = threadIdx.x, pos = *p.pos + row, half = p.rot_dim / 2;
    const float *zc = p.z + (size_t)row * p.ldz + p.q_rank, *zr = zc + p.kv_rank;
    T *c = (T *)p.ccache + (size_t)pos * p.ldc, *r = (T *)p.rcache + (size_t)pos * p.ldr;
    const bool regs = p.kv_rank <= 256 * REGS;
    float v[REGS], w[REGS], ss = 0.f;
    if (regs) {
#pragma unroll
        for (int j = 0; j < REGS; ++j) {
            const int i = min(tid + 256 * j, p.kv_rank - 1);
            v[j] = zc[i], w[j] = p.kv_weight[i];
        }
    }
    for (int i = tid; i < half; i += 256) {
        const float cs = p.rope_cos[(size_t)pos * half + i], sn = p.rope_sin[(size_t)pos * half + i];
        const float a = zr[i], b = zr[i + half];
        st_act(r, i, a * cs - b * sn);
        st_act(r, i + half, b * cs + a * sn);
    }
    if (regs) {
#pragma unroll
        for (int j = 0; j < REGS; ++j) ss += tid + 256 * j < p.kv_rank ? v[j] * v[j] : 0.f;
    } else {
        for (int i = tid; i < p.kv_rank; i += 256) ss += zc[i] * zc[i];
    }
    const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)p.kv_rank + p.eps);
    if (regs) {
#pragma unroll
        for (int j = 0; j < REGS; ++j)
            if (tid + 256 * j < p.kv_rank) st_act(c, tid + 256 * j, v[j] * inv * w[j]);
    } else {
        for (int i = tid; i < p.kv_rank; i += 256) st_act(c, i, zc[i] * inv * p.kv_weight[i]);
    }
}

// a row's latent queries
template <class T>
__device__ void latent_queries(const LatentRows &p, int row, float *slot) {
    constexpr int REGS = 8;  // of q_rank <= 2048
    const int tid = threadIdx.x;
    const float *z = p.z + (size_t)row * p.ldz;
    T *o = (T *)p.cq + (size_t)row * p.ldcq;
    const bool regs = p.q_rank > 0 && p.q_rank <= 256 * REGS;
    float v[REGS], w[REGS], ss = 0.f;
    if (regs) {
#pragma unroll
        for (int j = 0; j < REGS; ++j) {
            const int i = min(tid + 256 * j, p.q_rank - 1);
            v[j] = z[i], w[j] = p.q_weight[i];
        }
#pragma unroll
        for (int j = 0; j < REGS; ++j) ss += tid + 256 * j < p.q_rank ? v[j] * v[j] : 0.f;
    } else {
        for (int i = tid; i < p.q_rank; i += 256) ss += z[i] * z[i];
    }
    const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)p.q_rank + p.eps);
    if (regs) {
#pragma unroll
        for (int j = 0; j < REGS; ++j)
            if (tid + 256 * j < p.q_rank) st_act(o, tid + 256 * j, v[j] * inv * w[j]);
    } else {
        for (int i = tid; i < p.q_rank; i += 256) st_act(o, i, z[i] * inv * p.q_weight[i]);
    }
    for (int i = p.q_rank + tid; i < p.ldcq; i += 256) st_act(o, i, 0.f);
}

// blockIdx.y: the keys (where the layer has its own) and the queries, side by side
template <class T>
__global__ __launch_bounds__(256) void k_latent_rows(LatentRows p) {
    __shared__ float slot[4];
    if (p.kv_rank && blockIdx.y == 0)
        latent_row<T>(p, blockIdx.x, slot);
    else
        latent_queries<T>(p, blockIdx.x, slot);
}

hipError_t launch_latent_rows(const LatentRows &a, hipStream_t s) {
    const dim3 grid(a.m, (a.kv_rank ? 1 : 0) + (a.cq ? 1 : 0));
    if (grid.y == 0) return hipSuccess;
    hipLaunchKernelGGL(a.f32 ? k_latent_rows<float> : k_latent_rows<uint16_t>, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

// ---- matrix-vector product --------------------------------------------------------------------------------------------
// One launch per product of the decode step.  Every workgroup forms the whole input vector (L2-resident, a few KiB) in LDS --
// norm, residual + norm, or gated norm -- then its waves take rows: LPR lanes per row, 16 bytes of weights per lane and chunk,
// R rows x U chunks in flight.  The first block of weights is requested ahead of the input transform, and behind its loads.
struct GemvK {
    GemvArgs a;
    LatentRows lat;
    int kp;        // columns rounded up to whole LPR * 8 * U steps: length of the LDS vector
    int groups;    // row groups (R * 64 / LPR rows each) of one batch member
    int lat_wg;    // workgroup index that writes the latent row, or -1
};

// An argument's value as if it were read here: a condition on it is then made where it is used.  Made once and kept, the conditions of the instances with MORE took a pair of
// scalar registers each from the first load to the last store; eight to twelve were spilled, with scratch memory reserved for them.
template <bool MORE, class T>
__device__ __forceinline__ T here(T v) {
    if constexpr (MORE) asm volatile("" : "+s"(v));
    return v;
}

template <bool FIRST, class T>
__device__ __forceinline__ T &either(T &a, T &b) {
    if constexpr (FIRST) return a;
    return b;
}

// Loads return in order, so whatever a wave asked for ahead of its input it also waits for: the input's loads go out first, `weights` (the first rows' requests)
// behind them, the arithmetic last -- it runs while the weights are on their way.
// NR: sixteen-byte registers per thread, for vectors of up to 1024 NR elements; longer ones are formed in LDS.  slot: twelve floats.
template <bool MORE, int NR, class F>
__device__ __forceinline__ void form_input(const VecIn &in, const float *x, int cols, int kp, float *xs, float *slot, bool writer, F weights) {
    const int tid = threadIdx.x;
    const int n = in.n;
    if (in.kind == BITNET_HIP_IN_PLAIN) {
        if ((cols & 3) == 0 && ((uintptr_t)x & 15) == 0) {
            constexpr int NV = 8;  // sixteen-byte loads in flight per thread
            const int c4 = cols >> 2, k4 = kp >> 2;
            f32x4 v[NV];
            auto load = [&](int i0) {
#pragma unroll
                for (int j = 0; j < NV; ++j) v[j] = reinterpret_cast<const f32x4 *>(x)[min(i0 + 256 * j, c4 - 1)];
            };
            auto store = [&](int i0) {
#pragma unroll
                for (int j = 0; j < NV; ++j) {
                    const int i = i0 + 256 * j;
                    if (i < k4) reinterpret_cast<f32x4 *>(xs)[i] = i < c4 ? v[j] : f32x4{0.f, 0.f, 0.f, 0.f};
                }
            };
            load(tid);
            weights();
            store(tid);
            for (int i0 = tid + 256 * NV; i0 < k4; i0 += 256 * NV) {
                load(i0);
                store(i0);
            }
        } else {
            weights();
            for (int i = tid; i < kp; i += 256) xs[i] = i < cols ? x[i] : 0.f;
        }
        __syncthreads();
        return;
    }
    auto added = [&] { return here<MORE>(in.kind) >= BITNET_HIP_IN_RESIDUAL_NORM && here<MORE>(in.y); };
    auto normed = [&] { return added() && here<MORE>(in.post_weight); };
    auto last_norm = [&] { return here<MORE>(in.kind) < BITNET_HIP_IN_CONCAT; };
    auto two = [&] { return here<MORE>(in.kind) == BITNET_HIP_IN_CONCAT; };
    if ((n & 3) == 0 && n <= 1024 * NR) {
        // (MORE: a bias waits for the registers of a gate on what is added, a gate on the norm for those of the added norm's weight; with registers of their own two workgroups
        // of 13824 x 4096 fit a CU instead of three: 28.4 us, 23.1 without a gate)
        f32x4 xv[NR], yv[NR], pw[NR], sc[NR], yg[NR], wv[NR], b_own[NR], g_own[NR];
        auto &bv = either<MORE>(yg, b_own), &gv = either<MORE>(pw, g_own);
        const int n4 = n >> 2;
        auto scaled = [&] { return normed() && here<MORE>(in.scale); };
        auto y_gated = [&] { return MORE && added() && here<MORE>(in.y_gate); };
        auto shifted = [&] { return last_norm() && here<MORE>(in.center) && here<MORE>(in.bias); };
        auto gated = [&] { return last_norm() && here<MORE>(in.gate); };
        auto load = [&](f32x4 (&v)[NR], const float *from) {
#pragma unroll
            for (int j = 0; j < NR; ++j) v[j] = reinterpret_cast<const f32x4 *>(from)[min(tid + 256 * j, n4 - 1)];
        };
        load(xv, x);
        if (added()) load(yv, in.y);
        if (normed()) load(pw, in.post_weight);
        if (scaled()) load(sc, in.scale);
        if (y_gated()) load(yg, in.y_gate);
        if (last_norm()) load(wv, in.weight);
        if (two()) load(wv, in.x2);
        if (shifted() && !y_gated()) load(bv, in.bias);
        if (gated() && !(MORE && normed())) load(gv, in.gate);
        weights();
        auto squares = [&](const f32x4 (&v)[NR]) {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < NR; ++j) ss += tid + 256 * j < n4 ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.f;
            return ss;
        };
        const float count = (float)in.mean_n, eps = in.eps, offset = in.offset;
        auto inverse = [=](float ss) { return 1.0f / sqrtf(ss / count + eps); };
        if (added()) {
            const bool of_norm = normed(), of_scale = scaled(), of_gate = y_gated();
            const float inv = of_norm ? inverse(group_total<4>(squares(yv), slot)) : 1.0f;
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int i = tid + 256 * j;
                f32x4 v = yv[j] * (of_norm ? inv : in.mult);
                if (of_norm) v *= offset + pw[j];
                if (of_scale) v *= sc[j];
                if (of_gate) v *= yg[j];
                xv[j] += v;
                if (writer && in.x_out && i < n4) reinterpret_cast<f32x4 *>(in.x_out)[i] = xv[j];
            }
        }
        if (shifted() && y_gated()) load(bv, in.bias);
        if (MORE && gated() && normed()) load(gv, in.gate);
        if (!last_norm()) {
            const bool concat = two();
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int i = tid + 256 * j;
                if (i >= n4) continue;
                reinterpret_cast<f32x4 *>(xs)[i] = xv[j];
                if (concat) reinterpret_cast<f32x4 *>(xs)[n4 + i] = wv[j];
            }
            for (int i = (concat ? 2 : 1) * n + tid; i < kp; i += 256) xs[i] = 0.f;
            __syncthreads();
            return;
        }
        if (here<MORE>(in.center)) {
            float t = 0.f;
#pragma unroll
            for (int j = 0; j < NR; ++j) t += tid + 256 * j < n4 ? (xv[j].x + xv[j].y) + (xv[j].z + xv[j].w) : 0.f;
            const float mean = group_total<4>(t, slot + 4) / (float)in.mean_n;
#pragma unroll
            for (int j = 0; j < NR; ++j) xv[j] -= mean;
        }
        const float inv = inverse(group_total<4>(squares(xv), slot + 8));
        const bool of_gate = gated(), of_bias = shifted();
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const int i = tid + 256 * j;
            if (i >= n4) continue;
            f32x4 r = xv[j] * inv * (offset + wv[j]);
            if (of_gate) r *= gv[j];
            if (of_bias) r += bv[j];
            reinterpret_cast<f32x4 *>(xs)[i] = r;
            if (writer && in.h_out) reinterpret_cast<f32x4 *>(in.h_out)[i] = r;
        }
    } else {
        weights();
        float ss = 0.f;
        if (added() && !normed()) {
            for (int i = tid; i < n; i += 256) {
                const float v = x[i] + in.mult * in.y[i] * (MORE && in.y_gate ? in.y_gate[i] : 1.0f);
                xs[i] = v;
                if (writer && in.x_out) in.x_out[i] = v;
                ss += v * v;
            }
        } else if (added()) {
            for (int i = tid; i < n; i += 256) ss += in.y[i] * in.y[i];
            const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)in.mean_n + in.eps);
            ss = 0.f;
            for (int i = tid; i < n; i += 256) {
                const float v = x[i] + (in.scale ? in.scale[i] : 1.0f) * (MORE && in.y_gate ? in.y_gate[i] : 1.0f) * (in.y[i] * inv * (in.offset + in.post_weight[i]));
                xs[i] = v;
                if (writer && in.x_out) in.x_out[i] = v;
                ss += v * v;
            }
        } else {
            for (int i = tid; i < n; i += 256) {
                xs[i] = x[i];
                ss += x[i] * x[i];
            }
        }
        if (!last_norm()) {
            const bool concat = two();
            for (int i = tid; concat && i < n; i += 256) xs[n + i] = in.x2[i];
            for (int i = (concat ? 2 : 1) * n + tid; i < kp; i += 256) xs[i] = 0.f;
            __syncthreads();
            return;
        }
        if (in.center) {  // (a thread comes back to its own elements only)
            float t = 0.f;
            for (int i = tid; i < n; i += 256) t += xs[i];
            const float mean = group_sum<4>(t, slot) / (float)in.mean_n;
            ss = 0.f;
            for (int i = tid; i < n; i += 256) {
                xs[i] -= mean;
                ss += xs[i] * xs[i];
            }
        }
        const float inv = 1.0f / sqrtf(group_sum<4>(ss, slot) / (float)in.mean_n + in.eps);
        for (int i = tid; i < n; i += 256) {
            xs[i] = xs[i] * inv * (in.offset + in.weight[i]) * (in.gate ? in.gate[i] : 1.0f) + (in.center && in.bias ? in.bias[i] : 0.f);
            if (writer && in.h_out) in.h_out[i] = xs[i];
        }
    }
    for (int i = n + tid; i < kp; i += 256) xs[i] = 0.f;
    __syncthreads();
}

template <int LPR>
__device__ __forceinline__ float lanes_total(float v) {
    if (LPR == 8) {
        v += dpp<0x141>(v);       // row_half_mirror
        v += dpp<0xb1>(v);        // quad_perm [1,0,3,2]
        return v + dpp<0x4e>(v);  // quad_perm [2,3,0,1]
    }
    v = row_sum(v);
    return LPR == 64 ? rows_sum(v) : v;
}

struct GemvPlainK {
    const float *x, *bias;
    const uint16_t *w;
    float *y;
    int rows, cols, ld, act0, act1, act_split;
};

// MORE: whatever bitnet_hip_epilogue and a gate on the residual ask for
template <int LPR, int R, int U, bool MORE, int NR>
__global__ __launch_bounds__(256, MORE && R * U >= 20 ? 2 : 1) void k_dense_gemv(GemvK p) {
    extern __shared__ __attribute__((aligned(16))) float xs[];
    __shared__ float slot[12];
    __shared__ float wbv[4];
    __shared__ int wbi[4];
    const GemvArgs &a = p.a;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // (every argument at once: read where they are used, behind branches, they are a chain of scalar loads ahead of the first vector load)
    asm volatile("" ::"s"(a.in.x), "s"(a.in.y), "s"(a.in.post_weight), "s"(a.in.scale), "s"(a.in.weight), "s"(a.in.bias), "s"(a.in.gate), "s"(a.in.x_out), "s"(a.in.kind), "s"(a.in.n),
                 "s"(a.in.center), "s"(a.in.mean_n), "s"(a.in.x2), "s"(a.w), "s"(a.rows), "s"(a.cols), "s"(a.ld), "s"(p.kp), "s"(p.groups), "s"(p.lat_wg));
    if ((int)blockIdx.x == p.lat_wg) {  // (the whole workgroup)
        if (blockIdx.y > 0) return;
        if (p.lat.f32) {
            if (p.lat.cq) latent_queries<float>(p.lat, 0, slot);
            latent_row<float>(p.lat, 0, slot);
        } else {
            if (p.lat.cq) latent_queries<uint16_t>(p.lat, 0, slot);
            latent_row<uint16_t>(p.lat, 0, slot);
        }
        return;
    }
    const int n_wg = p.lat_wg >= 0 ? p.lat_wg : (int)gridDim.x;
    const int b = blockIdx.y;
    const int sub = lane / LPR, l = lane % LPR;
    constexpr int G = 64 / LPR;
    const uint16_t *wb = a.w + (size_t)b * a.w_batch;
    const int step = LPR * 8 * U;
    const int last_col = a.cols - 8;
    int g = blockIdx.x * 4 + wave;
    u32x4 w[R][U];
    auto fetch = [&](int grp, int k0) {
        const int row0 = (grp * G + sub) * R;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = row0 + r < a.rows ? row0 + r : a.rows - 1;
            const uint16_t *wr = wb + (size_t)row * a.ld;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int col = k0 + (u * LPR + l) * 8;
                w[r][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wr + (col < last_col ? col : last_col)));
            }
        }
    };
    // the earlier positions of a convolution's rows, a tap per lane; summed behind the product
    const Epilogue &e = a.more;
    const bool conv = MORE && e.conv, mul = MORE && e.mul;
    // (arguments read where they are used: with a convolution's they do not all fit the scalar registers)
    auto late = [] {
        auto *k = (const __attribute__((address_space(4))) GemvK *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(k));
        return k;
    };
    const int pos = conv ? *e.pos : 0;
    int mul_at = 0;
    float past[R];
    auto fetch_past = [&](int grp) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int ch = (grp * G + sub) * R + r - e.conv_from;
            past[r] = 0.f;
            if (ch < 0 || ch >= e.channels) continue;
            for (int j = l; j < e.taps - 1; j += LPR) {
                const int at = pos - (e.taps - 1) + j;
                if (at >= 0) past[r] += e.conv[(size_t)j * e.channels + ch] * e.ring[(size_t)(at % e.taps) * e.channels + ch];
            }
        }
    };
    // (the taps are summed as they arrive: ahead of the weights, too)
    form_input<MORE, NR>(a.in, a.in.x + (size_t)b * a.x_batch, a.cols, p.kp, xs, slot, blockIdx.x == 0 && b == 0, [&] {
        if (conv && g < p.groups) fetch_past(g);
        if (g < p.groups) fetch(g, 0);
        if (mul) mul_at = *e.mul_at;
    });
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (; g < p.groups; g += n_wg * 4) {
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.f;
        for (int k0 = 0; k0 < p.kp; k0 += step) {
            u32x4 c[R][U];
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int u = 0; u < U; ++u) c[r][u] = w[r][u];
            if (k0 + step < p.kp)
                fetch(g, k0 + step);
            else if (g + n_wg * 4 < p.groups)
                fetch(g + n_wg * 4, 0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const f32x4 x0 = *reinterpret_cast<const f32x4 *>(xs + k0 + (u * LPR + l) * 8);
                const f32x4 x1 = *reinterpret_cast<const f32x4 *>(xs + k0 + (u * LPR + l) * 8 + 4);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const u32x4 v = c[r][u];
                    acc[r] = fmaf(x0.x, __builtin_bit_cast(float, v.x << 16), acc[r]);
                    acc[r] = fmaf(x0.y, __builtin_bit_cast(float, v.x & 0xffff0000u), acc[r]);
                    acc[r] = fmaf(x0.z, __builtin_bit_cast(float, v.y << 16), acc[r]);
                    acc[r] = fmaf(x0.w, __builtin_bit_cast(float, v.y & 0xffff0000u), acc[r]);
                    acc[r] = fmaf(x1.x, __builtin_bit_cast(float, v.z << 16), acc[r]);
                    acc[r] = fmaf(x1.y, __builtin_bit_cast(float, v.z & 0xffff0000u), acc[r]);
                    acc[r] = fmaf(x1.z, __builtin_bit_cast(float, v.w << 16), acc[r]);
                    acc[r] = fmaf(x1.w, __builtin_bit_cast(float, v.w & 0xffff0000u), acc[r]);
                }
            }
        }
        const int row0 = (g * G + sub) * R;
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = lanes_total<LPR>(acc[r]);
        if (conv) {
            float f[R];
#pragma unroll
            for (int r = 0; r < R; ++r) f[r] = lanes_total<LPR>(past[r]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int row = row0 + r, ch = row - e.conv_from;
                if (ch < 0 || ch >= e.channels || row >= a.rows) continue;
                if (a.bias) acc[r] += a.bias[row];
                if (l == 0) e.ring[(size_t)(pos % e.taps) * e.channels + ch] = acc[r];  // (no earlier position's slot)
                acc[r] = acc[r] * e.conv[(size_t)(e.taps - 1) * e.channels + ch] + f[r];
            }
            if (g + n_wg * 4 < p.groups) fetch_past(g + n_wg * 4);
        }
        if (R > 1 && (MORE ? row0 < a.gated : a.gated)) {
            if (l == 0)
#pragma unroll
                for (int r = 0; r + 1 < R; r += 2) {
                    const int row = row0 + r;  // (even, and so is the number of rows in pairs, in whole groups)
                    if (row >= a.rows) continue;
                    const float b0 = a.bias ? a.bias[row] : 0.f, b1 = a.bias ? a.bias[row + 1] : 0.f;
                    a.y[(size_t)b * a.y_batch + (row >> 1)] = activate(acc[r] + b0, a.act0) * (acc[r + 1] + b1);
                }
        } else if (l == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int row = row0 + r, ch = row - e.conv_from;
                if (row >= a.rows) continue;
                float v = acc[r];
                if (a.bias && (!conv || ch < 0 || ch >= e.channels)) v += a.bias[row];
                const int act = MORE && row >= e.act2_from ? e.act2 : row < a.act_split ? a.act0 : a.act1;
                v = MORE && act == BITNET_HIP_ACT_XIELU ? activate(v, act, late()->a.more.act_a, late()->a.more.act_b) : activate(v, act);
                if (mul) {
                    const auto &f = late()->a.more;
                    v *= bf2f(f.mul[(size_t)min(max(f.mul_tokens[mul_at], 0), f.mul_rows - 1) * f.ld_mul + row]);
                }
                a.y[(size_t)b * a.y_batch + row - (MORE ? a.gated >> 1 : 0)] = v;
                if (a.best_val) {
                    const float t = v != v ? -INFINITY : v;
                    if (t > bv || (t == bv && row < bi)) {
                        bv = t;
                        bi = row;
                    }
                }
            }
        }
    }
    if (a.best_val) {
        // one candidate per row group of lanes, then per wave
#pragma unroll
        for (int off = 32; off >= LPR; off >>= 1) {
            const float ov = __shfl_xor(bv, off, 64);
            const int oi = __shfl_xor(bi, off, 64);
            if (ov > bv || (ov == bv && oi < bi)) {
                bv = ov;
                bi = oi;
            }
        }
        if (lane == 0) {
            wbv[wave] = bv;
            wbi[wave] = bi;
        }
        __syncthreads();
        if (tid == 0) {
            for (int i = 1; i < 4; ++i)
                if (wbv[i] > bv || (wbv[i] == bv && wbi[i] < bi)) {
                    bv = wbv[i];
                    bi = wbi[i];
                }
            a.best_val[blockIdx.x] = bv;
            a.best_idx[blockIdx.x] = bi;
        }
    }
}

// A plain vector needs no norm ahead of the products, so it does not go through LDS either: the four waves of a workgroup share its R rows' columns, chunk by chunk of 512, a lane takes the
// vector's elements at its own columns to registers, and vector, bias and weights are requested at once (U chunks per wave in flight).  Launch and one latency bound it below 1 MB of
// weights, memory above.  us, k_dense_gemv / this form: 64 x 3072 3.7 / 2.7, 1536 x 1536 4.0 / 3.3, 2560 x 2560 5.4 / 5.2, 3072 x 8192 11.6 / 11.1, 6912 x 2560 9.4 / 8.8,
// 32768 x 16384 195 / 159; steps: Lasapel 1b 176.6 -> 171.6, 3b 273.6 -> 268.9, Lurepel 1b at 900 keys 162.3 -> 158.3, Sipelorn 1b 242.7 -> 237.
template <int R, int U>
__global__ __launch_bounds__(256, 3) void k_dense_gemv_plain(GemvPlainK p) {
    __shared__ float parts[4][R];
    asm volatile("" ::"s"(p.x), "s"(p.w), "s"(p.bias), "s"(p.y), "s"(p.rows), "s"(p.cols), "s"(p.ld), "s"(p.act0), "s"(p.act1), "s"(p.act_split));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), row0 = blockIdx.x * R, row = row0 + tid;
    const int chunks = (p.cols + 511) / 512, batches = ((chunks + 3) / 4 + U - 1) / U;
    // What a lane has past the columns counts for nothing, an infinite weight included.  With one chunk per wave it is zero, out of a buffer load's bounds; else it is the row's last
    // columns again, and the sum stays as it was.  us with bounds / by choice: 16384 x 512 6.1 / 6.5, 13824 x 640 5.8 / 6.1; 2560 x 6912 8.8 / 8.2, 4096 x 5120 9.4 / 8.8.
    constexpr bool BOUNDED = U == 1;
    float bias = 0.f, acc[R];
    if (p.bias) bias = p.bias[min(row, p.rows - 1)];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    for (int b = 0; b < batches; ++b) {
        u32x4 w[U][R];
        f32x4 v[U][2];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = (wave + 4 * (U * b + u)) * 512 + lane * 8;
            const unsigned col = min(at, p.cols - 8);
            in[u] = at < p.cols;
            v[u][0] = *reinterpret_cast<const f32x4 *>(p.x + col), v[u][1] = *reinterpret_cast<const f32x4 *>(p.x + col + 4);
            const uint16_t *wr = p.w + (size_t)row0 * p.ld;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                w[u][r] = BOUNDED ? __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bounded(wr, p.cols * 2), 2 * at, 0, kBufferNt))
                                  : __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wr + col));
                if (row0 + r + 1 < p.rows) wr += p.ld;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            f32x4 x[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) x[h] = in[u] ? v[u][h] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float t = acc[r];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    t = fmaf(x[c >> 1][2 * c & 3], __builtin_bit_cast(float, w[u][r][c] << 16), t);
                    t = fmaf(x[c >> 1][(2 * c & 3) + 1], __builtin_bit_cast(float, w[u][r][c] & 0xffff0000u), t);
                }
                if (!BOUNDED) asm volatile("" : "+v"(t));  // (a choice below, not a branch, which would take the loads along)
                acc[r] = BOUNDED || in[u] ? t : acc[r];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float t = lanes_total<64>(acc[r]);
        if (lane == 0) parts[wave][r] = t;
    }
    __syncthreads();
    if (tid < R && row < p.rows)
        p.y[row] = activate(((parts[0][tid] + parts[1][tid]) + (parts[2][tid] + parts[3][tid])) + bias, row < p.act_split ? p.act0 : p.act1);
}

// LPR lanes per row take rows of up to 64, 256 and any number of columns: one, two and five steps at the most are needed of them
template <int LPR, int R, bool MORE>
static void gemv_go(int u, const GemvK &k, dim3 grid, hipStream_t s) {
    const size_t lds = (size_t)k.kp * 4;
    void (*fn)(GemvK);
    if constexpr (LPR == 64) {
        auto pick = [&](auto nr) {
            constexpr int NR = decltype(nr)::value;
            return u == 1 ? k_dense_gemv<64, R, 1, MORE, NR> : u == 2 ? k_dense_gemv<64, R, 2, MORE, NR> : u == 3 ? k_dense_gemv<64, R, 3, MORE, NR>
                 : u == 4 ? k_dense_gemv<64, R, 4, MORE, NR> : k_dense_gemv<64, R, 5, MORE, NR>;
        };
        fn = k.a.in.n <= 3072 ? pick(std::integral_constant<int, 3>()) : pick(std::integral_constant<int, 4>());
    } else {
        fn = LPR == 16 && u > 1 ? k_dense_gemv<LPR, R, 2, MORE, 1> : k_dense_gemv<LPR, R, 1, MORE, 1>;
    }
    if (lds > 65536) (void)hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(fn, grid, dim3(256), lds, s, k);
}

static bool gemv_has_more(const GemvArgs &a) {
    const bool pairs = a.gated && a.gated < a.rows;
    return a.in.y_gate || pairs || a.more.conv || a.more.mul || a.more.act2_from < a.rows || a.act0 == BITNET_HIP_ACT_XIELU || a.act1 == BITNET_HIP_ACT_XIELU;
}

template <int LPR, int R>
static void gemv_pick_u(int u, const GemvK &k, dim3 grid, hipStream_t s) {
    if (gemv_has_more(k.a))
        gemv_go<LPR, R, true>(u, k, grid, s);
    else
        gemv_go<LPR, R, false>(u, k, grid, s);
}

// What k_dense_gemv_plain takes: a vector as it lies there, it and the weights on 16 bytes, no epilogue beyond bias and activation, rows of more than half a wave.  Many short rows stay with k_dense_gemv, whose
// workgroups take several groups of them, us there / here: 16384 x 512 6.8 / 6.1, 65536 x 520 17.5 / 17.5, x 768 20.1 / 18.7, 128256 x 264 23 / 31, x 512 26 / 33, x 520 27.9 / 31.6,
// x 640 29.4 / 32.4, x 768 33.8 / 34.6, x 1024 43 / 38.  One, two or four rows per workgroup:
// us with R = 1, 2, 4 at 512 x 1536 2.8, 2.9, 3.0, 1024 x 4096 4.0, 4.0, 4.0, 2560 x 6912 11.4, 9.0, 9.4, 3072 x 8192 14.3, 11.4, 11.1, 16384 x 4096 27.9, 24.8, 23.4.
static bool gemv_is_plain(const GemvArgs &a) {
    return a.in.kind == BITNET_HIP_IN_PLAIN && (((uintptr_t)a.in.x | (uintptr_t)a.w) & 15) == 0 && a.batch == 1 && !a.gated && !a.best_val && !a.latent && !a.more.conv && !a.more.mul &&
           a.cols > (a.rows <= 16384 ? 256 : a.rows <= 65536 ? 512 : 768) && a.more.act2_from >= a.rows && a.act0 != BITNET_HIP_ACT_XIELU && a.act1 != BITNET_HIP_ACT_XIELU;
}

template <int R>
static hipError_t gemv_plain_go(const GemvArgs &a, hipStream_t s) {
    GemvPlainK k{a.in.x, a.bias, a.w, a.y, a.rows, a.cols, a.ld, a.act0, a.act1, a.act_split ? a.act_split : a.rows};
    const int each = ((a.cols + 511) / 512 + 3) / 4;
    auto fn = each <= 1 ? k_dense_gemv_plain<R, 1> : each <= 2 ? k_dense_gemv_plain<R, 2> : each <= 3 || each == 5 || each == 6 ? k_dense_gemv_plain<R, 3> : k_dense_gemv_plain<R, 4>;
    hipLaunchKernelGGL(fn, dim3((a.rows + R - 1) / R), dim3(256), 0, s, k);
    return hipGetLastError();
}

// A vector that is formed on the way -- summed, normed, gated -- without going through LDS: wave w of a workgroup takes the columns of the chunks w, w + waves, .. of 512 of ALL its rows, a lane forms
// the vector at its own eight columns per chunk in registers, once, and keeps it for the workgroup's rows, which follow one another four at a time, the next four on their way.  Requests go out in the
// order vectors, what the rows' ends need, weights.  What an rms norm divides by follows the product, so its sum costs no meeting of the waves; a layer norm's mean and squares about it are put together
// from the waves' own means in one.  The waves' partial sums meet in LDS once, behind the last row, and a thread finishes each row.  Bound by the launch and two dependent latencies below some
// 10 MB, by memory above.  us per launch in a chain, k_dense_gemv / this form, rms norm | added and normed twice | layer norm of a sum:
//   256 x 2560 4.0 / 2.9 | 5.0 / 3.9 | 4.9 / 4.1    1932 x 1536 4.5 / 3.5 | 5.6 / 4.5 | 5.3 / 4.5    2112 x 2560 6.0 / 4.7 | 7.5 / 5.9 | 7.2 / 5.6    5376 x 1536 6.6 / 5.2 | 7.9 / 6.1 | 7.5 / 6.0
//   6912 x 2560 9.5 / 8.1 | 10.4 / 9.1 | 10.2 / 9.1    10240 x 2560 13.4 / 11.2 | 15.0 / 12.0 | 14.4 / 11.7    12288 x 3072 15.4 / 15.8 | 16.4 / 16.0 | 15.8 / 15.4    3072 x 6144 14.5 / 8.3 | 22.8 / 9.9 | 21.6 / 10.3
struct GemvFormK {
    GemvArgs a;
    LatentRows lat;
    int rows_wg;  // rows of a workgroup, a multiple of R
    int lat_wg;   // workgroup index that writes the latent row, or -1
};
constexpr int kFormedRows = 256;  // most rows of a workgroup (a thread finishes each, so no more than its threads either)

// R rows at a time, U chunks per wave; NORM: 0 none, 1 rms, 2 layer norm; MORE as k_dense_gemv's
template <int R, int U, int NORM, bool MORE>
__global__ __launch_bounds__(512) void k_dense_gemv_formed(GemvFormK p) {
    __shared__ __attribute__((aligned(16))) float slots[4][8];
    __shared__ __attribute__((aligned(16))) float parts[kFormedRows + R][8];
    const GemvArgs &a = p.a;
    const VecIn &in = a.in;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = (int)blockDim.x >> 6;
    asm volatile("" ::"s"(in.x), "s"(in.y), "s"(in.post_weight), "s"(in.scale), "s"(in.weight), "s"(in.bias), "s"(in.gate), "s"(in.x_out), "s"(in.kind), "s"(in.n), "s"(in.mean_n), "s"(a.w),
                 "s"(a.rows), "s"(a.cols), "s"(a.ld), "s"(p.rows_wg), "s"(p.lat_wg), "s"(a.bias));
    if ((int)blockIdx.x == p.lat_wg) {  // (four waves)
        if (p.lat.f32) {
            if (p.lat.cq) latent_queries<float>(p.lat, 0, slots[0]);
            latent_row<float>(p.lat, 0, slots[0]);
        } else {
            if (p.lat.cq) latent_queries<uint16_t>(p.lat, 0, slots[0]);
            latent_row<uint16_t>(p.lat, 0, slots[0]);
        }
        return;
    }
    const int row0 = blockIdx.x * p.rows_wg, n_rows = min(p.rows_wg, a.rows - row0);
    const bool writer = blockIdx.x == 0;
    int col[U];
    bool inside[U];
#pragma unroll
    for (int u = 0; u < U; ++u) col[u] = (wave + nw * u) * 512 + lane * 8, inside[u] = col[u] < a.cols;
    typedef f32x4 Vec[U][2];
    const int bytes = in.n * 4;
    auto load = [&](Vec &v, const float *from, int behind = 0) {  // (elements ahead of `behind` have offsets past any buffer's end)
        const auto r = bounded(from, bytes);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) v[u][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, 4 * (col[u] - behind) + 16 * h, 0, 0));
    };
    const bool added = in.kind >= BITNET_HIP_IN_RESIDUAL_NORM && in.y, normed = added && in.post_weight, scaled = normed && in.scale, y_gated = MORE && added && in.y_gate;
    const bool gated = NORM && in.gate, shifted = NORM == 2 && in.bias, two = NORM == 0 && in.kind == BITNET_HIP_IN_CONCAT;
    Vec xv, yv, pw, sc, yg, wv, bv, gv;
    load(xv, in.x);
    if (added) load(yv, in.y);
    if (normed) load(pw, in.post_weight);
    if (scaled) load(sc, in.scale);
    if (y_gated) load(yg, in.y_gate);
    if (NORM) load(wv, in.weight);
    if (two) load(wv, in.x2, in.n);
    if (shifted) load(bv, in.bias);
    if (gated) load(gv, in.gate);
    // a thread finishes one row: what it needs for that
    const Epilogue &e = a.more;
    const int row = row0 + tid;
    const bool finishes = tid < n_rows;
    const bool conv = MORE && e.conv, mul = MORE && e.mul;
    float bias = 0.f;
    if (a.bias && finishes) bias = a.bias[row];
    constexpr int TAPS = 3;  // earlier positions of a convolution requested ahead
    int pos = 0;
    const int ch = MORE ? row - e.conv_from : -1;
    const bool convolved = conv && finishes && ch >= 0 && ch < e.channels;
    float past[TAPS], tap[TAPS], last_tap = 0.f;
    if (conv) {
        pos = *e.pos;
        if (convolved) {
            last_tap = e.conv[(size_t)(e.taps - 1) * e.channels + ch];
#pragma unroll
            for (int j = 0; j < TAPS; ++j) {  // (j + 1 positions back)
                const int at = pos - 1 - j, t = e.taps - 2 - j;
                past[j] = 0.f, tap[j] = 0.f;
                if (t >= 0 && at >= 0) past[j] = e.ring[(size_t)(at % e.taps) * e.channels + ch], tap[j] = e.conv[(size_t)t * e.channels + ch];
            }
        }
    }
    int mul_token = 0;
    if (mul) mul_token = e.mul_tokens[*e.mul_at];
    SharedRows<R, U> weights(a.w + (size_t)row0 * a.ld, n_rows, a.ld, col, inside);
    weights.request();
    auto squares = [&](const Vec &v) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) ss += (v[u][h].x * v[u][h].x + v[u][h].y * v[u][h].y) + (v[u][h].z * v[u][h].z + v[u][h].w * v[u][h].w);
        return ss;
    };
    auto total = [&](const float *slot) { return waves_total(slot, nw); };
    const float count = (float)in.mean_n;
    auto inverse = [&](float ss) { return 1.0f / sqrtf(ss / count + in.eps); };
    if (added) {
        float inv = 1.f;
        if (normed) {
            const float t = wave_sum(squares(yv));
            if (lane == 0) slots[0][wave] = t;
            __syncthreads();
            inv = inverse(total(slots[0]));
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4 v = yv[u][h] * (normed ? inv : in.mult);
                if (normed) v *= in.offset + pw[u][h];
                if (scaled) v *= sc[u][h];
                if (y_gated) v *= yg[u][h];
                xv[u][h] += v;
                if (writer && in.x_out && col[u] < in.n) *reinterpret_cast<f32x4 *>(in.x_out + col[u] + 4 * h) = xv[u][h];
            }
    }
    if (two)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) xv[u][h] += wv[u][h];
    if (NORM == 1) {  // what it is divided by follows the product
        const float t = wave_sum(squares(xv));
        if (lane == 0) slots[2][wave] = t;
    }
    float mean = 0.f, inv = 1.f;
    if (NORM == 2) {
        // sums of a wave's own columns and of its squares about its own mean, put together without a second meeting
        auto columns = [&](int wv_) {
            int c = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) c += min(max(a.cols - (wv_ + nw * u) * 512, 0), 512);
            return (float)c;
        };
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) s += (xv[u][h].x + xv[u][h].y) + (xv[u][h].z + xv[u][h].w);
        s = wave_sum(s);
        const float own = s / fmaxf(columns(wave), 1.f);
        Vec d;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) d[u][h] = inside[u] ? xv[u][h] - own : f32x4{0.f, 0.f, 0.f, 0.f};
        const float m2 = wave_sum(squares(d));
        if (lane == 0) slots[1][wave] = s, slots[3][wave] = m2;
        __syncthreads();
        mean = total(slots[1]) / count;
        float ss = total(slots[3]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float c = columns(i), off = slots[1][i] / fmaxf(c, 1.f) - mean;
            ss += i < nw && c > 0.f ? c * (off * off) : 0.f;
        }
        inv = inverse(ss);
    }
    if (NORM) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4 v = NORM == 2 ? (xv[u][h] - mean) * inv : xv[u][h];
                v *= in.offset + wv[u][h];
                if (gated) v *= gv[u][h];
                if (shifted) v += bv[u][h];
                xv[u][h] = v;
                if (NORM == 2 && writer && in.h_out && inside[u]) *reinterpret_cast<f32x4 *>(in.h_out + col[u] + 4 * h) = v;
            }
    }
    weights.run(xv, parts, wave, lane);
    __syncthreads();
    if (NORM == 1) {
        inv = inverse(total(slots[2]));
        if (writer && in.h_out)
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (inside[u]) *reinterpret_cast<f32x4 *>(in.h_out + col[u] + 4 * h) = xv[u][h] * inv;
    }
    auto sum = [&](int r) {
        const float t = total(parts[r]);
        return NORM == 1 ? t * inv : t;
    };
    float best = -INFINITY;
    int best_row = 0x7fffffff;
    if (finishes && row < a.gated) {  // (even, and so are the rows in pairs and those of a workgroup)
        if (tid & 1) return;
        const float up_bias = a.bias ? a.bias[row + 1] : 0.f;
        a.y[row >> 1] = activate(sum(tid) + bias, a.act0) * (sum(tid + 1) + up_bias);
    } else if (finishes) {
        float v = sum(tid) + bias;
        if (convolved) {
            float f = 0.f;
            for (int j = e.taps - 2; j >= TAPS; --j) {
                const int at = pos - 1 - j;
                if (at >= 0) f += e.conv[(size_t)(e.taps - 2 - j) * e.channels + ch] * e.ring[(size_t)(at % e.taps) * e.channels + ch];
            }
#pragma unroll
            for (int j = TAPS - 1; j >= 0; --j) f += tap[j] * past[j];
            e.ring[(size_t)(pos % e.taps) * e.channels + ch] = v;  // (no earlier position's slot)
            v = v * last_tap + f;
        }
        const int act = MORE && row >= e.act2_from ? e.act2 : row < a.act_split ? a.act0 : a.act1;
        v = MORE && act == BITNET_HIP_ACT_XIELU ? activate(v, act, e.act_a, e.act_b) : activate(v, act);
        if (mul) v *= bf2f(e.mul[(size_t)min(max(mul_token, 0), e.mul_rows - 1) * e.ld_mul + row]);
        a.y[row - (a.gated >> 1)] = v;
        best = v != v ? -INFINITY : v;
        best_row = row;
    }
    if (a.best_val) {  // (no pairs)
        auto better = [&](float v, int i) {
            if (v > best || (v == best && i < best_row)) best = v, best_row = i;
        };
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const float v = __shfl_xor(best, off, 64);
            const int i = __shfl_xor(best_row, off, 64);
            better(v, i);
        }
        if (lane == 0) slots[0][wave] = best, slots[1][wave] = __builtin_bit_cast(float, best_row);
        __syncthreads();
        if (tid == 0) {
            for (int i = 1; i < nw; ++i) better(slots[0][i], __builtin_bit_cast(int, slots[1][i]));
            a.best_val[blockIdx.x] = best;
            a.best_idx[blockIdx.x] = best_row;
        }
    }
}

struct FormedSplit {
    int u, waves;  // chunks of 512 columns per wave
};
static FormedSplit formed_split(const GemvArgs &a) {
    const int chunks = (a.cols + 511) / 512, most = a.latent ? 4 : 8, u = (chunks + most - 1) / most;
    return {u, a.latent ? 4 : (chunks + u - 1) / u};
}
// What k_dense_gemv_formed takes: a vector to be formed, whole in eights, it and the weights on 16 bytes (a lane's columns are inside or outside as one, and loads past the end give zeros, so that an
// infinite weight counts for its own row alone), more than half a wave's columns and no more than two chunks for each of eight waves.  Past 2^26 weights (a head) memory is all that
// counts and k_dense_gemv, whose waves take whole rows, is as fast or faster: us there / here 32768 x 1536 21.7 / 18.9, 16384 x 2560 17.8 / 15.8, 32768 x 3072 35.9 / 36.7, 128256 x 2560 100.2 / 101.2.
// Below, of 10 widths from 1024 to 8192 columns by 8 sizes from 4 to 64 million weights and 28 round shapes, this form is faster at all but one: 3072 columns behind one rms norm where k_dense_gemv's
// rounds of 3072 rows are whole, 11264 rows 14.56 / 14.60, 12000 14.5 / 14.9, 12288 15.2 / 15.4, and 12289 15.6 / 15.2, 13029 17.4 / 15.7 again; no line by sizes keeps those rows and no others.
static bool gemv_is_formed(const GemvArgs &a) {
    const VecIn &in = a.in;
    const uintptr_t all = (uintptr_t)in.x | (uintptr_t)in.y | (uintptr_t)in.post_weight | (uintptr_t)in.scale | (uintptr_t)in.y_gate | (uintptr_t)in.weight | (uintptr_t)in.bias |
                          (uintptr_t)in.gate | (uintptr_t)in.x2 | (uintptr_t)in.x_out | (uintptr_t)in.h_out | (uintptr_t)a.w;
    return in.kind != BITNET_HIP_IN_PLAIN && in.n % 8 == 0 && (in.kind == BITNET_HIP_IN_CONCAT ? 2 : 1) * in.n == a.cols && a.cols > 256 && a.cols <= 8192 && (all & 15) == 0 && a.batch == 1 &&
           (!a.latent || a.cols <= 4096) && (!a.best_val || a.rows <= 1024 * std::min(64 * formed_split(a).waves, kFormedRows)) && (size_t)a.rows * a.cols <= ((size_t)1 << 26) &&
           (!a.more.conv || a.more.conv_from >= a.gated) && (size_t)kFormedRows * a.ld < ((size_t)1 << 30);
}

template <int R, int U>
static void gemv_formed_go(const GemvFormK &k, dim3 grid, dim3 block, hipStream_t s) {
    const GemvArgs &a = k.a;
    const int norm = a.in.kind == BITNET_HIP_IN_RESIDUAL || a.in.kind == BITNET_HIP_IN_CONCAT ? 0 : a.in.center ? 2 : 1;
    void (*fn)(GemvFormK) = gemv_has_more(a) ? (norm == 0 ? k_dense_gemv_formed<R, U, 0, true> : norm == 1 ? k_dense_gemv_formed<R, U, 1, true> : k_dense_gemv_formed<R, U, 2, true>)
                                             : (norm == 0 ? k_dense_gemv_formed<R, U, 0, false> : norm == 1 ? k_dense_gemv_formed<R, U, 1, false> : k_dense_gemv_formed<R, U, 2, false>);
    hipLaunchKernelGGL(fn, grid, block, 0, s, k);
}

static hipError_t launch_gemv_formed(const GemvArgs &a, int *n_wg_out, hipStream_t s) {
    GemvFormK k;
    k.a = a;
    k.a.latent = nullptr;
    if (a.act_split == 0) k.a.act_split = a.rows;
    if (k.a.in.mean_n == 0) k.a.in.mean_n = a.in.n;
    const auto [u, waves] = formed_split(a);
    // Up to 256 rows a row per CU.  Else steps of four rows, one or two workgroups per CU (of one or two waves up to four), the count that leaves a CU the fewest steps in turn: a launch lasts as long as
    // the CUs with the most.  One workgroup has no other's loads to hide its sums behind (1.15), but of five waves and more a second one is worth its forming from two steps on only.  us, rows per
    // workgroup: 2112 x 2560 12 5.9, 8 6.3; 2560 x 2560 12 6.1, 8 6.3, 4 6.6; 4096 x 1536 8 5.3, 16 5.5, 4 5.7; 5000 x 3072 20 8.6, 12 8.9; 6912 x 2560 16 9.1, 28 9.6, 36 10.1;
    // 3000 x 512 4 3.4, 12 4.6; 12000 x 1024 12 6.7, 16 7.1, 24 7.3.  One, two or four rows at a time: 1932 x 1536 5.2, 4.7, 4.5; 10240 x 2560 12.9, 12.4, 11.5.
    const bool single = a.rows <= 256 && !a.gated;
    int each = 1;
    if (!single) {
        double least = 0;
        for (int per = 1; per <= (waves <= 2 ? 4 : 2); ++per) {
            const int n = (a.rows + 1024 * per - 1) / (1024 * per);
            if (per > 1 && n == 1 && waves >= 5) break;
            const double cost = per * n * (per == 1 ? 1.15 : 1.0);
            if (per == 1 || cost <= least) least = cost, each = 4 * n;
        }
        each = std::min({each, 64 * waves, kFormedRows});
        // Workgroups that begin a multiple of 256 KiB apart wait for the same memory where two per CU run at once, or nearly: four rows more.  us, k_dense_gemv / without / with it, rms norm | added and
        // normed twice: 16384 x 4096 25.6 / 27.7 / 23.3 | 25.7 / 26.4 / 24.1, 15000 x 4096 23.5 / 23.9 / 22.0 | 25.0 / 23.6 / 22.6, 8192 x 8192 32.5 / 30.8 / 24.8 | 43.6 / 31.6 / 26.9.  Fewer
        // workgroups: 7000 x 8192 (438) 24.6 / 23.8 | 25.9 / 25.8, 6200 x 8192 (388) 23.1 / 23.3 | 24.7 / 25.3.
        if ((size_t)each * a.ld * 2 % ((size_t)1 << 18) == 0 && (a.rows + each - 1) / each > 448 && each + 4 <= std::min(64 * waves, kFormedRows)) each += 4;
    }
    k.rows_wg = each;
    const int n_wg = (a.rows + each - 1) / each;
    if (n_wg_out) *n_wg_out = n_wg;
    k.lat_wg = a.latent ? n_wg : -1;
    if (a.latent) k.lat = *a.latent;
    const dim3 grid(n_wg + (a.latent ? 1 : 0)), block(64 * waves);
    if (u == 1)
        single ? gemv_formed_go<1, 1>(k, grid, block, s) : gemv_formed_go<4, 1>(k, grid, block, s);
    else
        single ? gemv_formed_go<1, 2>(k, grid, block, s) : gemv_formed_go<4, 2>(k, grid, block, s);
    return hipGetLastError();
}

hipError_t launch_dense_gemv(const GemvArgs &a, int *n_wg_out, hipStream_t s) {
    if (gemv_is_plain(a)) return a.rows >= 3072 ? gemv_plain_go<4>(a, s) : a.rows > 512 ? gemv_plain_go<2>(a, s) : gemv_plain_go<1>(a, s);
    if (gemv_is_formed(a)) return launch_gemv_formed(a, n_wg_out, s);
    GemvK k;
    k.a = a;
    k.a.latent = nullptr;
    if (a.act_split == 0) k.a.act_split = a.rows;
    if (k.a.in.mean_n == 0) k.a.in.mean_n = a.in.n;
    const int lpr = a.cols <= 64 ? 8 : a.cols <= 256 ? 16 : 64;
    const int chunks = (a.cols + lpr * 8 - 1) / (lpr * 8);
    int u = chunks < 5 ? chunks : 5;
    if (chunks > 5)
        for (int c = 4; c >= 3; --c)
            if ((chunks + c - 1) / c * c < (chunks + u - 1) / u * u) u = c;
    const int step = lpr * 8 * u;
    k.kp = (a.cols + step - 1) / step * step;
    if ((size_t)k.kp * 4 > 150 * 1024) return hipErrorInvalidValue;
    // rows per lane group: enough workgroups to reach every CU twice, then more rows in flight per wave
    const int per = 64 / lpr;
    auto wgs = [&](int r) { return ((long)a.rows + 4l * per * r - 1) / (4l * per * r) * a.batch; };
    int r = 1;
    if (wgs(4) >= 1024) r = 4;
    else if (wgs(2) >= 512 || a.gated) r = 2;
    k.groups = (a.rows + per * r - 1) / (per * r);
    int n_wg = (k.groups + 3) / 4;
    const int cap = 768;  // three workgroups per CU: each forms the whole input again (measured: 512 and 1024 are slower)
    if (a.batch == 1 && n_wg > cap) {
        const int rounds = (n_wg + cap - 1) / cap;
        n_wg = (n_wg + rounds - 1) / rounds;
    }
    if (n_wg_out) *n_wg_out = n_wg;
    k.lat_wg = a.latent ? n_wg : -1;
    if (a.latent) k.lat = *a.latent;
    const dim3 grid(n_wg + (a.latent ? 1 : 0), a.batch);
    if (lpr == 8)
        r == 4 ? gemv_pick_u<8, 4>(u, k, grid, s) : r == 2 ? gemv_pick_u<8, 2>(u, k, grid, s) : gemv_pick_u<8, 1>(u, k, grid, s);
    else if (lpr == 16)
        r == 4 ? gemv_pick_u<16, 4>(u, k, grid, s) : r == 2 ? gemv_pick_u<16, 2>(u, k, grid, s) : gemv_pick_u<16, 1>(u, k, grid, s);
    else
        r == 4 ? gemv_pick_u<64, 4>(u, k, grid, s) : r == 2 ? gemv_pick_u<64, 2>(u, k, grid, s) : gemv_pick_u<64, 1>(u, k, grid, s);
    return hipGetLastError();
}

// ---- many-row matmul --------------------------------------------------------------------------------------------------
// C[m][n] = act(A[m][k] . W[n][k]^T + bias).  Workgroup tile TN x TM in WN x WM waves, K steps of 64 columns staged in LDS by LDS-DMA,
// ST buffers; from 256 x 256 in eight waves of 128 x 64 (half the bytes per product of 128 x 128, and a fragment read from LDS feeds
// four to eight MFMAs) down to 64 x 64 with four buffers, the one that fills the chip best (launch_dense_gemm).  LDS image of a row: eight 16-byte units, unit q stored at
// q ^ ((row >> 1) & 7) (activations) or q ^ weight_key(row) (weights): the sixteen rows of a ds_read_b128 cover all 64 banks once.  The
// MFMA's A operand is the weight tile (rows = output columns n), its B operand the activation tile; for bf16
// outputs row r of weight fragment i is column 4 FN (r / 4) + 4 i + r % 4 of the wave's tile, so that a lane ends up with 4 FN consecutive
// columns of one output row (stores of 32-byte pieces cost more than the arithmetic of a short product); f32 outputs keep 16 i + r, four
// lanes of 16 bytes side by side.
constexpr int kTileK = 64;

// 64 lanes x 16 bytes from (scalar base + lane offset) to LDS bytes [lds_dst, lds_dst + 1024); invisible to hipcc's vmcnt bookkeeping
__device__ __forceinline__ void dma1k(unsigned lane_off, const void *sbase, unsigned lds_dst) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(lane_off), "s"(sbase), "s"(lds_dst)
                 : "memory");
}

template <int FN, bool CF32>
__device__ __forceinline__ int weight_key(int row) {
    return CF32 ? (row >> 1) & 7 : ((row / (4 * FN)) & 3) * 2 + ((row >> 1) & 1);
}

// The activations of the matmul's epilogues, the same in every tile and in the form for few rows: a call's results do not hang on the launcher's choice.
// v_exp and v_rcp where the call allows them; exp(v) - 1 of xIELU loses what a bf16 output does not keep.
__device__ __forceinline__ float sigmoid_fast(float v) { return __builtin_amdgcn_rcpf(1.0f + __expf(-v)); }
__device__ __forceinline__ float silu_fast(float v) { return v * sigmoid_fast(v); }
__device__ __forceinline__ float gelu_fast(float v) { return v * sigmoid_fast(2.0f * gelu_argument(v)); }
__device__ __forceinline__ float xielu_fast(float v, const Epilogue &e) { return 0.5f * v + (v > 0.f ? e.act_a * v * v : e.act_b * (__expf(v) - 1.0f - v)); }
// gated columns
__device__ __forceinline__ float activate_pair(float v, int act) {
    return act == BITNET_HIP_ACT_SILU ? silu_fast(v) : act == BITNET_HIP_ACT_GELU_TANH ? gelu_fast(v) : activate(v, act);
}
// The fast GELU where one activation covers whole waves of columns in every tile (up to 128 of them); a wave that two activations or the last column run
// through has always taken expf and a division, and its tile must not decide.
__device__ __forceinline__ bool gelu_is_fast(const GemmArgsD &p) { return p.act_split >= p.n && p.n % 128 == 0; }
__device__ __forceinline__ float activate_column(float v, int act, bool fast_gelu, const Epilogue &e) {
    const float sg = sigmoid_fast(v), r = fmaxf(v, 0.0f);
    return act == BITNET_HIP_ACT_SILU ? v * sg : act == BITNET_HIP_ACT_SIGMOID ? sg : act == BITNET_HIP_ACT_RELU2 ? r * r : act == BITNET_HIP_ACT_XIELU ? xielu_fast(v, e)
         : act == BITNET_HIP_ACT_GELU_TANH && fast_gelu ? gelu_fast(v) : activate(v, act);
}

__host__ __device__ __forceinline__ bool rows_on_16_bytes(const void *c, size_t ldc, size_t c_batch, bool f32) {
    const size_t mask = f32 ? 3 : 7;
    return ((ldc | c_batch) & mask) == 0 && ((uintptr_t)c & 15) == 0;
}

// GROUPED: the row tiles come from a device list, (matrix, first row, rows) each; a matrix's tiles follow one another.
// GATED (bf16 outputs): columns 2 i and 2 i + 1 make column i of the output.
// MUL (bf16 outputs): row i of the output is multiplied by a table's row, the one of its token.
template <int TN, int TM, int WN, int WM, int ST, bool CF32, bool GROUPED = false, bool GATED = false, bool MUL = false>
__global__ __launch_bounds__(64 * WN * WM, 2) void k_dense_gemm(GemmArgsD p, int tiles_n, int tiles_m, int swizzle) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    constexpr int NW = WN * WM, DN = TN / NW / 8, DM = TM / NW / 8;  // DMA instructions per wave and step (eight rows each)
    constexpr int FN = TN / WN / 16, FM = TM / WM / 16;              // 16-row fragments per wave
    constexpr unsigned ABUF = TM * 128, BUF = ABUF + TN * 128;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup -> tile: consecutive workgroups land on the eight XCDs in turn; give each XCD a contiguous run of tiles, and walk
    // the tiles in groups of eight row tiles so that what runs together shares both operands in the XCD's L2
    int id = blockIdx.x;
    int m0, n0, m_end;
    const uint16_t *A = (const uint16_t *)p.a + (size_t)blockIdx.y * p.a_batch;
    const uint16_t *W = p.w + (size_t)blockIdx.y * p.w_batch;
    if (GROUPED) {
        const int total = *p.n_tiles * tiles_n, per = (total + 7) >> 3;
        if ((id >> 3) >= per) return;
        id = (id & 7) * per + (id >> 3);
        if (id >= total) return;
        const int4 tile = p.tiles[id / tiles_n];
        m0 = tile.y, m_end = tile.y + tile.z, n0 = id % tiles_n * TN;
        W += (size_t)tile.x * p.w_batch;
    } else {
        const int total = tiles_n * tiles_m;
        if (swizzle) id = (id & 7) * (total >> 3) + (id >> 3);
        const int gm = 8;
        const int group = id / (gm * tiles_n), first = group * gm, size = tiles_m - first < gm ? tiles_m - first : gm;
        const int tm = first + (id % (gm * tiles_n)) % size, tn = (id % (gm * tiles_n)) / size;
        m0 = tm * TM, n0 = tn * TN, m_end = p.m;
    }
    const int drow = lane >> 3;
    // (lane offsets from the tile's first row: a tile spans less than 4 GiB; rows past the end read the tile's own rows over again)
    const unsigned rows_m = min(TM, m_end - m0), rows_n = min(TN, p.n - n0);
    const bool gathered = GROUPED && p.gather;
    const uint16_t *A0 = gathered ? A : A + (size_t)m0 * p.lda, *W0 = W + (size_t)n0 * p.ldw;
    unsigned oa[DM], ow[DN];
#pragma unroll
    for (int i = 0; i < DM; ++i) {
        const int r = wave * (TM / NW) + i * 8 + drow, unit = (lane & 7) ^ ((r >> 1) & 7);
        const unsigned row = gathered ? (unsigned)p.gather[m0 + (unsigned)r % rows_m] : (unsigned)r % rows_m;
        oa[i] = (unsigned)(row * p.lda + unit * 8) * 2;
    }
#pragma unroll
    for (int i = 0; i < DN; ++i) {
        const int r = wave * (TN / NW) + i * 8 + drow, unit = (lane & 7) ^ weight_key<FN, CF32>(r);
        ow[i] = (unsigned)((unsigned)r % rows_n * p.ldw + unit * 8) * 2;
    }
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    auto stage = [&](int t) {
        const unsigned dst = base + (t % ST) * BUF;
#pragma unroll
        for (int i = 0; i < DM; ++i) dma1k(oa[i], A0 + t * kTileK, dst + wave * (TM / NW) * 128 + i * 1024);
#pragma unroll
        for (int i = 0; i < DN; ++i) dma1k(ow[i], W0 + t * kTileK, dst + ABUF + wave * (TN / NW) * 128 + i * 1024);
    };
    const int wn = (wave % WN) * (TN / WN), wm = (wave / WN) * (TM / WM);
    const int r16 = lane & 15, g = lane >> 4, sw = (r16 >> 1) & 7;
    constexpr int FS = CF32 ? 16 : 4;  // columns between fragments; neither step changes a row's key: one for all fragments
    const int wr = CF32 ? wn + r16 : wn + (r16 >> 2) * 4 * FN + (r16 & 3);
    f32x4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int steps = p.k / kTileK;
    // Fragments are read half a step (32 columns) ahead of the MFMAs that use them, reads and MFMAs interleaved: the middle of a step
    // waits for the next tile, and the barrier there also says that every wave has left the tile whose buffer is requested next.
    bf16x8 fa[2][FM], fw[2][FN];
    auto read = [&](int t, int kk) {
        const uint8_t *la = lds + (t % ST) * BUF, *lw = la + ABUF;
        const int q = ((kk * 4 + g) ^ sw) * 16, qw = ((kk * 4 + g) ^ weight_key<FN, CF32>(wr)) * 16;
#pragma unroll
        for (int j = 0; j < FM; ++j) fa[kk][j] = *reinterpret_cast<const bf16x8 *>(la + (wm + j * 16 + r16) * 128 + q);
#pragma unroll
        for (int i = 0; i < FN; ++i) fw[kk][i] = *reinterpret_cast<const bf16x8 *>(lw + (wr + i * FS) * 128 + qw);
    };
    auto multiply = [&](int kk) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = mfma_bf16(fw[kk][i], fa[kk][j], acc[i][j]);
#pragma unroll
        for (int i = 0; i < (FN + FM) / 2; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);                         // two LDS reads
            __builtin_amdgcn_sched_group_barrier(0x008, 2 * FN * FM / (FN + FM), 0);  // their share of the MFMAs
        }
    };
#pragma unroll
    for (int t = 0; t < ST; ++t)
        if (t < steps) stage(t);
    // (loads return in order: a tile is there once at most the later ones are outstanding)
    if (steps >= ST)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 1) * (DM + DN)) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    read(0, 0);
    for (int t = 0; t < steps; ++t) {
        read(t, 1);
        multiply(0);
        if (t + ST - 1 < steps)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((ST - 2) * (DM + DN)) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        if (t + ST < steps) stage(t + ST);
        read(t + 1, 0);  // (behind the last step: bytes nobody uses)
        multiply(1);
    }
    // this lane's columns: nl + i * FS + e
    const int nl = n0 + wn + g * (CF32 ? 4 : 4 * FN), nlast = nl + (FN - 1) * FS + 3;
    const bool vec = rows_on_16_bytes(p.c, p.ldc, p.c_batch, CF32);
    // the activation: one for the whole wave unless the split runs through its columns
    const int mine = nlast < p.act_split ? p.act0 : nl >= p.act_split ? p.act1 : -1, act0 = __builtin_amdgcn_readfirstlane(mine);
    const int act = __all(mine == act0) && (act0 != BITNET_HIP_ACT_GELU_TANH || gelu_is_fast(p)) ? act0 : -1;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        const int m = m0 + wm + j * 16 + r16;
        if (m >= m_end) continue;
        const size_t o = (size_t)blockIdx.y * p.c_batch + (size_t)m * p.ldc + nl;
        if (p.bias)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] += p.bias[min(nl + i * FS + e, p.n - 1)];
        if (GATED) {
            float r[2 * FN];
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int e = 0; e < 4; e += 2) r[2 * i + e / 2] = activate_pair(acc[i][j][e], p.act0) * acc[i][j][e + 1];
            uint16_t *dst = (uint16_t *)p.c + (size_t)blockIdx.y * p.c_batch + (size_t)m * p.ldc + nl / 2;
#pragma unroll
            for (int i = 0; i < 2 * FN; i += 4) {
                if (vec && nl + 2 * i + 7 < p.n) {
                    *reinterpret_cast<bf16x4 *>(dst + i) = bf16x4{(__bf16)r[i], (__bf16)r[i + 1], (__bf16)r[i + 2], (__bf16)r[i + 3]};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (nl + 2 * (i + e) < p.n) dst[i + e] = f2bf(r[i + e]);
                }
            }
            continue;
        }
        auto apply = [&](auto f) {
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] = f(acc[i][j][e], nl + i * FS + e);
        };
        if (act < 0)
            apply([&](float v, int n) { return activate_column(v, n < p.act_split ? p.act0 : p.act1, false, p.more); });
        else if (act == BITNET_HIP_ACT_SILU)
            apply([](float v, int) { return silu_fast(v); });
        else if (act == BITNET_HIP_ACT_SIGMOID)
            apply([](float v, int) { return sigmoid_fast(v); });
        else if (act == BITNET_HIP_ACT_RELU2)
            apply([](float v, int) { return activate(v, BITNET_HIP_ACT_RELU2); });
        else if (act == BITNET_HIP_ACT_GELU_TANH)
            apply([](float v, int) { return gelu_fast(v); });
        else if (act == BITNET_HIP_ACT_XIELU)
            apply([&](float v, int) { return xielu_fast(v, p.more); });
        if (MUL) {
            const int token = min(max(p.more.mul_tokens[*p.more.mul_at + m], 0), p.more.mul_rows - 1);
            const uint16_t *mul = p.more.mul + (size_t)token * p.more.ld_mul;
            apply([&](float v, int n) { return v * bf2f(mul[min(n, p.n - 1)]); });
        }
        if (CF32) {
#pragma unroll
            for (int i = 0; i < FN; ++i) {
                float *dst = (float *)p.c + o + i * FS;
                if (vec && nl + i * FS + 3 < p.n) {
                    *reinterpret_cast<f32x4 *>(dst) = acc[i][j];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (nl + i * FS + e < p.n) dst[e] = acc[i][j][e];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < FN; i += 2) {
                uint16_t *dst = (uint16_t *)p.c + o + i * FS;
                if (vec && nl + i * FS + 7 < p.n) {
                    *reinterpret_cast<bf16x8 *>(dst) =
                        bf16x8{(__bf16)acc[i][j][0],     (__bf16)acc[i][j][1],     (__bf16)acc[i][j][2],     (__bf16)acc[i][j][3],
                               (__bf16)acc[i + 1][j][0], (__bf16)acc[i + 1][j][1], (__bf16)acc[i + 1][j][2], (__bf16)acc[i + 1][j][3]};
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (nl + i * FS + e < p.n) dst[e] = f2bf(acc[i + (e >> 2)][j][e & 3]);
                }
            }
        }
    }
}

thread_local DenseTile g_last_dense_tile;

// TM: the rows of the plan's tiles
template <int TN, int TM, int WN, int WM, int ST>
static hipError_t grouped_go(const GemmArgsD &a, hipStream_t s) {
    const int tn = (a.n + TN - 1) / TN;
    constexpr size_t lds = (size_t)ST * (TN + TM) * 128;
    auto fn = a.gated ? k_dense_gemm<TN, TM, WN, WM, ST, false, true, true> : k_dense_gemm<TN, TM, WN, WM, ST, false, true>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    g_last_dense_tile = {TN, TM, WN * WM, 1};
    hipLaunchKernelGGL(fn, dim3((tn * a.max_tiles + 7) / 8 * 8), dim3(64 * WN * WM), lds, s, a, tn, 0, 0);
    return hipGetLastError();
}
// Experts' products.  wide: the workgroups of one row tile per expert, which is what decides; measured over 46 shapes (4 to 256 experts, 128 to 6400 columns of 128 to 5632, also in pairs) at
// 2 to 400 rows per expert, us with 64 x 64 in four buffers / in three / 128 x 64 / 128 x 128 in four waves / in eight:
//   64 x 64, four buffers: what the others do not take.  8 experts, 1024 x 4096, 16 rows 21 / 28 / 53; 128, 768 x 2048, 32 rows 79 / 81 / 89
//   128 x 64 (activations serve twice the columns): where nearly every CU gets two, from as many rows on as K is long.  64, 896 x 3072, 44 rows 74 / 75 / 70; 64, 1024 x 1024, 16 rows
//     31 / 30 / 27; 64, 1536 x 448, 8 rows 21 / 20 / 19; 64, 768 x 2560, 52 rows 67 / 68 / 60.  Not with rows of whole 4 KiB, whose beginnings meet on the same channels: 256, 512 x 2048, 44 rows 114 / 117 / 136
//   64 x 64, three buffers, of which a CU takes three: one to two workgroups per CU.  8, 4096 x 1024, 16 rows 17 / 15 / 19; not with such rows either
//   128 x 128 in eight waves: one round of workgroups (64, 448 x 1536, 72 rows 31 / 31 / 28 / 29 / 23), or two to three of them for long K while an expert has one tile (64, 1408 x 2048,
//     88 rows 108 / 109 / 96 / 99 / 91)
//   128 x 128 in four waves, two workgroups per CU, which overlap their ends: 64, 896 x 3072, 88 rows 107 / 107 / 106 / 79 / 82
// In the mean 3 % behind the best form; against 64 x 64 in four buffers below 96 rows per expert and 128 x 128 in four waves from there on 5.6 % ahead, nowhere more than 6 % behind.
static hipError_t launch_grouped(const GemmArgsD &a, hipStream_t s) {
    const int experts = a.max_tiles - a.m / a.tile;  // (how a plan counts its tiles)
    const long tn = (a.n + 127) / 128, wide = experts * tn;
    if (a.tile == 64) {
        const bool spread = a.k % 2048 != 0;
        const long rows_from = a.k <= 512 ? 0 : a.k <= 1024 ? 6 : wide >= 448 ? 40 : 50;
        if (wide >= (a.k <= 1024 ? 448 : 384) && (spread || a.k <= 1024) && a.m >= rows_from * experts) return grouped_go<128, 64, 2, 2, 2>(a, s);
        const long all = (long)experts * ((a.n + 63) / 64);
        return all > 256 && all <= 512 && spread ? grouped_go<64, 64, 2, 2, 3>(a, s) : grouped_go<64, 64, 2, 2, 4>(a, s);
    }
    if (a.tile != 128) return hipErrorInvalidValue;
    // (above 104 rows per expert some have a second tile)
    const long likely = wide + (a.m > 104l * experts ? wide / 14 : 0);
    const bool eight = a.max_tiles * tn <= 256 || (a.m <= 112l * experts && (likely <= 256 || (likely > 512 && likely <= 768 && a.k >= 1536)));
    return eight ? grouped_go<128, 128, 2, 4, 4>(a, s) : grouped_go<128, 128, 2, 2, 2>(a, s);
}

template <int TN, int TM, int WN, int WM, int ST, bool MUL = false>
static hipError_t gemm_go(const GemmArgsD &a, hipStream_t s) {
    const int tn = (a.n + TN - 1) / TN, tm = (a.m + TM - 1) / TM, swz = (tn * tm) % 8 == 0 ? 1 : 0;
    constexpr size_t lds = (size_t)ST * (TN + TM) * 128;
    auto fn = MUL       ? k_dense_gemm<TN, TM, WN, WM, ST, false, false, false, MUL>
              : a.gated ? k_dense_gemm<TN, TM, WN, WM, ST, false, false, true>
              : a.c_f32 ? k_dense_gemm<TN, TM, WN, WM, ST, true>
                        : k_dense_gemm<TN, TM, WN, WM, ST, false>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    g_last_dense_tile = {TN, TM, WN * WM, 1};
    hipLaunchKernelGGL(fn, dim3(tn * tm, a.batch), dim3(64 * WN * WM), lds, s, a, tn, tm, swz);
    return hipGetLastError();
}

// ---- few rows ---------------------------------------------------------------------------------------------------------
// The same product where its tiles of 64 x 64 would leave most of the chip idle, or wait for K steps one by one (a step of such a tile takes 0.3 to
// 0.4 us whatever is in flight: DMA, barrier, LDS reads and MFMAs of one workgroup follow one another).  A workgroup makes 16 FN columns of 16 FM rows;
// its eight waves share the K columns out, 64 at a time in turn, each with its own buffers (R) and no barrier, and add up in LDS at the end.
// Measured, us per launch, weights from HBM (this / 64 x 64 tiles): 16 x 2560 x 2560 7.3 / 13.2, 16 x 2560 x 6912 12.7 / 28.8, 61 x 2560 x 6912 19.4 / 34.1,
// 61 x 6912 x 2560 14.8 / 17.3, 128 x 1536 x 4096 12.2 / 20.6, 1024 x 72 x 2560 7.1 / 13.4.
template <int FN, int FM, int R, bool TALL>
__global__ __launch_bounds__(512, 2) void k_dense_gemm_few(GemmArgsD p, int tiles_n, int tiles_m) {
    extern __shared__ __attribute__((aligned(16))) f32x4 part[];  // [wave][fragment][lane]
    constexpr int NW = 8;
    const int units = p.k >> 6;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // each XCD a contiguous run of tiles: the row tiles of one weight tile side by side, or (TALL) the column tiles of one row tile
    const int total = tiles_n * tiles_m, per = (total + 7) >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || id >= total) return;
    const int tn = TALL ? id % tiles_n : id / tiles_m, tm = TALL ? id / tiles_n : id % tiles_m;
    const int m0 = tm * 16 * FM, n0 = tn * 16 * FN;
    const int r16 = lane & 15, g = lane >> 4;
    constexpr unsigned ROWS = 16 * (FM + FN), BUF = ROWS * 128;
    const uint16_t *A = (const uint16_t *)p.a + (size_t)blockIdx.y * p.a_batch + (size_t)m0 * p.lda;
    const uint16_t *W = p.w + (size_t)blockIdx.y * p.w_batch + (size_t)n0 * p.ldw;
    const int rows_m = min(16 * FM, p.m - m0), rows_n = min(16 * FN, p.n - n0);
    unsigned oa[2 * FM], ow[2 * FN];  // (lane offsets from the tile's first row, eight rows per instruction; rows past the end read the tile's own again)
#pragma unroll
    for (int i = 0; i < 2 * FM; ++i) {
        const int r = i * 8 + (lane >> 3);
        oa[i] = (unsigned)(min(r, rows_m - 1) * p.lda + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2;
    }
#pragma unroll
    for (int i = 0; i < 2 * FN; ++i) {
        const int r = i * 8 + (lane >> 3);
        ow[i] = (unsigned)(min(r, rows_n - 1) * p.ldw + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2;
    }
    uint8_t *mine = (uint8_t *)part + wave * R * BUF;
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mine;
    auto stage = [&](int u, int slot) {
        const int k = min(u, units - 1) * 64;
#pragma unroll
        for (int i = 0; i < 2 * FN; ++i) dma1k(ow[i], W + k, base + slot * BUF + i * 1024);
#pragma unroll
        for (int i = 0; i < 2 * FM; ++i) dma1k(oa[i], A + k, base + slot * BUF + (2 * FN + i) * 1024);
    };
    f32x4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < R; ++r) stage(wave + NW * r, r);
    const int sw = (r16 >> 1) & 7;
    for (int u = wave; u < units; u += NW * R) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * 2 * (FM + FN)) : "memory");
            const uint8_t *lw = mine + r * BUF, *la = lw + FN * 2048;
            bf16x8 fa[2][FM], fw[2][FN];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int q = ((h * 4 + g) ^ sw) * 16;
#pragma unroll
                for (int i = 0; i < FN; ++i) fw[h][i] = *reinterpret_cast<const bf16x8 *>(lw + (i * 16 + r16) * 128 + q);
#pragma unroll
                for (int j = 0; j < FM; ++j) fa[h][j] = *reinterpret_cast<const bf16x8 *>(la + (j * 16 + r16) * 128 + q);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            stage(u + NW * (r + R), r);
            if (u + NW * r < units) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < FN; ++i)
#pragma unroll
                        for (int j = 0; j < FM; ++j) acc[i][j] = mfma_bf16(fw[h][i], fa[h][j], acc[i][j]);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) part[(wave * FN * FM + i * FM + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    const bool vec = (p.ldc & 3) == 0 && (p.c_batch & 3) == 0 && ((uintptr_t)p.c & 15) == 0;
    for (int f = wave; f < FN * FM; f += NW) {
        f32x4 v = part[f * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += part[(w * FN * FM + f) * 64 + lane];
        const int n = n0 + f / FM * 16 + g * 4, m = m0 + f % FM * 16 + r16;
        if (m >= p.m) continue;
        const size_t row = (size_t)blockIdx.y * p.c_batch + (size_t)m * p.ldc;
        if (p.bias)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += p.bias[min(n + e, p.n - 1)];
        if (p.gated) {
            float r[2];
#pragma unroll
            for (int e = 0; e < 4; e += 2) r[e / 2] = activate_pair(v[e], p.act0) * v[e + 1];
            uint16_t *dst = (uint16_t *)p.c + row + n / 2;
            if (vec && n + 3 < p.n) {
                *reinterpret_cast<uint32_t *>(dst) = (uint32_t)f2bf(r[0]) | (uint32_t)f2bf(r[1]) << 16;
            } else {
                if (n < p.n) dst[0] = f2bf(r[0]);
                if (n + 2 < p.n) dst[1] = f2bf(r[1]);
            }
            continue;
        }
        if (p.act_split < p.n) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = activate_column(v[e], n + e < p.act_split ? p.act0 : p.act1, false, p.more);
        } else if (p.act0 != BITNET_HIP_ACT_NONE) {
            const bool fast_gelu = gelu_is_fast(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = activate_column(v[e], p.act0, fast_gelu, p.more);
        }
        if (p.more.mul) {
            const int token = min(max(p.more.mul_tokens[*p.more.mul_at + m], 0), p.more.mul_rows - 1);
            const uint16_t *mul = p.more.mul + (size_t)token * p.more.ld_mul;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= bf2f(mul[min(n + e, p.n - 1)]);
        }
        if (p.c_f32) {
            float *dst = (float *)p.c + row + n;
            if (vec && n + 3 < p.n) {
                *reinterpret_cast<f32x4 *>(dst) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < p.n) dst[e] = v[e];
            }
        } else {
            uint16_t *dst = (uint16_t *)p.c + row + n;
            if (vec && n + 3 < p.n) {
                *reinterpret_cast<bf16x4 *>(dst) = bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < p.n) dst[e] = f2bf(v[e]);
            }
        }
    }
}

template <int FN, int FM, int R>
static hipError_t gemm_few_go(const GemmArgsD &a, hipStream_t s) {
    const int tn = (a.n + 16 * FN - 1) / (16 * FN), tm = (a.m + 16 * FM - 1) / (16 * FM);
    constexpr size_t lds = 8 * 1024 * (FN * FM > 2 * R * (FN + FM) ? FN * FM : 2 * R * (FN + FM));
    // Activations that outgrow an XCD's L2 (4 MB) are read once, not once per column of tiles, where they are the larger operand.  us with this order / the other:
    // 2048 x 256 x 6912 18.9 / 35.2, 2685 x 160 x 4096 12.6 / 21.7, 1531 x 320 x 2560 10.4 / 14.6, 605 x 320 x 8192 15.4 / 19.5.
    const bool tall = (size_t)a.m * a.k * 2 > 4u << 20 && (size_t)a.m * 4 > (size_t)a.n * 5;
    auto fn = tall ? k_dense_gemm_few<FN, FM, R, true> : k_dense_gemm_few<FN, FM, R, false>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    g_last_dense_tile = {16 * FN, 16 * FM, 8, 8};
    hipLaunchKernelGGL(fn, dim3((tn * tm + 7) / 8 * 8, a.batch), dim3(512), lds, s, a, tn, tm);
    return hipGetLastError();
}

// f32 activations: f32 multiply-adds on a 64 x 64 tile, 4 x 4 per thread
template <bool GROUPED>
__global__ __launch_bounds__(256) void k_dense_gemm_f32(GemmArgsD p) {
    __shared__ float sa[16][68], sw[16][68];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    int m0 = blockIdx.y * 64, m_end = p.m;
    const int n0 = blockIdx.x * 64;
    const float *A = (const float *)p.a + (size_t)blockIdx.z * p.a_batch;
    const uint16_t *W = p.w + (size_t)blockIdx.z * p.w_batch;
    if (GROUPED) {
        if ((int)blockIdx.y >= *p.n_tiles) return;
        const int4 tile = p.tiles[blockIdx.y];
        m0 = tile.y, m_end = tile.y + tile.z;
        W += (size_t)tile.x * p.w_batch;
    }
    float acc[4][4] = {};
    const int lr = tid >> 2, lk = (tid & 3) * 4;
    int ar = m0 + lr < m_end ? m0 + lr : m_end - 1;
    if (GROUPED && p.gather) ar = p.gather[ar];
    const int wr = n0 + lr < p.n ? n0 + lr : p.n - 1;
    for (int k0 = 0; k0 < p.k; k0 += 16) {
        const f32x4 av = *reinterpret_cast<const f32x4 *>(A + (size_t)ar * p.lda + k0 + lk);
        const u32x2 wv = *reinterpret_cast<const u32x2 *>(W + (size_t)wr * p.ldw + k0 + lk);
        __syncthreads();
        sa[lk][lr] = av.x, sa[lk + 1][lr] = av.y, sa[lk + 2][lr] = av.z, sa[lk + 3][lr] = av.w;
        sw[lk][lr] = bf2f(wv.x & 0xffffu), sw[lk + 1][lr] = bf2f(wv.x >> 16), sw[lk + 2][lr] = bf2f(wv.y & 0xffffu), sw[lk + 3][lr] = bf2f(wv.y >> 16);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            float x[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = sa[k][ty * 4 + i], w[i] = sw[k][tx * 4 + i];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(x[i], w[j], acc[i][j]);
        }
    }
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= m_end) break;
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= p.n) break;
            if (p.gated && (j & 1)) continue;
            float v = activate(acc[i][j] + (p.bias ? p.bias[n] : 0.f), n < p.act_split ? p.act0 : p.act1, p.more.act_a, p.more.act_b);
            if (p.more.mul) v *= bf2f(p.more.mul[(size_t)min(max(p.more.mul_tokens[*p.more.mul_at + m], 0), p.more.mul_rows - 1) * p.more.ld_mul + n]);
            size_t o = (size_t)blockIdx.z * p.c_batch + (size_t)m * p.ldc + n;
            if (p.gated) {  // (n is even here, and so is the number of columns)
                v *= acc[i][j < 3 ? j + 1 : 3] + (p.bias ? p.bias[n + 1] : 0.f);
                o -= n / 2;
            }
            if (p.c_f32)
                ((float *)p.c)[o] = v;
            else
                ((uint16_t *)p.c)[o] = f2bf(v);
        }
    }
}

hipError_t launch_dense_gemm(const GemmArgsD &args, hipStream_t s) {
    GemmArgsD a = args;
    if (a.m <= 0 || a.n <= 0) return hipSuccess;
    if (a.act_split == 0) a.act_split = a.n;
    if (a.gated && !a.a_f32 && a.c_f32) return hipErrorInvalidValue;
    if (a.tiles) {
        if (a.a_f32) {
            if (a.tile != 64) return hipErrorInvalidValue;
            g_last_dense_tile = {64, 64, 4, 1};
            hipLaunchKernelGGL(k_dense_gemm_f32<true>, dim3((a.n + 63) / 64, a.max_tiles, 1), dim3(256), 0, s, a);
            return hipGetLastError();
        }
        if (a.c_f32) return hipErrorInvalidValue;
        return launch_grouped(a, s);
    }
    if (a.a_f32) {
        g_last_dense_tile = {64, 64, 4, 1};
        hipLaunchKernelGGL(k_dense_gemm_f32<false>, dim3((a.n + 63) / 64, (a.m + 63) / 64, a.batch), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    if (a.more.mul && (a.c_f32 || a.gated)) return hipErrorInvalidValue;
    // one round of workgroups of the form for few rows, its smallest tile first (two per CU fit but share the CU's LDS-DMA: behind 256 the larger tile is ahead, and behind
    // that the tiles of 64 x 64: 61 x 10240 x 2560 takes 20.3 to 25.5 us in this form and 18.3 in the other); short K leaves its waves without work (256: 5.2 / 4.3 us), and
    // those of the largest tile below 1536 (36 x 8192 x 512 7.0 / 6.2, 145 x 2560 x 512 6.5 / 6.2, 52 x 8192 x 1024 8.4 / 8.0; 40 x 4608 x 1536 8.7 / 9.3) unless tiles of 64
    // columns are a quarter wider than the matrix needs (3500 x 72 x 512 6.3 / 8.0)
    auto one_round = [&](int tn, int tm) { return ((long)(a.n + tn - 1) / tn) * ((a.m + tm - 1) / tm) * a.batch <= 256; };
    if (a.k >= 512) {
        if (one_round(16, 16)) return gemm_few_go<1, 1, 2>(a, s);
        if (one_round(32, 32)) return gemm_few_go<2, 2, 1>(a, s);
        if (one_round(32, 64) && (a.k >= 1536 || ((long)a.n + 63) / 64 * 8 >= ((long)a.n + 31) / 32 * 5)) return gemm_few_go<2, 4, 1>(a, s);
    }
    if (a.more.mul) return gemm_go<64, 64, 2, 2, 4, true>(a, s);
    auto tiles = [&](int tn, int tm) { return (double)((a.n + tn - 1) / tn) * ((a.m + tm - 1) / tm) * a.batch; };
    if (a.k <= 1024 && tiles(64, 64) >= 1024) return gemm_go<64, 64, 2, 2, 2>(a, s);  // few steps: what counts is how many workgroups overlap their ends
    // The tile whose launch is the shortest by what was measured (us; every tile at 330 shapes, m 24 to 4100, n 320 to 13824, k 512 to 8192, each kind of output; the choice is 1.4 % behind
    // the best of them in the mean): a step of 64 columns and a round's start and end.  The large ones stand alone on their CU and run in rounds of 256.  Of 128 x 128 in four
    // waves two fit, which overlap their ends: ahead of the others where those fill their last round badly (565 x 12288 x 3072 52 us, 128 x 128 in eight waves 59;
    // 3667 x 2112 x 1024 23 / 28).  Of 64 x 128 two fit as well, but a second one costs more than half a round; a CU takes up to four of 64 x 64.  Three buffers where LDS has the
    // room: 128 x 256 takes 0.80 us a step with them and 0.96 with two.  4096 x 3072 x 3072: 256 x 256 leaves a quarter of the CUs out (76 us), 192 x 256 is one full round (69);
    // 2048 x 2560 x 6912: 128 x 192 80 us, 128 x 128 in four waves 114.
    // What is stored one by one: every tile's outputs, 25 us per 65536 of them, where rows do not start on sixteen bytes (4096 x 13824 x 2560: 256 x 256 412 us, 128 x 256 476,
    // 64 x 128 513), else those of the last column of tiles where it sticks out, which lengthen the launch by 25 us (256 x 256), 14, 6, 3.5 (128 x 192) or 1.6
    // (2297 x 4096 x 1536: 192 x 256 52 us, 128 x 192 42).
    const double steps = a.k / 64, slow = a.gated ? 12.5 / 65536 : 25.0 / 65536;
    const bool aligned = rows_on_16_bytes(a.c, a.ldc, a.c_batch, a.c_f32);
    auto stores = [&](int tn, int tm, double rounds) { return aligned ? (a.n % tn && !a.gated ? 25.0 / 65536 / 65536 * tn * tm * tn * tm : 0.0) : slow * tn * tm * std::max(rounds, 1.0); };
    auto alone = [&](int tn, int tm, double step, double ends) {
        const double rounds = std::ceil(tiles(tn, tm) / 256);
        return rounds * (steps * step + ends) + stores(tn, tm, rounds);
    };
    const double t64 = tiles(64, 64) / 256, t128 = tiles(64, 128) / 256, pairs = tiles(128, 128) / 512, whole = std::floor(pairs), rest = pairs - whole;
    const double us[] = {alone(256, 256, 1.27, 13), alone(192, 256, 1.06, 11), alone(128, 256, 0.80, 6), alone(128, 192, 0.68, 4.5), alone(128, 128, 0.48, 5.5),
                         whole * (0.88 * steps + 6) + (rest == 0 ? 0 : rest <= 0.5 ? 0.62 * steps + 6 : 0.88 * steps + 6) + stores(128, 128, 2 * pairs),
                         steps * (t128 <= 1 ? 0.40 : 0.62 * std::ceil(t128 / 2)) + 3.5 + stores(64, 128, t128), steps * 0.27 * std::max(t64, 1.0) + 3 + stores(64, 64, t64)};
    switch (std::min_element(std::begin(us), std::end(us)) - us) {
        case 0: return gemm_go<256, 256, 2, 4, 2>(a, s);
        case 1: return gemm_go<192, 256, 2, 4, 2>(a, s);
        case 2: return gemm_go<128, 256, 2, 4, 3>(a, s);
        case 3: return gemm_go<128, 192, 2, 4, 3>(a, s);
        case 4: return gemm_go<128, 128, 2, 4, 4>(a, s);
        case 5: return gemm_go<128, 128, 2, 2, 2>(a, s);
        case 6: return gemm_go<64, 128, 2, 2, 3>(a, s);
        default: return gemm_go<64, 64, 2, 2, 4>(a, s);
    }
}

}  // namespace bitnet_hip
