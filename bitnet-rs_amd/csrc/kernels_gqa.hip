// kernels_gqa.hip -- causal attention whose query heads share keys and values in groups, with one softmax map per head or two (gfx950).
// Optionally rotated queries and keys, chunks of positions that do not see each other, a window, a penalty that grows with the distance, a sink in the
// softmax's denominator, keys that are the values too, short convolutions ahead of it all, and a gate per head or column on the output.
//
// Two maps (differential attention) weigh the same values; a head's output is a1 - lambda a2, divided by its root mean square over the value
// columns.  Caches: keys [kv head][map][capacity][dimp], values transposed [kv head][vdimp][capacity].
//   k_gqa_rows     rows of projections: convolution, query and key norms, the query's factor at its position, keys and values into the caches
//   k_gqa_prefill  a prompt's portion: flash attention on S^T = K Q^T and O^T = V^T P^T, both maps of a query tile in one wave
//   k_gqa_step     the decode step: norms and append in the same launch, 32 keys per wave and step on the matrix cores
//   k_gqa_any      any size, f32 or bf16 cache, one wave per key
//   k_gqa_merge    records of the decode forms -> output
// Scores, maxima, sums and weights are f32; a weight (and the decode step's query) enters the matrix cores as a (high, low) pair of bf16 values.
// Scores are kept in base 2: the score times log2(e).
#include <algorithm>
#include <type_traits>

#include "dense.hpp"

namespace bitnet_hip {

constexpr float kLog2e = 1.44269504088896f;

// the first key a query at this position sees
__host__ __device__ __forceinline__ int gqa_first(const Gqa &p, int pos) {
    const int first = p.chunk ? pos - (int)((unsigned)pos % (unsigned)p.chunk) : 0;
    return p.window && pos - (int)p.window + 1 > first ? pos - (int)p.window + 1 : first;
}

// The records of a query at `pos`: tiles of keys from `base` (the tile that holds its first key) on, `per` tiles each.
struct GqaRange {
    int first, base, per, used;
};
__device__ __forceinline__ GqaRange gqa_range(const Gqa &p, int pos) {
    GqaRange r;
    r.first = gqa_first(p, pos);
    r.base = r.first & ~(kGqaTile - 1);
    const int tiles = (pos + 1 - r.base + kGqaTile - 1) / kGqaTile;
    r.per = (tiles + kGqaSplits - 1) / kGqaSplits;
    r.used = (tiles + r.per - 1) / r.per;
    return r;
}
// records a launch has to provide for
static int gqa_records(const Gqa &g) {
    size_t keys = g.capacity;
    if (g.chunk && g.chunk + kGqaTile < keys) keys = g.chunk + kGqaTile;  // (a chunk may start inside a tile)
    if (g.window && g.window + kGqaTile < keys) keys = g.window + kGqaTile;
    return (int)min((size_t)kGqaSplits, (keys + kGqaTile - 1) / kGqaTile);
}

// element i of a head at a position, v being its own and the lane's neighbour holding the other element of the pair; cs, sn: the tables' row
__device__ __forceinline__ float turn_neighbours(float v, int i, const float *cs, const float *sn, int dims) {
    const float o = dpp<0xb1>(v);  // quad_perm [1,0,3,2]
    if (i >= dims) return v;
    const float c = cs[i >> 1], s = sn[i >> 1];
    return (i & 1) ? v * c + o * s : v * c - o * s;
}
// what a head's gate (or that of a column of it) is the sigmoid of
__device__ __forceinline__ float gate_logit(const Gqa &p, int row, int h, int column) {
    const size_t i = (size_t)row * p.ldgate + (p.gate_columns ? (size_t)h * p.vdimp + column : (size_t)h);
    return p.gate_f32 ? ((const float *)p.gate)[i] : bf2f(((const uint16_t *)p.gate)[i]);
}
// a head's distance penalty: what is taken off the natural score is weight * log2(1 + rate * distance)
struct FarPenalty {
    float weight, rate;
};
__device__ __forceinline__ FarPenalty far_penalty(const Gqa &p, int h) {
    FarPenalty f{0.f, 0.f};
    if (p.far_weight) f.weight = p.far_weight[h] * 0.69314718055994531f, f.rate = p.far_rate[h];
    return f;
}
__device__ __forceinline__ float nearer(float score, const FarPenalty &f, int distance) { return fmaf(-f.weight, __log2f(fmaf(f.rate, (float)distance, 1.0f)), score); }
// columns of a row of projections that a convolution covers
__host__ __device__ __forceinline__ int gqa_channels(const Gqa &p) {
    if (p.queries_only) return (int)(p.heads * p.maps * p.dimp);
    return (int)((p.heads + p.kv_heads) * p.maps * p.dimp + (p.values_are_keys ? 0 : p.kv_heads * p.vdimp));
}
// column c of the row of projections t (negative: an earlier portion's; zero ahead of the sequence)
template <class TR>
__device__ __forceinline__ float raw_value(const Gqa &p, const TR *rows, size_t ld, int pos0, int t, int c, int channels) {
    if (t >= 0) return ld_act(rows + (size_t)t * ld, c);
    const int at = pos0 + t;
    return at >= 0 ? p.ring[(size_t)(at % (int)p.taps) * channels + c] : 0.f;
}

size_t gqa_scratch_floats(size_t heads, size_t maps, size_t vdimp, size_t nq) { return nq * heads * maps * kGqaSplits * (kGqaRecHead + vdimp); }
bool gqa_supported(int dimp, int vdimp) { return dimp <= 256 && vdimp <= 256; }

// ---- rows of projections ----------------------------------------------------------------------------------------------
// blockIdx.y: query heads x maps, key heads x maps (sixteen tokens per workgroup, four per wave), then value heads in groups of 32 columns (64
// tokens, every fourth workgroup).
constexpr int kRowTokens = 16, kRowCols = 32;

// Four tokens of a query or key head of up to 128 NJ columns: a lane holds neighbouring elements, so that a pair turns within it.  TAPS: those of the convolution
// (0: none, -1: any number).
template <class TR, class TC, int NJ, int TAPS>
__device__ __forceinline__ void head_rows(const Gqa &p, const TR *rows, size_t ld, int pos0, int t0, int n, int y, bool key, TC *cache, TR *queries, size_t ldq) {
    constexpr int U = kRowTokens / 4;
    constexpr bool CONV = TAPS != 0;
    const int lane = threadIdx.x & 63, dim = (int)p.dim, dimp = (int)p.dimp, turned = (int)p.rot_dims, half = turned >> 1;
    const float *w = key ? p.k_weight : p.q_weight;
    float v[U][NJ][2], cs[U][NJ], sn[U][NJ], factor[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = min(t0 + u, n - 1);
        const TR *row = rows + (size_t)t * ld + (size_t)y * dimp;
        factor[u] = key ? 1.0f : p.q_factor[pos0 + t];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int i = min(2 * lane + 128 * j, dimp - 2);
            if (CONV)
                v[u][j][0] = v[u][j][1] = 0.f;
            else
                v[u][j][0] = ld_act(row, i), v[u][j][1] = ld_act(row, i + 1);
            cs[u][j] = 1.0f, sn[u][j] = 0.f;
            if (turned && 2 * lane + 128 * j < turned) {
                const size_t at = (size_t)(pos0 + t) * half + lane + 64 * j;
                cs[u][j] = p.rope_cos[at], sn[u][j] = p.rope_sin[at];
            }
        }
    }
    if (TAPS > 0) {  // the tokens and those ahead of them once, in registers
        constexpr int T = TAPS > 0 ? TAPS : 1;
        const int channels = gqa_channels(p);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int c = y * dimp + min(2 * lane + 128 * j, dimp - 2);
            float f[T][2], raw[U + T - 1][2];
#pragma unroll
            for (int k = 0; k < T; ++k) f[k][0] = p.conv[(size_t)k * channels + c], f[k][1] = p.conv[(size_t)k * channels + c + 1];
            if (t0 >= T - 1) {
#pragma unroll
                for (int k = 0; k < U + T - 1; ++k) {
                    const TR *row = rows + (size_t)min(t0 - (T - 1) + k, n - 1) * ld;
                    raw[k][0] = ld_act(row, c), raw[k][1] = ld_act(row, c + 1);
                }
            } else {
#pragma unroll
                for (int k = 0; k < U + T - 1; ++k) {
                    const int t = min(t0 - (T - 1) + k, n - 1);
                    raw[k][0] = raw_value(p, rows, ld, pos0, t, c, channels), raw[k][1] = raw_value(p, rows, ld, pos0, t, c + 1, channels);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int k = 0; k < T; ++k) v[u][j][0] += f[k][0] * raw[u + k][0], v[u][j][1] += f[k][1] * raw[u + k][1];
        }
    } else if (CONV) {
        const int taps = (int)p.taps, channels = gqa_channels(p);
        for (int k = 0; k < taps; ++k)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int c = y * dimp + min(2 * lane + 128 * j, dimp - 2);
                const float f0 = p.conv[(size_t)k * channels + c], f1 = p.conv[(size_t)k * channels + c + 1];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int t = min(t0 + u, n - 1) - (taps - 1) + k;
                    v[u][j][0] += f0 * raw_value(p, rows, ld, pos0, t, c, channels), v[u][j][1] += f1 * raw_value(p, rows, ld, pos0, t, c + 1, channels);
                }
            }
    }
    float wv[NJ][2];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e) wv[j][e] = w && 2 * lane + 128 * j + e < dim ? w[2 * lane + 128 * j + e] : 1.0f;  // (padding columns hold zeros)
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (w || p.unit_norm) {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < NJ; ++j) ss += 2 * lane + 128 * j < dimp ? v[u][j][0] * v[u][j][0] + v[u][j][1] * v[u][j][1] : 0.f;
            factor[u] *= 1.0f / sqrtf(wave_sum(ss) / (float)dim + p.eps);
        }
        if (t0 + u >= n) continue;
        TR *row = queries + (size_t)(t0 + u) * ldq + (size_t)y * dimp;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int i = 2 * lane + 128 * j;
            if (i >= dimp) continue;
            const float a = v[u][j][0] * factor[u] * wv[j][0], b = v[u][j][1] * factor[u] * wv[j][1];
            const float x = a * cs[u][j] - b * sn[u][j], z = b * cs[u][j] + a * sn[u][j];
            if (key) {
                TC *dst = cache + (size_t)(pos0 + t0 + u) * dimp;
                st_act(dst, i, x), st_act(dst, i + 1, z);
            } else {
                st_act(row, i, x), st_act(row, i + 1, z);
            }
        }
    }
}

// TAPS (as head_rows): every column passes a convolution over time first, and the queries go to a place of their own
template <class TR, class TC, int NJ, int TAPS>
__global__ __launch_bounds__(256) void k_gqa_rows(Gqa p, const TR *rows, size_t ld, const int *pos_ptr, int n, TR *queries, size_t ldq) {
    constexpr int STRIDE = sizeof(TR) == 4 ? kRowCols + 1 : kRowCols + 2;
    constexpr bool CONV = TAPS != 0;
    __shared__ __attribute__((aligned(16))) TR tile[(64 + (TAPS < 0 ? kMaxTaps - 1 : TAPS > 0 ? TAPS - 1 : 0)) * STRIDE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, pos0 = *pos_ptr;
    const int nq = (int)(p.heads * p.maps), nk = (int)(p.kv_heads * p.maps), dim = (int)p.dim, dimp = (int)p.dimp, vdimp = (int)p.vdimp;
    int y = blockIdx.y;
    if (y < nq + nk) {
        const bool key = y >= nq;
        const float *w = key ? p.k_weight : p.q_weight;
        const int turned = (int)p.rot_dims, half = turned >> 1, t0 = blockIdx.x * kRowTokens + wave * (kRowTokens / 4);
        TC *cache = key ? (TC *)p.kcache + (size_t)(y - nq) * p.capacity * dimp : nullptr;
        if (t0 >= n) return;
        if (dimp <= 128 * NJ) {
            head_rows<TR, TC, NJ, TAPS>(p, rows, ld, pos0, t0, n, y, key, cache, queries, ldq);
            return;
        }
        const int channels = gqa_channels(p), taps = (int)p.taps;
        for (int t = t0; t < min(t0 + kRowTokens / 4, n); ++t) {
            TR *row = queries + (size_t)t * ldq + (size_t)y * dimp;
            auto value = [&](int i) {
                if (!CONV) return ld_act(rows + (size_t)t * ld + (size_t)y * dimp, i);
                float v = 0.f;
                for (int k = 0; k < taps; ++k) v += p.conv[(size_t)k * channels + y * dimp + i] * raw_value(p, rows, ld, pos0, t - (taps - 1) + k, y * dimp + i, channels);
                return v;
            };
            float ss = 0.f;
            if (w || p.unit_norm)
                for (int i = lane; i < dimp; i += 64) {
                    const float v = value(i);
                    ss += v * v;
                }
            const float norm = w || p.unit_norm ? 1.0f / sqrtf(wave_sum(ss) / (float)dim + p.eps) : 1.0f;
            const float factor = key ? norm : norm * p.q_factor[pos0 + t];
            const float *cs = p.rope_cos + (size_t)(pos0 + t) * half, *sn = p.rope_sin + (size_t)(pos0 + t) * half;
            for (int i = lane; i < dimp; i += 64) {
                float v = value(i) * factor * (w && i < dim ? w[i] : 1.0f);
                if (turned) v = turn_neighbours(v, i, cs, sn, turned);
                if (key)
                    st_act(cache + (size_t)(pos0 + t) * dimp, i, v);
                else
                    st_act(row, i, v);
            }
        }
        return;
    }
    if (blockIdx.x % (64 / kRowTokens)) return;
    y -= nq + nk;
    const int t0 = blockIdx.x * kRowTokens, groups = vdimp / kRowCols, head = y / groups, c0 = (y - head * groups) * kRowCols, count = min(64, n - t0);
    const int column = (p.values_are_keys ? nq : nq + nk) * dimp + head * vdimp + c0;
    const TR *src = rows + column;
    constexpr int V = 16 / sizeof(TR), PER = kRowCols / V;
    const int taps = TAPS > 0 ? TAPS : CONV ? (int)p.taps : 1, channels = gqa_channels(p);
    if (CONV) {  // the tokens ahead of the first one in the tile's last rows
        for (int i = tid; i < (taps - 1) * kRowCols; i += 256) {
            const int k = i / kRowCols, c = i % kRowCols;
            st_act(tile, (64 + k) * STRIDE + c, raw_value(p, rows, ld, pos0, t0 - (taps - 1) + k, column + c, channels));
        }
    }
#pragma unroll
    for (int j = 0; j < 64 * PER / 256; ++j) {
        const int i = tid + 256 * j, t = i / PER, c = i % PER * V;
        if (t < count) {
            const u32x4 x = *reinterpret_cast<const u32x4 *>(src + (size_t)(t0 + t) * ld + c);
            uint32_t *dst = reinterpret_cast<uint32_t *>(tile + t * STRIDE + c);
            dst[0] = x.x, dst[1] = x.y, dst[2] = x.z, dst[3] = x.w;
        }
    }
    __syncthreads();
    TC *cache = (TC *)p.vcache + ((size_t)head * vdimp + c0) * p.capacity + pos0 + t0;
    if (lane < count)
#pragma unroll
        for (int j = 0; j < kRowCols / 4; ++j) {
            const int v = wave * (kRowCols / 4) + j;
            float x;
            if (CONV) {
                x = 0.f;
#pragma unroll TAPS > 0 ? TAPS : 1
                for (int k = 0; k < taps; ++k) {
                    const int t = lane - (taps - 1) + k;
                    x += p.conv[(size_t)k * channels + column + v] * ld_act(tile, (t >= 0 ? t : 64 + taps - 1 + t) * STRIDE + v);
                }
            } else {
                x = ld_act(tile, lane * STRIDE + v);
            }
            st_act(cache + (size_t)v * p.capacity, lane, x);
        }
}

template <class TR, class TC>
static hipError_t rows_go(const Gqa &g, const void *rows, size_t ld, const int *pos, int n, void *q, size_t ldq, hipStream_t s) {
    const int keys = g.queries_only ? 0 : (int)(g.kv_heads * g.maps + g.kv_heads * (g.vdimp / kRowCols));
    const dim3 grid((n + kRowTokens - 1) / kRowTokens, (int)(g.heads * g.maps) + keys);
    auto pick = [&](auto narrow, auto wide) { return g.dimp <= 128 ? narrow : wide; };
    auto fn = g.taps == 0   ? pick(k_gqa_rows<TR, TC, 1, 0>, k_gqa_rows<TR, TC, 2, 0>)
              : g.taps == 2 ? pick(k_gqa_rows<TR, TC, 1, 2>, k_gqa_rows<TR, TC, 2, 2>)
              : g.taps == 3 ? pick(k_gqa_rows<TR, TC, 1, 3>, k_gqa_rows<TR, TC, 2, 3>)
              : g.taps == 4 ? pick(k_gqa_rows<TR, TC, 1, 4>, k_gqa_rows<TR, TC, 2, 4>)
                            : pick(k_gqa_rows<TR, TC, 1, -1>, k_gqa_rows<TR, TC, 2, -1>);
    hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, g, (const TR *)rows, ld, pos, n, (TR *)q, ldq);
    return hipGetLastError();
}

hipError_t launch_gqa_rows(const Gqa &g, void *rows, size_t ld, int rows_f32, int cache_f32, const int *pos, int n, void *q, size_t ldq, hipStream_t s) {
    if (rows_f32) return cache_f32 ? rows_go<float, float>(g, rows, ld, pos, n, q, ldq, s) : rows_go<float, uint16_t>(g, rows, ld, pos, n, q, ldq, s);
    return cache_f32 ? hipErrorInvalidValue : rows_go<uint16_t, uint16_t>(g, rows, ld, pos, n, q, ldq, s);
}

// ---- any size ---------------------------------------------------------------------------------------------------------
// One workgroup per (record, head and map, query); a wave takes every fourth key, its lanes the columns.
template <class TQ, class TC, int ND, int NV>
__global__ __launch_bounds__(256) void k_gqa_any(Gqa p, const TQ *q, size_t ldq, const int *pos_ptr, int q0, int nq, float *scratch) {
    extern __shared__ __attribute__((aligned(16))) float vec[];  // [4][vdimp]
    __shared__ float sm[4], sl[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const RecordPlace at = record_place();
    const int maps = (int)p.maps, each = (int)p.heads * maps, qi = at.member / each, hm = at.member - qi * each, h = hm / maps, map = hm - h * maps, kv = h / (int)(p.heads / p.kv_heads), dimp = (int)p.dimp, vdimp = (int)p.vdimp;
    if (qi >= nq) return;
    const int pos = *pos_ptr + q0 + qi;
    const GqaRange range = gqa_range(p, pos);
    if (at.record >= range.used) return;
    const int start = range.base + at.record * range.per * kGqaTile, k0 = max(start, range.first), k1 = min(start + range.per * kGqaTile, pos + 1);
    const TQ *qr = q + (size_t)qi * ldq + (size_t)hm * dimp;
    const TC *K = (const TC *)p.kcache + (size_t)(kv * maps + map) * p.capacity * dimp, *V = (const TC *)p.vcache + (size_t)kv * vdimp * p.capacity;
    float qv[ND], acc[NV];
#pragma unroll
    for (int j = 0; j < ND; ++j) qv[j] = lane + 64 * j < dimp ? ld_act(qr, lane + 64 * j) : 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = 0.f;
    const FarPenalty far = far_penalty(p, h);
    float m = -INFINITY, l = 0.f;
    for (int key = k0 + wave; key < k1; key += 4) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < ND; ++j)
            if (lane + 64 * j < dimp) s += qv[j] * ld_act(K + (size_t)key * dimp, lane + 64 * j);
        s = nearer(wave_sum(s), far, pos - key) * kLog2e;
        const float mn = fmaxf(m, s), al = exp2f(m - mn), w = exp2f(s - mn);
        l = l * al + w;
        m = mn;
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (lane + 64 * j < vdimp) acc[j] = acc[j] * al + w * ld_act(V + (size_t)(lane + 64 * j) * p.capacity, key);
    }
    if (lane == 0) sm[wave] = m, sl[wave] = l;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (lane + 64 * j < vdimp) vec[wave * vdimp + lane + 64 * j] = acc[j];
    __syncthreads();
    const float M = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
    float w[4], L = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        w[i] = sm[i] == -INFINITY ? 0.f : exp2f(sm[i] - M);
        L += w[i] * sl[i];
    }
    float *rec = scratch + (((size_t)qi * p.heads * maps + hm) * kGqaSplits + at.record) * (kGqaRecHead + vdimp);
    for (int i = tid; i < vdimp; i += 256)
        rec[kGqaRecHead + i] = (w[0] * vec[i] + w[1] * vec[vdimp + i]) + (w[2] * vec[2 * vdimp + i] + w[3] * vec[3 * vdimp + i]);
    if (tid == 0) rec[0] = M, rec[1] = L;
}

template <class TQ, class TC>
static hipError_t any_go(const Gqa &g, const void *q, size_t ldq, const int *pos, int q0, int nq, float *scratch, hipStream_t s) {
    const int splits = gqa_records(g);
    const size_t lds = 4 * g.vdimp * sizeof(float);
    if (g.dimp > 1024 || g.vdimp > 1024) return hipErrorInvalidValue;
    auto fn = g.dimp <= 64 && g.vdimp <= 64 ? k_gqa_any<TQ, TC, 1, 1> : g.dimp <= 256 && g.vdimp <= 256 ? k_gqa_any<TQ, TC, 4, 4> : k_gqa_any<TQ, TC, 16, 16>;
    hipLaunchKernelGGL(fn, record_grid(splits, g.heads * g.maps * nq), dim3(256), lds, s, g, (const TQ *)q, ldq, pos, q0, nq, scratch);
    return hipGetLastError();
}

hipError_t launch_gqa_any(const Gqa &g, const void *q, size_t ldq, int q_f32, int cache_f32, const int *pos, int q0, int nq, float *scratch, hipStream_t s) {
    if (q_f32) return cache_f32 ? any_go<float, float>(g, q, ldq, pos, q0, nq, scratch, s) : any_go<float, uint16_t>(g, q, ldq, pos, q0, nq, scratch, s);
    return cache_f32 ? hipErrorInvalidValue : any_go<uint16_t, uint16_t>(g, q, ldq, pos, q0, nq, scratch, s);
}

// ---- decode step, matrix cores ----------------------------------------------------------------------------------------
// One workgroup per (record, kv head and 16 of its query heads), four waves; a wave takes every fourth block of 32 keys by itself, with maximum,
// sum and output of its own, and the four meet at the end.  S^T = K Q^T: row 4 g + e of score tile t is key 8 g + 4 t + e of the block, so that a
// lane's weights of both tiles are the eight consecutive keys 8 g .. 8 g + 7 which it needs as an operand of O^T = V^T P^T.
// Exponentials are the hardware's: exp2f scales its argument and result so that what lies under 2^-126 of the largest weight stays a number; here it is zero, which no sum that
// holds a one can tell.  12 and 24 heads of two maps of 64 / 128 columns, 200 and 1000 keys: 9.4 -> 9.1 us; one map of 128 / 128: 8.25 -> 8.05.
// The launch is a chain of latencies (150 and 2090 keys take the same): arguments -> position -> rotation and keys -> scores -> weights -> output.  Hence: what the host knows is
// divided there (64-bit divisions by arguments were a quarter of the launch), all arguments are requested at once, raw rows and norms' weights ahead of the position, and the
// new key's row is one more of the rows that the waves share out.  Records are the slowest index of the launch, which has one for every 128 keys of the capacity: as the fastest
// they put several of the workgroups that have keys on the same compute units at some capacities (24 heads of 6 kv heads at 2000 keys, us with this order / that: capacity 8192 6.0 / 8.2,
// two maps 6.9 / 9.1, capacity 8320 7.0 / 8.9, 5888 and 9600 7.0 / 7.1).  Beside another launch, 12 heads of 128 / 128 at 2090 keys 8.6 -> 6.2 us, 24 of two maps of 64 / 128 at 216 keys 12.2 -> 10.2.
struct GqaStepK {
    const float *row, *q_weight, *k_weight, *q_factor, *rope_cos, *rope_sin, *far_weight, *far_rate;
    const int *pos;
    uint16_t *K, *V;
    float *scratch, eps;
    int heads, group, dim, dimp, vdimp, capacity, turned, chunk, window, normed, append, k_at, v_at;  // normed: 1 queries, 2 keys
};

template <int NK, int NV, int MAPS>
__global__ __launch_bounds__(256, NV > 8 || NK * MAPS >= 8 ? 1 : 2) void k_gqa_step(GqaStepK p) {
    extern __shared__ __attribute__((aligned(16))) float area[];  // queries [maps][16][NK * 32]; then the waves' outputs
    __shared__ float sm[4][MAPS][16], sl[4][MAPS][16];
    __shared__ __attribute__((aligned(16))) uint16_t newk[MAPS][NK * 32], newv[NV * 16];
    // (every argument at once: read where they are used they are a chain of scalar loads)
    asm volatile("" ::"s"(p.row), "s"(p.q_weight), "s"(p.k_weight), "s"(p.q_factor), "s"(p.rope_cos), "s"(p.rope_sin), "s"(p.far_weight), "s"(p.far_rate), "s"(p.pos), "s"(p.K), "s"(p.V),
                 "s"(p.scratch), "s"(p.eps), "s"(p.heads), "s"(p.group), "s"(p.dim), "s"(p.dimp), "s"(p.vdimp), "s"(p.capacity), "s"(p.turned), "s"(p.chunk), "s"(p.window), "s"(p.normed),
                 "s"(p.append), "s"(p.k_at), "s"(p.v_at));
    const int posv = *p.pos;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int kv = blockIdx.x, first_head = blockIdx.y * 16, h0 = kv * p.group + first_head, nh = min(16, p.group - first_head);
    const int dimp = p.dimp, vdimp = p.vdimp;
    constexpr int QS = NK * 32 + 4, J = (NK + 1) / 2, QR = NK > 4 ? 1 : 4;  // QR: rows of a wave at a time
    uint16_t *K = p.K + (size_t)kv * MAPS * p.capacity * dimp, *V = p.V + (size_t)kv * vdimp * p.capacity;
    // row i of a wave: of the only map, or of its own of two
    const int map = MAPS == 2 ? wave & 1 : 0;
    auto head_of = [&](int i) { return MAPS == 2 ? (wave >> 1) + 2 * i : wave + 4 * i; };
    const bool keys = 3 - wave < MAPS && p.append;  // this wave's row of the new key: map 3 - wave
    float qv[QR][J], kv_[J], wq[J], wk[J];
    auto rows = [&](int i0) {
#pragma unroll
        for (int i = 0; i < QR; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const float v = p.row[((size_t)(h0 + min(head_of(i0 + i), nh - 1)) * MAPS + map) * dimp + min(lane + 64 * j, dimp - 1)];
                qv[i][j] = lane + 64 * j < dimp ? v : 0.f;
            }
    };
    rows(0);
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int at = min(lane + 64 * j, p.dim - 1);
        kv_[j] = 0.f, wq[j] = wk[j] = 1.0f;
        if (keys && lane + 64 * j < dimp) kv_[j] = p.row[p.k_at + (kv * MAPS + 3 - wave) * dimp + lane + 64 * j];
        if (p.q_weight) wq[j] = p.q_weight[at];
        if (p.k_weight) wk[j] = p.k_weight[at];
    }
    float raw_v = 0.f;
    if (p.append && tid < vdimp) raw_v = p.row[p.v_at + kv * vdimp + tid];  // (vdimp <= 256)
    const int pos = __builtin_amdgcn_readfirstlane(posv), n_keys = pos + 1;
    struct {
        int first, base, per, used;
    } range;  // gqa_range
    range.first = p.chunk ? pos - (int)((unsigned)pos % (unsigned)p.chunk) : 0;
    if (p.window && pos - p.window + 1 > range.first) range.first = pos - p.window + 1;
    range.base = range.first & ~(kGqaTile - 1);
    const int tiles = (n_keys - range.base + kGqaTile - 1) / kGqaTile;
    range.per = (tiles + kGqaSplits - 1) / kGqaSplits;
    range.used = range.per == 1 ? tiles : (tiles + range.per - 1) / range.per;
    if ((int)blockIdx.z >= range.used) return;
    const int k0 = range.base + blockIdx.z * range.per * kGqaTile, k1 = min(k0 + range.per * kGqaTile, n_keys);
    float cs[J], sn[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        cs[j] = 1.0f, sn[j] = 0.f;
        if (p.turned && 64 * j < p.turned) {
            const size_t at = (size_t)pos * (p.turned >> 1) + (min(lane + 64 * j, p.turned - 1) >> 1);
            cs[j] = p.rope_cos[at], sn[j] = p.rope_sin[at];
        }
    }
    const float factor = p.q_factor[pos];
    u32x4 kf[2][MAPS][NK], vf[NV];
    auto fetch = [&](int kb) {  // (blocks lie below the capacity, a multiple of 128)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < MAPS; ++j)
#pragma unroll
                for (int kk = 0; kk < NK; ++kk)
                    kf[t][j][kk] = *reinterpret_cast<const u32x4 *>(K + ((size_t)j * p.capacity + kb + (r16 >> 2) * 8 + t * 4 + (r16 & 3)) * dimp + min(kk * 32, dimp - 32) + g * 8);
#pragma unroll
        for (int v = 0; v < NV; ++v) vf[v] = *reinterpret_cast<const u32x4 *>(V + (size_t)min(v * 16 + r16, vdimp - 1) * p.capacity + kb + g * 8);
    };
    constexpr bool kAhead = NK <= 4;  // the first block is requested ahead of the norms (registers allow it)
    const bool owner = k1 == n_keys && p.append;
    if (kAhead) fetch(k0 + wave * 32);
    // a row's element lane + 64 j: norm, weight, rotation by pairs of neighbours
    auto finished = [&](float v, float norm, float weight, int j) {
        const int i = lane + 64 * j;
        const float t = v * norm * (i < p.dim ? weight : 1.0f);
        if (!p.turned) return t;
        const float o = dpp<0xb1>(t);  // quad_perm [1,0,3,2]
        return i >= p.turned ? t : (i & 1) ? t * cs[j] + o * sn[j] : t * cs[j] - o * sn[j];
    };
    auto norm_of = [&](const float (&v)[J], bool normed) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) ss += v[j] * v[j];
        return normed ? 1.0f / sqrtf(wave_sum(ss) / (float)p.dim + p.eps) : 1.0f;
    };
    if (owner) {  // the record that holds the new position appends it (and puts it into its own fragments below)
        if (keys) {
            const float norm = norm_of(kv_, p.normed & 2);
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int i = lane + 64 * j;
                const float k = finished(kv_[j], norm, wk[j], j);
                if (i < dimp) {
                    const uint16_t b = f2bf(k);
                    K[((size_t)(3 - wave) * p.capacity + pos) * dimp + i] = b;
                    newk[3 - wave][i] = b;
                }
            }
        }
        if (tid < vdimp) {
            const uint16_t b = f2bf(raw_v);
            V[(size_t)tid * p.capacity + pos] = b;
            newv[tid] = b;
        }
    }
    for (int i0 = 0; head_of(i0) < nh; i0 += QR) {
        if (i0) rows(i0);
#pragma unroll
        for (int i = 0; i < QR; ++i) {
            if (head_of(i0 + i) >= nh) continue;
            const float norm = norm_of(qv[i], p.normed & 1) * factor;
#pragma unroll
            for (int j = 0; j < J; ++j)
                if (lane + 64 * j < NK * 32) area[(map * 16 + head_of(i0 + i)) * QS + lane + 64 * j] = finished(qv[i][j], norm, wq[j], j);
        }
    }
    __syncthreads();
    SplitFrag q[MAPS][NK];  // (lanes past the last head: whatever lies there; a column of the products is a head of its own)
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
            const float *src = area + (m * 16 + r16) * QS + kk * 32 + g * 8;
            q[m][kk] = split8(*reinterpret_cast<const f32x4 *>(src), *reinterpret_cast<const f32x4 *>(src + 4));
        }
    FarPenalty far{0.f, 0.f};
    if (p.far_weight) far.weight = p.far_weight[min(h0 + r16, p.heads - 1)] * 0.69314718055994531f, far.rate = p.far_rate[min(h0 + r16, p.heads - 1)];
    f32x4 o[NV][MAPS];
    float m[MAPS], l[MAPS];
#pragma unroll
    for (int j = 0; j < MAPS; ++j) {
        m[j] = -INFINITY, l[j] = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v) o[v][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int kb = k0 + wave * 32; kb < k1; kb += 128) {
        if (!kAhead || kb >= k0 + 128) fetch(kb);
        if (kb + 32 <= range.first) continue;  // (another chunk's keys)
        if (owner && pos - kb < 32) {  // the new position, which memory need not show yet
            const int at = pos - kb, t = (at >> 2) & 1;
            const bool mine = r16 == (at >> 3) * 4 + (at & 3);
#pragma unroll
            for (int j = 0; j < MAPS; ++j)
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) {
                    const u32x4 k = *reinterpret_cast<const u32x4 *>(&newk[j][min(kk * 32, dimp - 32) + g * 8]);
                    if (mine && t == 0) kf[0][j][kk] = k;
                    if (mine && t == 1) kf[1][j][kk] = k;
                }
            if (g == at >> 3) {
                const uint32_t keep = (at & 1) ? 0xffffu : 0xffff0000u, sh = (at & 1) * 16;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const uint32_t n = (uint32_t)newv[min(v * 16 + r16, vdimp - 1)] << sh;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (e == (at & 7) >> 1) vf[v][e] = (vf[v][e] & keep) | n;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < MAPS; ++j) {
            f32x4 s[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f32x4 hi = f32x4{0.f, 0.f, 0.f, 0.f}, lo = hi;
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) {  // (steps past dimp: the query is zero there)
                    hi = mfma_bf16(__builtin_bit_cast(bf16x8, kf[t][j][kk]), q[j][kk].hi, hi);
                    lo = mfma_bf16(__builtin_bit_cast(bf16x8, kf[t][j][kk]), q[j][kk].lo, lo);
                }
                s[t] = hi + lo;
                if (MAPS == 1 && p.far_weight)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[t][e] = nearer(s[t][e], far, pos - (kb + g * 8 + t * 4 + e));
                s[t] *= kLog2e;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int key = kb + g * 8 + t * 4 + e;
                    s[t][e] = key < k1 && key >= range.first ? s[t][e] : -INFINITY;
                }
            }
            float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])), fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
            mx = fmaxf(m[j], rows_max(mx));
            const float al = __builtin_amdgcn_exp2f(m[j] - mx);
            m[j] = mx;
            f32x4 w[2];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) w[t][e] = __builtin_amdgcn_exp2f(s[t][e] - mx);
            l[j] = l[j] * al + ((w[0][0] + w[0][1]) + (w[0][2] + w[0][3])) + ((w[1][0] + w[1][1]) + (w[1][2] + w[1][3]));
            const SplitFrag pf = split8(w[0], w[1]);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                o[v][j] *= al;
                o[v][j] = mfma_bf16(__builtin_bit_cast(bf16x8, vf[v]), pf.hi, o[v][j]);
                o[v][j] = mfma_bf16(__builtin_bit_cast(bf16x8, vf[v]), pf.lo, o[v][j]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < MAPS; ++j) {
        const float t = rows_sum(l[j]);
        if (g == 0) sm[wave][j][r16] = m[j], sl[wave][j][r16] = t;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MAPS; ++j) {
        const float M = fmaxf(fmaxf(sm[0][j][r16], sm[1][j][r16]), fmaxf(sm[2][j][r16], sm[3][j][r16]));
        const float w = m[j] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[j] - M);
        if (r16 < nh)
#pragma unroll
            for (int v = 0; v < NV; ++v)
                if (v * 16 < vdimp) *reinterpret_cast<f32x4 *>(area + ((size_t)(wave * MAPS + j) * nh + r16) * vdimp + v * 16 + g * 4) = o[v][j] * w;
    }
    __syncthreads();
    const int n_rows = MAPS * nh;
    for (int r = tid >> 5; r < n_rows; r += 8) {
        const int j = MAPS == 2 && r >= nh ? 1 : 0, hh = r - j * nh;
        float *rec = p.scratch + ((size_t)((h0 + hh) * MAPS + j) * kGqaSplits + blockIdx.z) * (kGqaRecHead + vdimp);
        for (int c = (tid & 31) * 4; c < vdimp; c += 128) {
            const float *src = area + (size_t)r * vdimp + c;
            const size_t step = (size_t)n_rows * vdimp;
            *reinterpret_cast<f32x4 *>(rec + kGqaRecHead + c) = (*reinterpret_cast<const f32x4 *>(src) + *reinterpret_cast<const f32x4 *>(src + step)) +
                                                                (*reinterpret_cast<const f32x4 *>(src + 2 * step) + *reinterpret_cast<const f32x4 *>(src + 3 * step));
        }
        if ((tid & 31) == 0) {
            const float M = fmaxf(fmaxf(sm[0][j][hh], sm[1][j][hh]), fmaxf(sm[2][j][hh], sm[3][j][hh]));
            float L = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) L += sm[w][j][hh] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sm[w][j][hh] - M) * sl[w][j][hh];
            rec[0] = M, rec[1] = L;
        }
    }
}

template <int NK, int NV>
static hipError_t step_go(const Gqa &g, const GqaStep &a, hipStream_t s) {
    const int splits = gqa_records(g), group = (int)(g.heads / g.kv_heads), nh = min(16, group);
    const size_t queries = g.maps * 16 * (NK * 32 + 4), outs = 4 * g.maps * nh * g.vdimp, lds = (queries > outs ? queries : outs) * sizeof(float);
    auto fn = g.maps == 2 ? k_gqa_step<NK, NV, 2> : k_gqa_step<NK, NV, 1>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    GqaStepK k;
    k.row = a.row, k.q_weight = g.q_weight, k.k_weight = g.k_weight, k.q_factor = g.q_factor, k.rope_cos = g.rope_cos, k.rope_sin = g.rope_sin, k.far_weight = g.far_weight;
    k.far_rate = g.far_rate, k.pos = a.pos, k.K = (uint16_t *)g.kcache, k.V = (uint16_t *)g.vcache, k.scratch = a.scratch, k.eps = g.eps, k.heads = (int)g.heads, k.group = group;
    k.dim = (int)g.dim, k.dimp = (int)g.dimp, k.vdimp = (int)g.vdimp, k.capacity = (int)g.capacity, k.turned = (int)g.rot_dims, k.append = !g.queries_only;
    k.chunk = g.chunk < g.capacity ? (int)g.chunk : 0, k.window = g.window < g.capacity ? (int)g.window : 0;  // (as large as the cache: no position has keys outside)
    k.normed = (g.q_weight || g.unit_norm ? 1 : 0) | (g.k_weight || g.unit_norm ? 2 : 0);
    k.k_at = (int)(g.heads * g.maps * g.dimp), k.v_at = g.values_are_keys ? k.k_at : (int)((g.heads + g.kv_heads) * g.maps * g.dimp);
    hipLaunchKernelGGL(fn, dim3(g.kv_heads, (group + 15) / 16, splits), dim3(256), lds, s, k);
    return hipGetLastError();
}

hipError_t launch_gqa_step(const Gqa &g, const GqaStep &a, hipStream_t s) {
    if (!gqa_supported((int)g.dimp, (int)g.vdimp)) return hipErrorInvalidValue;
    if (g.dimp <= 64 && g.vdimp <= 64) return step_go<2, 4>(g, a, s);
    if (g.dimp <= 64 && g.vdimp <= 128) return step_go<2, 8>(g, a, s);
    if (g.dimp <= 128 && g.vdimp <= 128) return step_go<4, 8>(g, a, s);
    return step_go<8, 16>(g, a, s);
}

// ---- records -> output ------------------------------------------------------------------------------------------------
template <class TO>
__global__ __launch_bounds__(256) void k_gqa_merge(Gqa p, const int *pos_ptr, int q0, const float *scratch, TO *out, size_t ldo) {
    extern __shared__ __attribute__((aligned(16))) float part[];  // [maps][2][vdimp]
    static_assert(kGqaSplits == 128, "two records per lane of a wave");
    __shared__ float ws[2][kGqaSplits], sinv[2], slot[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.x, qi = blockIdx.z, maps = (int)p.maps, vdimp = (int)p.vdimp;
    const float z = p.gate ? gate_logit(p, qi, h, min(tid, vdimp - 1)) : 0.f, sink = p.sink ? p.sink[h] * kLog2e : -INFINITY;  // (ahead of the chain that starts with the position)
    const int used = gqa_range(p, *pos_ptr + q0 + qi).used;
    const size_t stride = kGqaRecHead + vdimp;
    const float *rec = scratch + ((size_t)qi * p.heads + h) * maps * kGqaSplits * stride;
    // 32 lanes of four columns; eight groups share maps and records.  Each group's first records are requested ahead of the weights.
    const int grp = tid >> 5, gm = maps == 2 ? grp & 1 : 0, gs = maps == 2 ? grp >> 1 : grp, gn = maps == 2 ? 4 : 8, i0 = (tid & 31) * 4;
    const float *vec = rec + (size_t)gm * kGqaSplits * stride + kGqaRecHead;
    constexpr int AHEAD = 4;
    f32x4 first[AHEAD];
#pragma unroll
    for (int e = 0; e < AHEAD; ++e) first[e] = *reinterpret_cast<const f32x4 *>(vec + min(gs + e * gn, used - 1) * stride + min(i0, vdimp - 4));
    if (wave < maps) {
        const float *r = rec + (size_t)wave * kGqaSplits * stride;
        float mv[2], lv[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int i = lane + 64 * e;
            mv[e] = i < used ? r[i * stride] : -INFINITY;
            lv[e] = i < used ? r[i * stride + 1] : 0.f;
        }
        const float M = fmaxf(sink, rows_max(row_max(fmaxf(mv[0], mv[1]))));
        float den = 0.f;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float w = lane + 64 * e < used ? exp2f(mv[e] - M) : 0.f;
            ws[wave][lane + 64 * e] = w;
            den += w * lv[e];
        }
        den = wave_sum(den) + (p.sink ? exp2f(sink - M) : 0.f);
        if (lane == 0) sinv[wave] = 1.0f / den;
    }
    __syncthreads();
    const float gate = p.gate ? activate(z, BITNET_HIP_ACT_SIGMOID) : 1.0f;
    for (int i = i0; i < vdimp; i += 128) {
        const float *r = vec + i;
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        int k0 = gs;
        if (i == i0) {
#pragma unroll
            for (int e = 0; e < AHEAD; ++e) acc += ws[gm][gs + e * gn] * first[e];  // (weights past the last record are zero)
            k0 += AHEAD * gn;
        }
#pragma unroll 8
        for (int k = k0; k < used; k += gn) acc += ws[gm][k] * *reinterpret_cast<const f32x4 *>(r + k * stride);
        *reinterpret_cast<f32x4 *>(part + (size_t)grp * vdimp + i) = acc;
    }
    __syncthreads();
    float v = 0.f;
    const bool live = tid < vdimp;  // (vdimp <= 256; wider heads loop below)
    TO *dst = out + (size_t)qi * ldo + (size_t)h * vdimp;
    auto value = [&](int i) {
        if (maps == 1) {
            float t = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) t += part[k * vdimp + i];
            const float own = p.gate_columns && vdimp > 256 ? activate(gate_logit(p, qi, h, i), BITNET_HIP_ACT_SIGMOID) : gate;
            return t * (sinv[0] * own);
        }
        const float a = (part[i] + part[2 * vdimp + i]) + (part[4 * vdimp + i] + part[6 * vdimp + i]);
        const float b = (part[vdimp + i] + part[3 * vdimp + i]) + (part[5 * vdimp + i] + part[7 * vdimp + i]);
        return a * sinv[0] - p.lambda * (b * sinv[1]);
    };
    if (vdimp <= 256) {
        v = live ? value(tid) : 0.f;
        if (maps == 2) v *= gate * p.out_scale / sqrtf(group_sum<4>(v * v, slot) / (float)p.vdim + p.eps);
        if (live) st_act(dst, tid, v);
        return;
    }
    float ss = 0.f, f = 1.0f;
    for (int i = tid; i < vdimp; i += 256) v = value(i), ss += v * v;
    if (maps == 2) f = gate * p.out_scale / sqrtf(group_sum<4>(ss, slot) / (float)p.vdim + p.eps);
    for (int i = tid; i < vdimp; i += 256) st_act(dst, i, value(i) * f);
}

hipError_t launch_gqa_merge(const Gqa &g, const int *pos, int q0, int nq, const float *scratch, void *out, size_t ldo, int out_bf16, hipStream_t s) {
    const size_t lds = 8 * g.vdimp * sizeof(float);
    if (lds > 65536) return hipErrorInvalidValue;
    if (out_bf16)
        hipLaunchKernelGGL(k_gqa_merge<uint16_t>, dim3(g.heads, 1, nq), dim3(256), lds, s, g, pos, q0, scratch, (uint16_t *)out, ldo);
    else
        hipLaunchKernelGGL(k_gqa_merge<float>, dim3(g.heads, 1, nq), dim3(256), lds, s, g, pos, q0, scratch, (float *)out, ldo);
    return hipGetLastError();
}

// ---- records -> output -> product -------------------------------------------------------------------------------------
// The merge of up to four records and the product behind it in one launch, for weights that begin off four bytes (k_gqa_project below takes all others, more records and every step of the models): every
// workgroup forms the whole output in LDS, as k_dense_gemv forms its input, and its waves take rows of the product.  Nothing that is requested hangs on the position: a thread asks for all records
// of its columns, with their maxima and sums, and makes their weights itself; what the position says only masks them.  The product's weights go out behind.
struct GqaOutK {
    Gqa g;
    const int *pos;
    const float *scratch, *bias;
    const uint16_t *w;
    float *y;
    int rows, cols, ld, kp, records;
    unsigned magic;  // ceil(2^20 / pieces of a head)
};
constexpr int kOutRecords = 4, kOutPieces = 4, kOutChunks = 3;  // records, pieces of four columns per thread, chunks of 512 columns in flight

__global__ __launch_bounds__(256) void k_gqa_out(GqaOutK p) {
    extern __shared__ __attribute__((aligned(16))) float xs[];
    constexpr int NU = kOutPieces, NB = kOutRecords, U = kOutChunks;
    const Gqa &g = p.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, vdimp = (int)g.vdimp, pieces = (int)g.heads * (vdimp >> 2);
    const int here = *p.pos;
    const unsigned stride = kGqaRecHead + vdimp;
    float2 ml[NU][NB];
    f32x4 vec[NU][NB], zc[NU];
    float sink[NU], z[NU];
#pragma unroll
    for (int j = 0; j < NU; ++j) {
        if (j > 0 && 256 * j >= pieces) continue;
        const int u = min(tid + 256 * j, pieces - 1), h = (int)((unsigned)u * p.magic >> 20);
        const float *rec = p.scratch + (unsigned)h * (kGqaSplits * stride), *v = rec + kGqaRecHead + (u - h * (vdimp >> 2)) * 4;
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            if (e >= 2 && p.records <= 2) continue;
            ml[j][e] = *reinterpret_cast<const float2 *>(rec + e * stride);
            vec[j][e] = *reinterpret_cast<const f32x4 *>(v + e * stride);
        }
        sink[j] = g.sink ? g.sink[h] * kLog2e : -INFINITY;
        z[j] = g.gate && !g.gate_columns ? ((const float *)g.gate)[h] : 0.f;
        zc[j] = g.gate && g.gate_columns ? *reinterpret_cast<const f32x4 *>((const float *)g.gate + 4 * u) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int l8 = lane * 8, last_col = p.cols - 8;
    u32x4 w[U];
    auto fetch = [&](int row, int k0) {
        const uint16_t *wr = p.w + (size_t)row * p.ld;
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wr + min(k0 + u * 512 + l8, last_col)));
    };
    int row = blockIdx.x * 4 + wave;
    const int n = gridDim.x * 4;
    if (row < p.rows) fetch(row, 0);
    const int used = min(gqa_range(g, here).used, p.records <= 2 ? 2 : NB);
#pragma unroll
    for (int j = 0; j < NU; ++j) {
        if (j > 0 && 256 * j >= pieces) continue;
        float M = sink[j], den = 0.f, e2[NB];
#pragma unroll
        for (int e = 0; e < NB; ++e) M = e < used ? fmaxf(M, ml[j][e].x) : M;
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            e2[e] = e < used ? exp2f(ml[j][e].x - M) : 0.f;
            den += e < used ? e2[e] * ml[j][e].y : 0.f;
        }
        if (g.sink) den += exp2f(sink[j] - M);
        const float f = (g.gate && !g.gate_columns ? activate(z[j], BITNET_HIP_ACT_SIGMOID) : 1.0f) / den;
        f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < NB; ++e)
            if (e < used) v += e2[e] * vec[j][e];
        v *= f;
        if (g.gate && g.gate_columns)
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] *= activate(zc[j][c], BITNET_HIP_ACT_SIGMOID);
        if (tid + 256 * j < pieces) reinterpret_cast<f32x4 *>(xs)[tid + 256 * j] = v;
    }
    for (int i = 4 * pieces + tid; i < p.kp; i += 256) xs[i] = 0.f;
    __syncthreads();
    for (; row < p.rows; row += n) {
        float acc = 0.f;
        for (int k0 = 0; k0 < p.kp; k0 += U * 512) {
            u32x4 c[U];
#pragma unroll
            for (int u = 0; u < U; ++u) c[u] = w[u];
            if (k0 + U * 512 < p.kp)
                fetch(row, k0 + U * 512);
            else if (row + n < p.rows)
                fetch(row + n, 0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const f32x4 x[2] = {*reinterpret_cast<const f32x4 *>(xs + k0 + u * 512 + l8), *reinterpret_cast<const f32x4 *>(xs + k0 + u * 512 + l8 + 4)};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc = fmaf(x[i >> 1][2 * i & 3], __builtin_bit_cast(float, c[u][i] << 16), acc);
                    acc = fmaf(x[i >> 1][(2 * i & 3) + 1], __builtin_bit_cast(float, c[u][i] & 0xffff0000u), acc);
                }
            }
        }
        acc = wave_sum(acc);
        if (lane == 0) p.y[row] = acc + (p.bias ? p.bias[row] : 0.f);
    }
}

// the most records that one launch may take in place of two; 0: none
int gqa_out_records(const Gqa &g, int cols) {
    if (g.maps != 1 || g.heads * g.vdimp > 4096 || (size_t)cols < g.heads * g.vdimp || cols > 4096 || (g.gate && !g.gate_f32)) return 0;
    return kOutRecords;
}

hipError_t launch_gqa_out(const GqaOut &a, hipStream_t s) {
    if (a.records < 1 || a.records > gqa_out_records(a.g, a.cols)) return hipErrorInvalidValue;
    // (its loads want four bytes; us, an instance of k_gqa_out for these sizes / this, weights on sixteen bytes and on eight, at 200 | 500 keys: 12 heads of 128, 1536 rows 3.3 / 2.9 | 3.9 / 3.0; 24, 3072 rows
    // 5.2 / 4.3 | 6.3 / 4.7; 32 of 64, 3072 rows 4.0 / 4.1 | 5.1 / 4.4.  The one instance that is left, against those: 3.3 / 3.8 | 4.0 / 4.1; 5.3 / 6.0 | 6.5 / 6.8; 4.1 / 5.1 | 5.1 / 5.8)
    if ((uintptr_t)a.w % 4 == 0 && a.ld <= 32768) return launch_gqa_project(a, s);
    GqaOutK k;
    k.g = a.g, k.pos = a.pos, k.scratch = a.scratch, k.bias = a.bias, k.w = a.w, k.y = a.y, k.rows = a.rows, k.cols = a.cols, k.ld = a.ld, k.records = a.records;
    k.kp = (a.cols + 512 * kOutChunks - 1) / (512 * kOutChunks) * (512 * kOutChunks);
    k.magic = ((1u << 20) + a.g.vdimp / 4 - 1) / (unsigned)(a.g.vdimp / 4);
    int n_wg = (a.rows + 3) / 4;
    if (n_wg > 768) {
        const int rounds = (n_wg + 767) / 768;
        n_wg = (n_wg + rounds - 1) / rounds;
    }
    hipLaunchKernelGGL(k_gqa_out, dim3(n_wg), dim3(256), (size_t)k.kp * sizeof(float), s, k);
    return hipGetLastError();
}

// Up to twelve records on the lanes of k_dense_gemv_formed (dense.hpp, SharedRows): each merges the records of its own eight columns in registers, for all rows of its workgroup, and nothing goes
// through LDS ahead of the products.  As above nothing that is requested hangs on the position.
struct GqaProjectK {
    Gqa g;
    const int *pos;
    const float *scratch, *bias;
    const uint16_t *w;
    float *y;
    int rows, ld, rows_wg;
    unsigned magic;  // ceil(2^20 / eights of a head)
};
constexpr int kProjectRows = 64;

template <int NB>
__global__ __launch_bounds__(512) void k_gqa_project(GqaProjectK p) {
    __shared__ __attribute__((aligned(16))) float parts[kProjectRows + 4][8];
    const Gqa &g = p.g;
    const int here = *p.pos;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), vdimp = (int)g.vdimp, n = (int)g.heads * vdimp;
    const unsigned stride = kGqaRecHead + vdimp;
    const int row0 = blockIdx.x * p.rows_wg, n_rows = min(p.rows_wg, p.rows - row0);
    const int at = wave * 512 + lane * 8, col[1] = {min(at, n - 8)}, head = (int)((unsigned)(col[0] >> 3) * p.magic >> 20);
    const bool inside[1] = {at < n};
    const float *rec = p.scratch + (unsigned)head * (kGqaSplits * stride), *v = rec + kGqaRecHead + (col[0] - head * vdimp);
    float2 ml[NB];
    f32x4 vec[NB][2], zc[2];
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        ml[e] = *reinterpret_cast<const float2 *>(rec + e * stride);
        vec[e][0] = *reinterpret_cast<const f32x4 *>(v + e * stride), vec[e][1] = *reinterpret_cast<const f32x4 *>(v + e * stride + 4);
    }
    const float sink = g.sink ? g.sink[head] * kLog2e : -INFINITY, z = g.gate && !g.gate_columns ? ((const float *)g.gate)[head] : 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h) zc[h] = g.gate && g.gate_columns ? *reinterpret_cast<const f32x4 *>((const float *)g.gate + col[0] + 4 * h) : f32x4{0.f, 0.f, 0.f, 0.f};
    const float bias = p.bias && tid < n_rows ? p.bias[row0 + tid] : 0.f;
    SharedRows<4, 1> weights(p.w + (size_t)row0 * p.ld, n_rows, p.ld, col, inside);
    weights.request();
    const int used = gqa_range(g, here).used;
    float M = sink;
#pragma unroll
    for (int e = 0; e < NB; ++e) M = e < used ? fmaxf(M, ml[e].x) : M;
    float den = g.sink ? exp2f(sink - M) : 0.f;
    f32x4 x[1][2] = {{f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}}};
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        if (e >= used) continue;
        const float w = exp2f(ml[e].x - M);
        den += w * ml[e].y;
        x[0][0] += w * vec[e][0], x[0][1] += w * vec[e][1];
    }
    const float f = (g.gate && !g.gate_columns ? activate(z, BITNET_HIP_ACT_SIGMOID) : 1.0f) / den;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        x[0][h] *= f;
        if (g.gate && g.gate_columns)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[0][h][c] *= activate(zc[h][c], BITNET_HIP_ACT_SIGMOID);
        if (!inside[0]) x[0][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    weights.run(x, parts, wave, lane);
    __syncthreads();
    if (tid < n_rows) p.y[row0 + tid] = waves_total(parts[tid], (int)blockDim.x >> 6) + bias;
}

int gqa_project_records(const Gqa &g, int cols) { return g.maps != 1 || g.heads * g.vdimp > 4096 || (size_t)cols < g.heads * g.vdimp || (g.gate && !g.gate_f32) ? 0 : 12; }

hipError_t launch_gqa_project(const GqaOut &a, hipStream_t s) {
    if (a.records < 1 || a.records > gqa_project_records(a.g, a.cols)) return hipErrorInvalidValue;
    GqaProjectK k;
    k.g = a.g, k.pos = a.pos, k.scratch = a.scratch, k.bias = a.bias, k.w = a.w, k.y = a.y, k.rows = a.rows, k.ld = a.ld;
    k.magic = ((1u << 20) + a.g.vdimp / 8 - 1) / (unsigned)(a.g.vdimp / 8);
    const int waves = ((int)(a.g.heads * a.g.vdimp) + 511) / 512;
    k.rows_wg = std::min({(a.rows + 1023) / 1024 * 4, kProjectRows, 64 * waves});
    hipLaunchKernelGGL(a.records <= 2 ? k_gqa_project<2> : a.records <= 4 ? k_gqa_project<4> : a.records <= 8 ? k_gqa_project<8> : k_gqa_project<12>, dim3((a.rows + k.rows_wg - 1) / k.rows_wg), dim3(64 * waves), 0, s, k);
    return hipGetLastError();
}

// buffers of a tile in LDS: two where the two tiles that are under way on a compute unit (one of the largest heads) leave room
constexpr int prefill_buffers(int nk, int nv, int maps) { return (nv > 8 || nk > 4 ? 2 : 4) * (maps * 64 * (nk * 64 + 32) + nv * 16 * (64 * 2 + 32)) <= 163840 ? 2 : 1; }

// ---- prompt -----------------------------------------------------------------------------------------------------------
// One workgroup: one head, four waves; a wave holds two slots of 16 queries: both maps of one query tile, or two tiles of the only map.  Key tiles
// of 64 (every map's) and the values of the tile staged through registers into LDS one step ahead.
// G = 2: two such groups of four waves share the keys of the same queries, tile by tile in turn, and meet in LDS at the end.  A prompt's last queries see all of its keys and its
// first next to none: with one group per workgroup the longest walk takes 2.2 us a tile whatever its neighbour does, with two it is half as long at 3.3 us a step.
// Heads that need more than 256 registers keep one group; two_groups says when the others take two.
// Bound by the two waves of a SIMD and their waits, not by memory (16 heads, 4096 tokens: matrix cores 40 %, vector instructions half of the time).  Hence: rows of a tile lie 32 bytes past a
// multiple of 64 apart (reads of 16 rows by 64 bytes without bank conflicts: 16 bytes past it they took twice the cycles), keys in the order in which a lane's weights are eight
// neighbours (one 16-byte read of the values where two of 8 were), a key's row is written by neighbouring threads, operands are read four ahead of their products, and two
// buffers take one barrier a step, with the stores between the weights and their products.  us, each of these in turn, 16 heads of 128 columns at 4096 tokens: 130.9, 124.5 (order), 121.0
// (writes), 120.5 (rows), 111.9 (reads ahead), 109.7 (buffers).  24 heads, 3000 tokens 121 -> 105; 32 heads, 1531 49.4 -> 42; 24 of two maps, 1531 62 -> 53, 300 13.9 -> 12.5.
// FAR: with a distance penalty, gates per column, or both.
// records: gridDim.y workgroups share a block's tiles of keys, in stretches, and each leaves its outputs, maxima and sums for k_gqa_merge_parts (which counts the sink).
template <int NK, int NV, int MAPS, bool FAR, int G>
__global__ __launch_bounds__(256 * G, NV > 8 || NK > 4 ? 1 : 2) void k_gqa_prefill(Gqa p, const uint16_t *Q, size_t ldq, int n_ctx, int nq, uint16_t *out, size_t ldo, int n_qb, float *records) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int SLOTS = 2, QW = 16 * SLOTS / MAPS, KS = NK * 64 + 32, VS = 64 * 2 + 32, NVL = NV / 2, AHEAD = 4;
    const int grp = G == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4;
    constexpr int KB = MAPS * 64 * KS, TILE = KB + NV * 16 * VS, BUFS = prefill_buffers(NK, NV, MAPS);
    uint8_t *lk = lds + grp * BUFS * TILE;
    const int heads = (int)p.heads, dimp = (int)p.dimp, vdimp = (int)p.vdimp;
    // Consecutive workgroups go to the eight XCDs in turn.  Longest blocks first; an XCD keeps heads / 8 neighbouring heads of its own (their keys
    // and values stay in its L2), the heads left over move from XCD to XCD with the block so that all eight carry the same work.
    const int x = blockIdx.x & 7, rest = blockIdx.x >> 3, own = heads >> 3, left = heads & 7, per = own + (left ? 1 : 0);
    const int level = rest / per, slot = rest - level * per, r = (x + 8 * left - (level % 8) * left) & 7;
    if (slot == own && r >= left) return;
    const int h = slot < own ? x * own + slot : 8 * own + r, qb = n_qb - 1 - level;
    const int kv = h / (int)(p.heads / p.kv_heads), q0 = qb * 4 * QW, pos0 = n_ctx - nq, qw = q0 + wave * QW;
    bf16x8 qf[SLOTS][NK];
    int qpos[SLOTS], qfirst[SLOTS];
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) {
        const int tile = t / MAPS, map = t % MAPS, qi = min(qw + tile * 16 + r16, nq - 1);
        qpos[t] = pos0 + qw + tile * 16 + r16;
        qfirst[t] = gqa_first(p, qpos[t]);
        const uint16_t *q = Q + (size_t)qi * ldq + (size_t)(h * MAPS + map) * dimp;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
            u32x4 v = *reinterpret_cast<const u32x4 *>(q + min(kk * 32, dimp - 32) + g * 8);
            const uint32_t keep = kk * 32 < dimp ? 0xffffffffu : 0u;
            qf[t][kk] = __builtin_bit_cast(bf16x8, u32x4{v.x & keep, v.y & keep, v.z & keep, v.w & keep});
        }
    }
    f32x4 o[NV][SLOTS];
    float m[SLOTS], l[SLOTS];
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) {
        // (finite: with chunks a tile may hold no key that a query sees; the sink counts once per query, four lanes share one)
        m[t] = MAPS == 1 && p.sink && grp == 0 && !records ? p.sink[h] * kLog2e : -1e30f, l[t] = MAPS == 1 && p.sink && g == 0 && grp == 0 && !records ? 1.0f : 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v) o[v][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint16_t *K = (const uint16_t *)p.kcache + (size_t)kv * MAPS * p.capacity * dimp, *V = (const uint16_t *)p.vcache + (size_t)kv * vdimp * p.capacity;
    u32x4 kreg[MAPS][NK], vreg[NVL];
    // keys: a row of the tile by KC neighbouring threads; row p of 32 in LDS is key 8 (p >> 2 & 3) + 4 (p >> 4) + (p & 3)
    constexpr int KC = NK * 4, KR = 256 / KC;
    const unsigned koff = (unsigned)((tid / KC) * dimp * 2 + min((tid % KC) * 16, dimp * 2 - 16));
    uint8_t *kw[NK];
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        const int key = tid / KC + j * KR, row = (key & 32) + (key >> 2 & 1) * 16 + (key >> 3 & 3) * 4 + (key & 3);
        kw[j] = lk + row * KS + (tid % KC) * 16;
    }
    const size_t voff = (size_t)(tid >> 3) * p.capacity * 2 + (tid & 7) * 16;
#pragma unroll
    for (int j = 0; j < NVL; ++j) vreg[j] = u32x4{0u, 0u, 0u, 0u};
    auto fetch = [&](int key0) {  // (whole tiles: the capacity is a multiple of 64)
#pragma unroll
        for (int mp = 0; mp < MAPS; ++mp) {
            const char *kb = (const char *)(K + ((size_t)mp * p.capacity + key0) * dimp);
#pragma unroll
            for (int j = 0; j < NK; ++j) kreg[mp][j] = *reinterpret_cast<const u32x4 *>(kb + (size_t)(j * KR * 2) * dimp + koff);
        }
        const char *vb = (const char *)(V + key0);
#pragma unroll
        for (int j = 0; j < NVL; ++j)
            if (j * 32 < vdimp) vreg[j] = *reinterpret_cast<const u32x4 *>(vb + (size_t)j * 64 * p.capacity + voff);
    };
    int n_tiles = (min(n_ctx, pos0 + q0 + 4 * QW) + 63) / 64;
    const FarPenalty far = far_penalty(p, h);
    // tiles from the first key of the workgroup's first query on; a wave leaves out what lies ahead of its own first key
    int t_first = gqa_first(p, pos0 + q0) >> 6;
    const int w_first = gqa_first(p, pos0 + qw), w_last = gqa_first(p, pos0 + qw + QW - 1);
    if (records) {
        const int each = (n_tiles - t_first + (int)gridDim.y - 1) / (int)gridDim.y;
        t_first = min(t_first + (int)blockIdx.y * each, n_tiles), n_tiles = min(t_first + each, n_tiles);
    }
    auto store = [&](int at) {
#pragma unroll
        for (int mp = 0; mp < MAPS; ++mp)
#pragma unroll
            for (int j = 0; j < NK; ++j) *reinterpret_cast<u32x4 *>(kw[j] + at + mp * 64 * KS) = kreg[mp][j];
#pragma unroll
        for (int j = 0; j < NVL; ++j) *reinterpret_cast<u32x4 *>(lk + at + KB + ((tid >> 3) + 32 * j) * VS + (tid & 7) * 16) = vreg[j];
    };
    fetch(max(min(t_first + grp, n_tiles - 1), 0) * 64);
    if (BUFS == 2) {
        store(0);
        if (t_first + grp + G < n_tiles) fetch((t_first + grp + G) * 64);
    }
    SplitFrag pf[2][SLOTS];
    auto values = [&](const uint8_t *from) {
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const bf16x8 a = *reinterpret_cast<const bf16x8 *>(from + (v * 16 + r16) * VS + ks * 64 + g * 16);
#pragma unroll
                for (int t = 0; t < SLOTS; ++t) {
                    o[v][t] = mfma_bf16(a, pf[ks][t].hi, o[v][t]);
                    o[v][t] = mfma_bf16(a, pf[ks][t].lo, o[v][t]);
                }
            }
        reads_ahead<NV * 2, 2 * SLOTS, AHEAD>();
    };
    int at = 0;  // the tile's buffer
    for (int t0 = t_first; t0 < n_tiles; t0 += G) {
        const int kt0 = t0 + grp, key0 = kt0 * 64;
        __syncthreads();
        if (BUFS == 1) {
            store(0);
            __syncthreads();
            if (kt0 + G < n_tiles) fetch(key0 + G * 64);
        }
        const bool seen = !(key0 > pos0 + qw + QW - 1 || key0 + 63 < w_first || (G == 2 && kt0 >= n_tiles));  // (else: no key of the tile is seen by this wave's queries)
        const uint8_t *kt_ = lk + at;
        if (seen) {
        f32x4 s[4][SLOTS];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) s[kt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < NK; ++kk)
#pragma unroll
                for (int t = 0; t < SLOTS; ++t) {
                    const bf16x8 a = *reinterpret_cast<const bf16x8 *>(kt_ + ((t % MAPS) * 64 + kt * 16 + r16) * KS + kk * 64 + g * 16);
                    s[kt][t] = mfma_bf16(a, qf[t][kk], s[kt][t]);
                }
        }
        reads_ahead<4 * NK * MAPS, SLOTS / MAPS, AHEAD>();
        __builtin_amdgcn_sched_barrier(0);
        if (FAR && p.far_weight)
#pragma unroll
            for (int t = 0; t < SLOTS; ++t)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[kt][t][i] = nearer(s[kt][t][i], far, qpos[t] - (key0 + (kt >> 1) * 32 + g * 8 + (kt & 1) * 4 + i));
        if (key0 + 63 > pos0 + qw)  // the diagonal
#pragma unroll
            for (int t = 0; t < SLOTS; ++t)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[kt][t][i] = key0 + (kt >> 1) * 32 + g * 8 + (kt & 1) * 4 + i > qpos[t] ? -INFINITY : s[kt][t][i];
        if (key0 < w_last)  // an earlier chunk of some of the queries
#pragma unroll
            for (int t = 0; t < SLOTS; ++t)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[kt][t][i] = key0 + (kt >> 1) * 32 + g * 8 + (kt & 1) * 4 + i < qfirst[t] ? -INFINITY : s[kt][t][i];
        float mn[SLOTS];
        bool grows = false;
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            float mx = fmaxf(fmaxf(s[0][t][0], s[0][t][1]), fmaxf(s[0][t][2], s[0][t][3]));
#pragma unroll
            for (int kt = 1; kt < 4; ++kt) mx = fmaxf(mx, fmaxf(fmaxf(s[kt][t][0], s[kt][t][1]), fmaxf(s[kt][t][2], s[kt][t][3])));
            mn[t] = fmaxf(m[t], rows_max(mx) * kLog2e);
            grows = grows || mn[t] > m[t];
        }
        if (__any(grows)) {
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) {
                const float al = __builtin_amdgcn_exp2f(m[t] - mn[t]);
                m[t] = mn[t];
                l[t] *= al;
#pragma unroll
                for (int v = 0; v < NV; ++v) o[v][t] *= al;
            }
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) {
                f32x4 w[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[j][i] = __builtin_amdgcn_exp2f(fmaf(s[2 * ks + j][t][i], kLog2e, -m[t]));
                    l[t] += (w[j][0] + w[j][1]) + (w[j][2] + w[j][3]);
                }
                pf[ks][t] = split8(w[0], w[1]);
            }
        }
        if (BUFS == 2) {
            at ^= TILE;
            if (kt0 + G < n_tiles) store(at);
            if (kt0 + 2 * G < n_tiles) fetch(key0 + 2 * G * 64);
        }
        if (seen) values(kt_ + KB);
    }
    if (G == 2) {
        f32x4 *po = reinterpret_cast<f32x4 *>(lds);                                       // [wave][slot][NV][lane]
        float2 *pm = reinterpret_cast<float2 *>(lds + (size_t)4 * SLOTS * NV * 64 * 16);  // [wave][slot][lane]
        __syncthreads();
        if (grp == 1) {
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) {
#pragma unroll
                for (int v = 0; v < NV; ++v) po[((wave * SLOTS + t) * NV + v) * 64 + lane] = o[v][t];
                pm[(wave * SLOTS + t) * 64 + lane] = float2{m[t], l[t]};
            }
        }
        __syncthreads();
        if (grp == 1) return;
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            const float2 b = pm[(wave * SLOTS + t) * 64 + lane];
            const float mx = fmaxf(m[t], b.x), wa = __builtin_amdgcn_exp2f(m[t] - mx), wb = __builtin_amdgcn_exp2f(b.x - mx);
            m[t] = mx, l[t] = l[t] * wa + b.y * wb;
#pragma unroll
            for (int v = 0; v < NV; ++v) o[v][t] = o[v][t] * wa + po[((wave * SLOTS + t) * NV + v) * 64 + lane] * wb;
        }
    }
    if (records) {
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            const int qi = qw + t / MAPS * 16 + r16;
            const float sum = rows_sum(l[t]);
            if (qi >= nq) continue;
            float *rec = records + ((((size_t)qi * heads + h) * MAPS + t % MAPS) * gridDim.y + blockIdx.y) * (kGqaRecHead + vdimp);
            if (g == 0) rec[0] = m[t], rec[1] = sum;
#pragma unroll
            for (int v = 0; v < NV; ++v)
                if (v * 16 < vdimp) *reinterpret_cast<f32x4 *>(rec + kGqaRecHead + v * 16 + g * 4) = o[v][t];
        }
        return;
    }
    float inv[SLOTS], gate[SLOTS / MAPS];
#pragma unroll
    for (int t = 0; t < SLOTS / MAPS; ++t) gate[t] = 1.0f;
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) inv[t] = 1.0f / rows_sum(l[t]);
    if (p.gate && !(FAR && p.gate_columns))
#pragma unroll
        for (int t = 0; t < SLOTS / MAPS; ++t) gate[t] = activate(gate_logit(p, min(qw + t * 16 + r16, nq - 1), h, 0), BITNET_HIP_ACT_SIGMOID);
    if (MAPS == 2) {
        float ss = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            o[v][0] = o[v][0] * inv[0] - (p.lambda * inv[1]) * o[v][1];
            ss += (o[v][0].x * o[v][0].x + o[v][0].y * o[v][0].y) + (o[v][0].z * o[v][0].z + o[v][0].w * o[v][0].w);
        }
        inv[0] = p.out_scale / sqrtf(rows_sum(ss) / (float)p.vdim + p.eps);
    }
#pragma unroll
    for (int t = 0; t < SLOTS / MAPS; ++t) {
        const int qi = qw + t * 16 + r16;
        if (qi >= nq) continue;
        uint16_t *dst = out + (size_t)qi * ldo + (size_t)h * vdimp + g * 4;
#pragma unroll
        for (int v = 0; v < NV; ++v)
            if (v * 16 < vdimp) {
                f32x4 q = o[v][t] * (inv[t] * gate[t]);
                if (FAR && p.gate_columns) {
                    float z[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) z[i] = gate_logit(p, qi, h, v * 16 + g * 4 + i);
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[i] *= __builtin_amdgcn_rcpf(1.0f + __expf(-z[i]));
                }
                *reinterpret_cast<bf16x4 *>(dst + v * 16) = bf16x4{(__bf16)q.x, (__bf16)q.y, (__bf16)q.z, (__bf16)q.w};
            }
    }
}

thread_local int g_last_gqa_groups;

// Two groups fill a CU, and halve its walks; of one group two workgroups fit.  They pay while the launch is as long as its longest walk: with four tiles or more in it, a CU's
// share of all tiles not much above it, and no second round behind walks that are all long (the shortest walk of the first round and the longest of the second one in turn).
// Heads count as a multiple of eight, as the launch deals them to the XCDs (20 heads take what 24 do).  us with two / with one: 24 heads, 2600 tokens
// 80 / 90 (share / walk 1.05), 32 heads, 2048 63 / 75 (1.06), 40 heads, 1664 63 / 62 (1.09), 24 heads, 3000 105 / 105 (1.19), 3328 124 / 121 (1.27), 4096 173 / 153 (1.55); two maps,
// 24 heads, 1280 39 / 44, 1531 57 / 53, 2048 88 / 75; five tiles 13.1 / 13.9, four 13.0 / 12.4.
static bool two_groups(const Gqa &g, int rows, int n_ctx, int nq) {
    const int at_once = 256, pos0 = n_ctx - nq, heads = ((int)g.heads + 7) / 8 * 8, blocks = (nq + rows - 1) / rows, all_tiles = (n_ctx + 63) / 64;
    long longest = 0, total = 0, second = 0;
    for (int qb = blocks - 1, done = 0; qb >= 0 && total <= 2l * at_once * all_tiles; --qb, done += heads) {
        const int q0 = qb * rows, tiles = (std::min(n_ctx, pos0 + q0 + rows) + 63) / 64 - (gqa_first(g, pos0 + q0) >> 6);
        longest = std::max<long>(longest, tiles), total += (long)heads * tiles;
        for (int i : {at_once - 1, at_once})
            if ((long)heads * blocks > at_once && done <= i && i < done + heads) second += tiles;
    }
    return longest >= 4 && 16 * total <= 17 * at_once * longest && 10 * second <= 11 * longest;
}

// The records of a query's head (gridDim.y of the launch above, one behind the other for every map) -> its output: a wave each, vdimp / 4 lanes of four columns, as many groups of them as fit a wave
// sharing the records.
template <int MAPS>
__global__ __launch_bounds__(256) void k_gqa_merge_parts(Gqa p, const float *records, int parts, int nq, uint16_t *out, size_t ldo) {
    const int lane = threadIdx.x & 63, at = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), heads = (int)p.heads, vdimp = (int)p.vdimp;
    if (at >= nq * heads) return;
    const int qi = at / heads, h = at - qi * heads, lanes = vdimp >> 2, groups = 64 / lanes, grp = lane / lanes, c = (lane - grp * lanes) * 4;
    const size_t stride = kGqaRecHead + vdimp;
    const float *rec = records + (size_t)at * MAPS * parts * stride;
    f32x4 v[MAPS], z = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.gate)
#pragma unroll
        for (int e = 0; e < 4; ++e) z[e] = gate_logit(p, qi, h, c + e);
    const float sink = p.sink ? p.sink[h] * kLog2e : -1e30f;
#pragma unroll
    for (int j = 0; j < MAPS; ++j) {
        const float *r = rec + (size_t)j * parts * stride;
        const float m = lane < parts ? r[lane * stride] : -1e30f, l = lane < parts ? r[lane * stride + 1] : 0.f;
        const float M = fmaxf(sink, rows_max(row_max(m))), w = __builtin_amdgcn_exp2f(m - M);
        v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int i0 = 0; i0 < parts; i0 += groups) {  // (all lanes take part; past the last record the weight is zero)
            const int i = i0 + grp;
            v[j] += __shfl(w, min(i, 63), 64) * *reinterpret_cast<const f32x4 *>(r + min(i, parts - 1) * stride + kGqaRecHead + c);
        }
        f32x4 t = v[j];
        const float den = wave_sum(w * l) + (p.sink ? __builtin_amdgcn_exp2f(sink - M) : 0.f);
        for (int o = 1; o < groups; ++o)
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] += __shfl(v[j][e], lane + o * lanes, 64);
        v[j] = t * (1.0f / den);
    }
    f32x4 q = v[0];
    if (MAPS == 2) {
        q -= p.lambda * v[MAPS - 1];
        q *= p.out_scale / sqrtf(wave_sum(grp == 0 ? (q.x * q.x + q.y * q.y) + (q.z * q.z + q.w * q.w) : 0.f) / (float)p.vdim + p.eps);
    }
    if (p.gate)
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] *= activate(z[e], BITNET_HIP_ACT_SIGMOID);
    if (grp == 0) *reinterpret_cast<bf16x4 *>(out + (size_t)qi * ldo + (size_t)h * vdimp + c) = bf16x4{(__bf16)q.x, (__bf16)q.y, (__bf16)q.z, (__bf16)q.w};
}

// Few queries behind many keys: a launch whose blocks leave CUs without a workgroup lasts as long as its longest walk, so a block's tiles are cut into stretches, of two tiles (a step of two
// groups) at least and no more of them than there are CUs for (heads count as a multiple of eight, as the launch deals them to the XCDs: 12 heads in 21 stretches take 32 us where 15 take 24).
// A step of a walk that is saved is worth 2.7 us (7 of one group); the launch that puts the records together costs 5 and 0.7 ns for each query's head, 1.4 for each of a head's two maps.
// us without / with, heads, keys, queries: 12, 2090, 90 51 / 18; 24, 2090, 90 52 / 22; 12, 600, 20 18.3 / 11.1; 12, 1000, 200 28.7 / 18.9; 12, 450, 130 17.7 / 14.5; 12, 8000, 30 168 / 27;
// 24 of two maps, 2090, 90 49 / 28; 2 of 256 columns, 2000, 50 131 / 22; 8, 2000, 2000 50 / 40.  What stays whole: 12, 400, 400 15.9 / 18.1; 16, 512, 512 18.6 / 21.2; 24 of two maps,
// 600, 100 18.3 / 20.6; 12, 100, 3 8.4.
static int gqa_prefill_parts(const Gqa &g, int n_ctx, int nq) {
    const int rows = g.maps == 2 ? 64 : 128, blocks = (nq + rows - 1) / rows, heads = ((int)g.heads + 7) / 8 * 8;
    const int tiles = (n_ctx + 63) / 64 - (gqa_first(g, n_ctx - nq + (blocks - 1) * rows) >> 6), most = std::min<long>(256 / ((long)heads * blocks), 32);
    if (most < 2) return 1;
    const int each = ((tiles + most - 1) / most + 1) & ~1, saved = (tiles + 1) / 2 - each / 2;
    return 2.7 * saved > 5.0 + (g.maps == 2 ? 1.4e-3 : 7e-4) * (double)nq * (double)(g.heads * g.maps) ? (tiles + each - 1) / each : 1;
}
size_t gqa_prefill_floats(const Gqa &g, int n_ctx, int nq) {
    const int parts = gqa_prefill_parts(g, n_ctx, nq);
    return parts > 1 ? (size_t)nq * g.heads * g.maps * parts * (kGqaRecHead + g.vdimp) : 0;
}

template <int NK, int NV, int G>
static hipError_t gqa_prefill_go(const Gqa &g, const uint16_t *q, size_t ldq, int n_ctx, int nq, uint16_t *out, size_t ldo, float *records, hipStream_t s) {
    const int rows = g.maps == 2 ? 64 : 128, n_qb = (nq + rows - 1) / rows, parts = records ? gqa_prefill_parts(g, n_ctx, nq) : 1;
    if constexpr (G == 2)
        if (parts == 1 && !two_groups(g, rows, n_ctx, nq)) return gqa_prefill_go<NK, NV, 1>(g, q, ldq, n_ctx, nq, out, ldo, nullptr, s);
    g_last_gqa_groups = G;
    const size_t tiles = (size_t)G * prefill_buffers(NK, NV, (int)g.maps) * ((size_t)g.maps * 64 * (NK * 64 + 32) + (size_t)NV * 16 * (64 * 2 + 32)), sums = G == 2 ? (size_t)4 * 2 * 64 * (NV * 16 + 8) : 0;
    const size_t lds = tiles > sums ? tiles : sums;
    auto fn = g.maps == 2 ? k_gqa_prefill<NK, NV, 2, false, G> : g.far_weight || g.gate_columns ? k_gqa_prefill<NK, NV, 1, true, G> : k_gqa_prefill<NK, NV, 1, false, G>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(8 * ((g.heads + 7) / 8) * n_qb, parts), dim3(256 * G), lds, s, g, q, ldq, n_ctx, nq, out, ldo, n_qb, parts > 1 ? records : nullptr);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || parts == 1) return e;
    hipLaunchKernelGGL(g.maps == 2 ? k_gqa_merge_parts<2> : k_gqa_merge_parts<1>, dim3((nq * (int)g.heads + 3) / 4), dim3(256), 0, s, g, records, parts, nq, out, ldo);
    return hipGetLastError();
}

// records: gqa_prefill_floats(g, n_ctx, nq) of them, or none where a block's keys stay together
hipError_t launch_gqa_prefill(const Gqa &g, const uint16_t *q, size_t ldq, int n_ctx, int nq, uint16_t *out, size_t ldo, float *records, hipStream_t s) {
    if (!gqa_supported((int)g.dimp, (int)g.vdimp)) return hipErrorInvalidValue;
    if (g.dimp <= 64 && g.vdimp <= 64) return gqa_prefill_go<2, 4, 2>(g, q, ldq, n_ctx, nq, out, ldo, records, s);
    if (g.dimp <= 64 && g.vdimp <= 128) return gqa_prefill_go<2, 8, 2>(g, q, ldq, n_ctx, nq, out, ldo, records, s);
    if (g.dimp <= 128 && g.vdimp <= 128) return gqa_prefill_go<4, 8, 2>(g, q, ldq, n_ctx, nq, out, ldo, records, s);
    return gqa_prefill_go<8, 16, 1>(g, q, ldq, n_ctx, nq, out, ldo, records, s);
}

}  // namespace bitnet_hip
