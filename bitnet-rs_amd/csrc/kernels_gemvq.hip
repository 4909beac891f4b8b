// kernels_gemvq.hip -- the I2_S / QK256 GEMV of the decode step on PRE-QUANTISED activations (qact.hpp).
//
// Same matrix-core formulation as k_gemv_mfma (kernels_mfma.hip: the vector ALUs only expand 2-bit codes to int8,
// v_mfma_i32_16x16x64_i8 does every multiply-add), with the three fixed costs round 1's profile charged to every
// wave removed (~650 VALU instructions per wave, 218 of them quantising activations,
// 120 LayerNorm statistics; 176 KB of loads per workgroup through a 64 B/clk vector-memory path):
//
//  * activations arrive as int8 digit planes + one power-of-two scale per 16 elements, written by the PRODUCING
//    kernel's epilogue (the previous GEMV, the attention combine, the embedding gather).  A wave copies its K range
//    (576 B per 256 columns) into LDS with two or three flat 16-byte loads -- no conversion, no row maximum;
//  * LayerNorm (applied after the product, bitnet_hip_weights_bind_ln) takes its row statistics from one
//    (sum, sum of squares) pair per producer tile instead of re-reading the row in every wave;
//  * the MFMA operands are swapped: the WEIGHTS are the B operand (16 output rows = the 16 columns of D), the
//    activations the A operand, whose 16 rows are (k-group kg, digit d, block half h) selectors -- row 4 kg + 2 d + h
//    holds digit plane d for the lanes of k-group kg in the MFMAs of parity h and zeros elsewhere.  One lane of D
//    then holds, for ONE weight row and ONE 32-weight block, the four exact integer sums (d, h) in its four
//    accumulator registers: digits recombine in integer arithmetic (v_lshl_add_u32), and the 32-block's weight scale
//    is applied once per lane: 7 VALU instructions per 32-block and lane instead of 12, one f16 scale load per
//    (row, block) instead of four.
//
// Per 1-KiB weight tile (16 rows x 256 columns) a wave issues 4 MFMAs, 44 VALU for the code expansion, 14 for
// digits + scales, 5 LDS reads.  Numerics: every 16-element partial sum is an exact integer; the activation is
// held to 2^-15 of its 16-group's maximum (qact.hpp); f32 accumulation in a fixed order (bit-reproducible).
// Reference semantics: Q/i2s_qk256.rs:196-274 (QK256), K/cpu/quantized_matmul.rs:57-96 (ternary x block scale),
// T:67-100 (LayerNorm), T:756-781 (silu(gate) * up), T:1073 / T:1125 (residual).
#include <cstdlib>

#include "common.hpp"
#include "qact.hpp"

namespace bitnet_hip {

namespace {

constexpr int kMaxGroupQ = 4;  // query heads per KV head in an attention chunk record (kAttnRecFloats = 2 * 4 + 4 * 128)
typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t umin32q(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ v4u ldq_nt16(const void *p) { return __builtin_nontemporal_load(reinterpret_cast<const v4u *>(p)); }
__device__ __forceinline__ v4i decode16q(uint32_t w, uint32_t lut) {
    v4i a;
    a[0] = (int)__builtin_amdgcn_perm(0u, lut, w & 0x03030303u);
    a[1] = (int)__builtin_amdgcn_perm(0u, lut, (w >> 2) & 0x03030303u);
    a[2] = (int)__builtin_amdgcn_perm(0u, lut, (w >> 4) & 0x03030303u);
    a[3] = (int)__builtin_amdgcn_perm(0u, lut, (w >> 6) & 0x03030303u);
    return a;
}
__device__ __forceinline__ float fmix_lo(float a, uint32_t h, float c) {  // a * f16(h.lo) + c
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(a), "v"(h), "v"(c));
    return r;
}
__device__ __forceinline__ float fmix_hi(float a, uint32_t h, float c) {  // a * f16(h.hi) + c
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(a), "v"(h), "v"(c));
    return r;
}
template <int CTRL>
__device__ __forceinline__ double wdpp_d(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double wave_sum_dq(double v) {
    v += wdpp_d<0xB1>(v);
    v += wdpp_d<0x4E>(v);
    v += wdpp_d<0x141>(v);
    v += wdpp_d<0x140>(v);
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    double r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, 16 * i);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), 16 * i);
        r[i] = __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
    }
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// In-kernel time stamps (s_memrealtime, 100 MHz): diagnostic build only (-DBH_STAMPS), 16 x u64 per workgroup.
#ifdef BH_STAMPS
#define BH_QSTAMP(i)                                                                                           \
    do {                                                                                                       \
        if (p.stamps && lane == 0 && (wave == 0 || wave == NW - 1))                                            \
            p.stamps[(size_t)blockIdx.x * 16 + (wave ? 8 : 0) + (i)] = __builtin_amdgcn_s_memrealtime();      \
    } while (0)
#else
#define BH_QSTAMP(i) \
    do {             \
    } while (0)
#endif

struct GemvQArgs {
    const uint8_t *tiles;    // [n_tiles][nblk][64 lanes][16 B] code tiles (k_retile)
    const void *stiles;      // [n_tiles][nblk][64 lanes] x {f16 x 2 | f32 x 2}: 32-block scales (k_retile_scales[_h]) or null
    int rows, cols, nblk;
    uint32_t lut;
    int ks_log2;             // K ranges per row tile = waves sharing a tile
    const uint8_t *qin;      // QAct records [nblk][576]
    const double *stats_in;  // LN: (sum, sum of squares) per 16 columns
    int n_stats;
    const float *ln_g;       // LN: g_r = W[r,:] . gamma (bitnet_hip_weights_bind_ln)
    float ln_eps;
    double inv_cols;
    const float *residual;   // optional: v = residual + W x
    float *y;                // optional f32 output
    int silu_mul;            // rows are (gate tile, up tile) pairs: v = silu(gate) * up
    uint8_t *qout;           // optional QAct output (for the next GEMV)
    const float *gamma_out;  // optional: the next GEMV's LayerNorm weight (u = v * gamma)
    double *stats_out;       // optional: (sum, sum of squares) per 16 output rows
    // MRG: the activation vector is the decode attention's output, assembled HERE from its per-chunk records
    // (launch_attn_decode(..., combine = false): (m, l)[4] + un-normalised P.V [4][128] per KV head and 64-position chunk)
    const float *attn_rec;
    const int *attn_pos;     // *attn_pos + 1 keys
    int attn_chunks_max, attn_group_log2, attn_chunk_log2;  // records per KV head, log2 heads per KV head, log2 positions per record (6 / 7)
    unsigned long long *stamps;  // diagnostic builds only
};

// NW waves per workgroup; RING = 256-column blocks per wave, all in flight at once; SC = weight scales per 32-block:
// 0 none (QK256), 1 f32, 2 f16; LN = LayerNorm after the product; NCP = 8-KiB passes of the cooperative QAct copy.
//
// Where a launch's time goes (in-kernel stamps, tools/stamp_gemvq.py, 2B-4T shapes): a CU's vector-memory path takes
// 64 B of requests per clock, so WHAT A WORKGROUP ASKS FOR is its start-up time -- with every wave fetching its own K
// range of the activations and its own copy of the statistics the last wave's weight loads were only requested 1.1 us
// after the kernel began (99 KB per workgroup, half of it duplicates).  Hence: the workgroup copies the activation
// vector into LDS ONCE (each thread 16 B), the statistics pairs likewise, and the per-row operands of the epilogue
// (g_r, residual, the next LayerNorm's gamma) are requested up front too -- behind the barrier they were dependent
// L2 / HBM round trips (0.7-0.8 us of a 2.5 us kernel).
// Every global load is unconditional and sits ahead of a scheduling fence (kernels_mfma.hip explains why).
// MRG = NE > 0: short contexts (<= 4 chunk records): instead of copying QAct records the workgroup merges the attention's
// chunk records itself -- thread t the elements t, t + NT, ... (NE of them) of the attention output: softmax merge of up to
// 4 records, then the 16-lane group quantisation of qact.hpp straight into the LDS image.  One launch (k_attn_combine) and
// one global round trip of the vector less per layer; every workgroup reads every live record (n_chunks x 10 KB), which
// is why the decoder takes this form up to 256 keys only.
template <int NW, int RING, int SC, int LN, int NCP, int NE = 0>
__global__ __launch_bounds__(NW * 64) void k_gemv_q(GemvQArgs p) {
    constexpr int NT = NW * 64;
    constexpr bool MRG = NE > 0;
    constexpr int ZB = RING * kQRec;  // zero bytes the dead A lanes read (no masking instructions)
    // every kernel argument in ONE scalar-load round: left alone hipcc fetches some of them where they are first used,
    // each a dependent round trip on the path to the first vector load
    asm volatile("" ::"s"(p.tiles), "s"(p.stiles), "s"(p.rows), "s"(p.nblk), "s"(p.lut), "s"(p.ks_log2), "s"(p.qin), "s"(p.stats_in), "s"(p.n_stats),
                 "s"(p.ln_g), "s"(p.residual), "s"(p.y), "s"(p.silu_mul), "s"(p.qout), "s"(p.gamma_out), "s"(p.stats_out));
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *zq = lds;                                // [ZB]
    uint8_t *cq = lds + ZB;                           // [NCP * 16 * NT] the whole QAct vector (padded)
    uint8_t *cs = cq + NCP * 16 * NT;                 // [NT * 16] statistics pairs (LN)
    float *part = reinterpret_cast<float *>(cs + (LN ? NT * 16 : 0));  // [NW][16] partial sums by (tile, K part)
    BH_QSTAMP(0);
    if (16 * tid < ZB) *reinterpret_cast<v4u *>(zq + 16 * tid) = v4u{0u, 0u, 0u, 0u};

    // ---- wave -> (row tile, K range of at most RING blocks), as k_gemv_mfma ------------------------------------
    const int ksplit = 1 << p.ks_log2;
    const int tiles_per_wg = NW >> p.ks_log2;
    const int n_tiles = p.rows >> 4;  // rows % 16 == 0 (launcher)
    int tile = blockIdx.x * tiles_per_wg + (wave >> p.ks_log2);
    tile = tile < n_tiles ? tile : n_tiles - 1;  // surplus waves redo the last tile; never stored
    int kpart = wave & (ksplit - 1);
    if (NW == 8 && p.ks_log2 == 3 && wave >= 4) kpart = 11 - wave;  // at most one long range per SIMD (kernels_mfma.hip)
    const int b0 = (kpart * p.nblk) >> p.ks_log2, b1 = ((kpart + 1) * p.nblk) >> p.ks_log2;

    // ---- 1. the activation vector (L2-resident, every workgroup reads it), statistics pairs, epilogue operands ----
    const uint32_t q_last = (uint32_t)kQRec * (uint32_t)p.nblk - 16u;
    v4u qa[NCP];  // native vectors: arrays of HIP's uint4 struct went through scratch memory at the scheduling fence
    float4 mo[MRG ? NE : 1][4];   // MRG: un-normalised P.V values of this thread's NE 4-element slots, chunks 0..3
    float2 mml[MRG ? NE : 1][4];  //      and their heads' (m, l)
    if (!MRG) {
#pragma unroll
        for (int i = 0; i < NCP; ++i) qa[i] = *reinterpret_cast<const v4u *>(p.qin + umin32q(16u * (uint32_t)(tid + NT * i), q_last));
    } else {
        // chunks 0..3 are requested before the position (hence the live chunk count) is known; dead records hold zeros or
        // an earlier token's finite values: only their m is masked below.  A thread takes 4 consecutive elements (one
        // 16-byte load per chunk); a wave's 256 elements lie in at most two heads, whose (m, l) pairs every lane fetches.
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            int e = 4 * (tid + NT * i);
            // (a whole wave past the columns asks for nothing and merges nothing: at 2560 of them that is the second slot of six of eight waves, us per launch at 129 to 192 keys 5.3 -> 5.0; ten waves
            // with a slot each give another 0.1)
            if (i > 0 && 4 * (wave * 64 + NT * i) >= p.cols) break;
            e = e < p.cols ? e : p.cols - 4;
            const int h = e >> 7, d = e & 127, kvh = h >> p.attn_group_log2, hg = h & ((1 << p.attn_group_log2) - 1);
            const float *rb = p.attn_rec + (size_t)kvh * p.attn_chunks_max * kAttnRecFloats;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float *rec = rb + (size_t)(c < p.attn_chunks_max ? c : p.attn_chunks_max - 1) * kAttnRecFloats;
                mml[i][c] = *reinterpret_cast<const float2 *>(rec + 2 * hg);
                mo[i][c] = *reinterpret_cast<const float4 *>(rec + 2 * kMaxGroupQ + hg * 128 + d);
            }
        }
    }
    v4u st = {0u, 0u, 0u, 0u};
    if (LN) st = *reinterpret_cast<const v4u *>(p.stats_in + 2 * (size_t)(tid < p.n_stats ? tid : p.n_stats - 1));
    // the storing thread's row(s); other threads request clamped, valid addresses and drop the values
    const int e_tl = tid >> 4, e_r = tid & 15;
    int e_row, e_g0 = 0, e_g1 = 0;
    if (!p.silu_mul) {
        e_row = 16 * (blockIdx.x * tiles_per_wg + e_tl) + e_r;
        e_row = e_row < p.rows ? e_row : p.rows - 1;
        e_g0 = e_row;
    } else {
        const int half_rows = p.rows >> 1;
        const int pg = blockIdx.x * (tiles_per_wg >> 1) + e_tl;
        e_row = 16 * pg + e_r;
        e_row = e_row < half_rows ? e_row : half_rows - 1;
        e_g0 = 32 * (e_row >> 4) + e_r;
        e_g1 = e_g0 + 16;
    }
    float e_lg0 = 0.0f, e_lg1 = 0.0f;
    if (LN) {
        e_lg0 = p.ln_g[e_g0];
        e_lg1 = p.ln_g[e_g1];
    }
    // nullable operands: a valid dummy address instead of a branch around the load (a load under a branch costs a full wait)
    const float e_res = (p.residual ? p.residual : reinterpret_cast<const float *>(p.qin))[p.residual ? e_row : 0];
    const float e_gam = (p.gamma_out ? p.gamma_out : reinterpret_cast<const float *>(p.qin))[p.gamma_out ? e_row : 0];
    // vmcnt retires in order: the activations must be REQUESTED ahead of the weight stream, or their arrival only
    // counts once every weight tile has landed
    __builtin_amdgcn_sched_barrier(0);
    // ---- 2. weight tiles (+ their scale tiles): read once by this wave only -> non-temporal -------------------
    const size_t tb0 = (size_t)tile * p.nblk;
    const uint8_t *wbase = p.tiles + (tb0 * 64 + lane) * 16;
    v4u wt[RING];
    uint32_t sh[SC == 2 ? RING : 1];
    float2 sf[SC == 1 ? RING : 1];
#pragma unroll
    for (int j = 0; j < RING; ++j) {
        const int blk = b0 + j < b1 ? b0 + j : b1 - 1;  // clamped: a short range re-reads its last tile
        wt[j] = ldq_nt16(wbase + (size_t)blk * 1024);
        if (SC == 2) sh[j] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(p.stiles) + (tb0 + blk) * 64 + lane);
        if (SC == 1) {
            const float *sp = reinterpret_cast<const float *>(p.stiles) + ((tb0 + blk) * 64 + lane) * 2;
            sf[j] = float2{__builtin_nontemporal_load(sp), __builtin_nontemporal_load(sp + 1)};
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of this wave is requested before anything waits
    BH_QSTAMP(1);

    // ---- 3. QAct records (and statistics pairs) -> LDS, once per workgroup ------------------------------------
    if (!MRG) {
#pragma unroll
        for (int i = 0; i < NCP; ++i) *reinterpret_cast<v4u *>(cq + 16 * (tid + NT * i)) = qa[i];
    } else {
        const int m_chunks = (*p.attn_pos + (1 << p.attn_chunk_log2)) >> p.attn_chunk_log2;  // live records, 1..4 (the caller switches to the combine kernel beyond that)
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int e = 4 * (tid + NT * i);
            if (i > 0 && 4 * (wave * 64 + NT * i) >= p.cols) break;
            // softmax merge: out = sum_c e^(m_c - M) o_c / sum_c e^(m_c - M) l_c   (k_attn_combine's value)
            float M = -INFINITY;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                mml[i][c].x = c < m_chunks ? mml[i][c].x : -INFINITY;
                M = fmaxf(M, mml[i][c].x);
            }
            float L = 0.0f;
            float4 a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float w = __expf(mml[i][c].x - M);
                L += w * mml[i][c].y;
                a.x += w * mo[i][c].x, a.y += w * mo[i][c].y, a.z += w * mo[i][c].z, a.w += w * mo[i][c].w;
            }
            const float rl = e < p.cols ? 1.0f / L : 0.0f;
            const float v[4] = {a.x * rl, a.y * rl, a.z * rl, a.w * rl};
            // qact_emit's arithmetic (qact.hpp) with the 16-element group spread over 4 lanes x 4 elements; destination = the
            // LDS image instead of a global record
            uint32_t u = __float_as_uint(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])))), o;
            o = qdpp_u<0xB1>(u), u = o > u ? o : u;  // quad_perm [1,0,3,2]
            o = qdpp_u<0x4E>(u), u = o > u ? o : u;  // quad_perm [2,3,0,1]: the maximum over the quad = the 16 elements
            int be = (int)(u >> 23);
            be = be < 32 ? 32 : be;
            be = be > 254 ? 254 : be;
            const float sc = __uint_as_float((uint32_t)(267 - be) << 23), as = __uint_as_float((uint32_t)(be - 13) << 23);
            uint32_t d0 = 0, d1 = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t t = ((uint32_t)qcvt_rpi(v[j] * sc) + 0x80u) ^ 0x80u;
                d0 |= (t & 0xffu) << (8 * j);
                d1 |= ((t >> 8) & 0xffu) << (8 * j);
            }
            if (e < p.cols) {
                const int grp = e >> 4, rec = grp >> 4, tp = grp & 15;
                uint8_t *qb = cq + kQRec * rec;
                *reinterpret_cast<uint32_t *>(qb + 16 * tp + (e & 15)) = d0;
                *reinterpret_cast<uint32_t *>(qb + 256 + 16 * tp + (e & 15)) = d1;
                if ((e & 15) == 0) reinterpret_cast<float *>(qb + 512)[4 * (tp >> 2) + 2 * (tp & 1) + ((tp & 3) >> 1)] = as;
            }
        }
    }
    if (LN) *reinterpret_cast<v4u *>(cs + 16 * tid) = st;
    // raw barrier: __syncthreads() would also wait for the weight loads in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // A-operand lane (k-group g, selector row c = 4 kg + 2 d + h): digit plane d of k-group kg, live in the MFMAs
    // of parity h only; every other (lane, MFMA) reads zeros.  D lane (g, c): selector group g, weight row c.
    const int g = lane >> 4, c = lane & 15;
    const bool mine = (c >> 2) == g;
    const uint8_t *wq = cq + kQRec * b0;  // this wave's K range
    const uint8_t *live = wq + 256 * ((c >> 1) & 1) + 64 * g;
    const uint8_t *ba0 = (mine && (c & 1) == 0) ? live : zq;  // MFMAs 0 and 2 of a block
    const uint8_t *ba1 = (mine && (c & 1) == 1) ? live : zq;  // MFMAs 1 and 3
    const uint8_t *sa = wq + 512 + 16 * g;                    // this lane's four group scales of a record
    BH_QSTAMP(2);

    float facc = 0.0f;
#pragma unroll
    for (int j = 0; j < RING; ++j) {
        if (j > 0 && b0 + j >= b1) continue;  // wave-uniform: a slot past this wave's range
        const float4 as = *reinterpret_cast<const float4 *>(sa + kQRec * j);  // (h0 p0, h0 p1, h1 p0, h1 p1)
        const uint32_t wd[4] = {wt[j][0], wt[j][1], wt[j][2], wt[j][3]};
#pragma unroll
        for (int pp = 0; pp < 2; ++pp) {  // the lane group's two 32-weight blocks
            v4i acc = {0, 0, 0, 0};
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i *>(ba0 + kQRec * j + 32 * pp),
                                                        decode16q(wd[2 * pp], p.lut), acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i *>(ba1 + kQRec * j + 32 * pp + 16),
                                                        decode16q(wd[2 * pp + 1], p.lut), acc, 0, 0, 0);
            // acc[2 d + h]: exact sums over the 16 weights of half h with digit plane d; |.| <= 16 * 2 * 128
            const int i0 = (int)(((uint32_t)acc[2] << 8) + (uint32_t)acc[0]), i1 = (int)(((uint32_t)acc[3] << 8) + (uint32_t)acc[1]);
            float t = (float)i0 * (pp ? as.y : as.x);
            t = fmaf((float)i1, pp ? as.w : as.z, t);
            if (SC == 2)
                facc = pp ? fmix_hi(t, sh[j], facc) : fmix_lo(t, sh[j], facc);
            else if (SC == 1)
                facc = fmaf(t, pp ? sf[j].y : sf[j].x, facc);
            else
                facc += t;
        }
    }
    // the four k-groups of a weight row sit in lanes c, c + 16, c + 32, c + 48: two lane swaps (v_permlane16_swap,
    // v_permlane32_swap) add them up in every wave at once -- (g0 + g1) + (g2 + g3) -- instead of 4 LDS reads per K part
    // in the one storing wave
    {
        // inline asm with the hazard pad inside (a VALU write needs 2 wait states before v_permlane*_swap reads it):
        // hipcc's __builtin_amdgcn_permlane16_swap folded the two results into one register here (ROCm 7.2)
        float a = facc, b = facc;
        asm volatile("v_nop\n\tv_nop\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
        facc = a + b;  // rows (g0 + g1, g0 + g1, g2 + g3, g2 + g3)
        a = facc, b = facc;
        asm volatile("v_nop\n\tv_nop\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
        facc = a + b;
    }
    if (lane < 16) part[(((wave >> p.ks_log2) << p.ks_log2) + kpart) * 16 + lane] = facc;
    BH_QSTAMP(3);

    // ---- 4. epilogue: the storing waves only ------------------------------------------------------------------
    const bool storing = wave * 64 < tiles_per_wg * 16;
    double ln_mean = 0.0, ln_rdenom = 1.0;
    if (LN && storing) {
        double s1 = 0.0, s2 = 0.0;
        for (int i = lane; i < p.n_stats; i += 64) {
            const double2 pr = *reinterpret_cast<const double2 *>(cs + 16 * i);
            s1 += pr.x;
            s2 += pr.y;
        }
        s1 = wave_sum_dq(s1);
        s2 = wave_sum_dq(s2);
        const double mean_d = s1 * p.inv_cols;
        const double var_d = s2 * p.inv_cols - mean_d * mean_d;
        ln_mean = (double)(float)mean_d;  // the f32 mean the reference subtracts
        const double denom = (double)sqrtf((float)(var_d > 0.0 ? var_d : 0.0) + p.ln_eps);
        double r = __builtin_amdgcn_rcp(denom);
        r = r * (2.0 - denom * r);
        ln_rdenom = r * (2.0 - denom * r);
    }
    __syncthreads();
    BH_QSTAMP(4);
    if (!storing) return;
    const int tl = e_tl, r = e_r;
    if (!p.silu_mul) {
        if (tl >= tiles_per_wg) return;
        const int t_glob = blockIdx.x * tiles_per_wg + tl;
        if (t_glob >= n_tiles) return;  // whole 16-lane rows leave together
        const int row = 16 * t_glob + r;
        float pv[NW];
#pragma unroll
        for (int kp = 0; kp < NW; ++kp) pv[kp] = part[((tl << p.ks_log2) + (kp < ksplit ? kp : 0)) * 16 + r];  // all reads in flight at once
        float v = 0.0f;
#pragma unroll
        for (int kp = 0; kp < NW; ++kp) v += kp < ksplit ? pv[kp] : 0.0f;  // fixed order: K parts 0, 1, ...
        if (LN) v = (float)(((double)v - ln_mean * (double)e_lg0) * ln_rdenom);
        if (p.residual) v += e_res;
        if (p.y) p.y[row] = v;
        if (p.qout) qact_emit(p.qout, p.stats_out, t_glob, r, v, p.gamma_out ? v * e_gam : v);
        BH_QSTAMP(5);
    } else {
        const int pairs_per_wg = tiles_per_wg >> 1;
        if (tl >= pairs_per_wg) return;
        const int p_glob = blockIdx.x * pairs_per_wg + tl;
        if (2 * p_glob >= n_tiles) return;
        const int row = 16 * p_glob + r;  // row of silu(gate) * up
        float pg[NW / 2], pu[NW / 2];  // paired matrices split K over at most NW / 2 waves
#pragma unroll
        for (int kp = 0; kp < NW / 2; ++kp) {
            pg[kp] = part[(((2 * tl) << p.ks_log2) + (kp < ksplit ? kp : 0)) * 16 + r];
            pu[kp] = part[(((2 * tl + 1) << p.ks_log2) + (kp < ksplit ? kp : 0)) * 16 + r];
        }
        float gv = 0.0f, uv = 0.0f;
#pragma unroll
        for (int kp = 0; kp < NW / 2; ++kp) {
            gv += kp < ksplit ? pg[kp] : 0.0f;
            uv += kp < ksplit ? pu[kp] : 0.0f;
        }
        if (LN) {  // stored rows of the paired matrix: (gate tile, up tile)
            gv = (float)(((double)gv - ln_mean * (double)e_lg0) * ln_rdenom);
            uv = (float)(((double)uv - ln_mean * (double)e_lg1) * ln_rdenom);
        }
        // FeedForward::forward T:756-781: silu(g) * u, silu(v) = v / (1 + e^-v); v_exp_f32 / v_rcp_f32 (1 ulp each) instead of the
        // ~40-instruction libm forms: this runs on ONE wave per workgroup, behind the barrier
        const float v = gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)) * uv;
        if (p.y) p.y[row] = v;
        if (p.qout) qact_emit(p.qout, p.stats_out, p_glob, r, v, p.gamma_out ? v * e_gam : v);
        BH_QSTAMP(5);
    }
}

// ---- standalone producers: any f32 vector -> QAct (tests, the first layer's input) ----------------------------
__global__ __launch_bounds__(256) void k_quant_act(const float *__restrict__ x, const float *__restrict__ gamma, int n,
                                                   uint8_t *__restrict__ qout, double *__restrict__ stats) {
    const int i = blockIdx.x * 256 + threadIdx.x;  // n % 16 == 0: whole 16-lane rows are in or out together
    if (i >= n) return;
    const float v = x[i];
    qact_emit(qout, stats, i >> 4, i & 15, v, gamma ? v * gamma[i] : v);
}

// TransformerModel::embed (T:1390-1426) of ONE token + the first block's QAct (its attention_norm gamma)
__global__ __launch_bounds__(256) void k_embed_q(const _Float16 *__restrict__ table, const int *__restrict__ tokens,
                                                 const int *__restrict__ offset_ptr, int hidden, int vocab, float *__restrict__ x_out,
                                                 const float *__restrict__ gamma, uint8_t *__restrict__ qout, double *__restrict__ stats) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= hidden) return;
    int tok = tokens[offset_ptr ? *offset_ptr : 0];
    tok = tok < 0 ? 0 : tok >= vocab ? vocab - 1 : tok;  // ids are range-checked on the host (Decoder::feed); never a wild read
    const float v = (float)table[(size_t)tok * hidden + i];
    x_out[i] = v;
    qact_emit(qout, stats, i >> 4, i & 15, v, gamma ? v * gamma[i] : v);
}

}  // namespace

bool gemvq_supported(const Weights &w) {
    if (!mfma_supported(w)) return false;
    if (w.cols % 256 != 0 || w.rows % 16 != 0) return false;   // whole records, whole producer tiles
    if (w.scaled && w.block_size != 32) return false;          // 256-block scales stay on k_gemv_mfma
    return true;
}

hipError_t launch_quant_act(const float *x, const float *gamma, size_t n, void *qout, double *stats, hipStream_t stream) {
    if (n == 0 || n % 16 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_quant_act, dim3((unsigned)div_ceil(n, 256)), dim3(256), 0, stream, x, gamma, (int)n, static_cast<uint8_t *>(qout), stats);
    return hipGetLastError();
}

hipError_t launch_embed_q(const void *table, const int *tokens, const int *offset_ptr, int hidden, int vocab, float *x_out,
                          const float *gamma, void *qout, double *stats, hipStream_t stream) {
    if (hidden <= 0 || hidden % 16 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_embed_q, dim3((unsigned)div_ceil((size_t)hidden, 256)), dim3(256), 0, stream, static_cast<const _Float16 *>(table), tokens,
                       offset_ptr, hidden, vocab, x_out, gamma, static_cast<uint8_t *>(qout), stats);
    return hipGetLastError();
}

hipError_t launch_gemv_q(const Weights &w, const GemvQIo &io, hipStream_t stream) {
    if (!w.tiles || !gemvq_supported(w) || (!io.qin && !io.attn_rec)) return hipErrorInvalidValue;
    const bool sc_any = w.scaled;
    const int sc = !sc_any ? 0 : w.scales_f16 ? 2 : 1;
    if (sc == 2 && !w.scale_tiles_h) return hipErrorInvalidValue;
    if (sc == 1 && !w.scale_tiles) return hipErrorInvalidValue;
    GemvQArgs a;
    a.tiles = w.tiles;
    a.stiles = sc == 2 ? (const void *)w.scale_tiles_h : sc == 1 ? (const void *)w.scale_tiles : nullptr;
    a.rows = (int)w.rows;
    a.cols = (int)w.cols;
    a.nblk = (int)(w.cols / 256);
    a.lut = w.lut;
    // (16-wave workgroups -- 4 waves per SIMD, half the K range each -- measured slower in round 2, gate|up 5.46 vs 5.23 us, and were removed)
    const int nw = 8;
    const int ksplit = mfma_pick_ksplit(w.rows, w.cols, io.silu_mul, 8);
    a.ks_log2 = ksplit == 8 ? 3 : ksplit == 4 ? 2 : ksplit == 2 ? 1 : 0;
    a.qin = static_cast<const uint8_t *>(io.qin);
    const bool ln = io.ln_gamma != nullptr;
    if (ln && !(w.ln_g && w.ln_gamma_bound == io.ln_gamma && io.stats_in)) return hipErrorInvalidValue;  // LayerNorm only in the after-product form
    a.stats_in = io.stats_in;
    a.n_stats = (int)(w.cols / 16);
    a.ln_g = w.ln_g;
    a.ln_eps = io.ln_eps;
    a.inv_cols = 1.0 / (double)w.cols;
    a.residual = io.residual;
    a.y = io.y;
    a.silu_mul = io.silu_mul ? 1 : 0;
    a.qout = static_cast<uint8_t *>(io.qout);
    a.gamma_out = io.gamma_out;
    a.stats_out = io.stats_out;
    a.attn_rec = io.attn_rec;
    a.attn_pos = io.attn_pos;
    a.attn_chunks_max = io.attn_chunks_max;
    a.attn_group_log2 = io.attn_group_log2;
    a.attn_chunk_log2 = io.attn_chunk_log2;
    a.stamps = g_mfma_stamps;
    if (io.silu_mul && (!w.paired || io.residual)) return hipErrorInvalidValue;
    const int tiles_per_wg = nw / ksplit;
    const unsigned grid = (unsigned)div_ceil(w.rows / 16, (size_t)tiles_per_wg);
    const int ring = (int)div_ceil((size_t)a.nblk, (size_t)ksplit);
    const size_t qbytes = (size_t)kQRec * a.nblk;
    const int ncp = (int)div_ceil(qbytes, (size_t)16 * nw * 64);
    if (ring > 5 || ncp > 3 || (ln && a.n_stats > nw * 64)) return hipErrorInvalidValue;
    void (*kfn)(GemvQArgs) = nullptr;
#define BH_QPICK2(RINGv, NCPv)                                                                                                        \
    if (!kfn && ring <= RINGv && ncp == NCPv)                                                                                         \
        kfn = ln ? (sc == 2 ? k_gemv_q<8, RINGv, 2, 1, NCPv> : sc == 1 ? k_gemv_q<8, RINGv, 1, 1, NCPv> : k_gemv_q<8, RINGv, 0, 1, NCPv>)  \
                 : (sc == 2 ? k_gemv_q<8, RINGv, 2, 0, NCPv> : sc == 1 ? k_gemv_q<8, RINGv, 1, 0, NCPv> : k_gemv_q<8, RINGv, 0, 0, NCPv>);
#define BH_QPICK(RINGv) BH_QPICK2(RINGv, 1) BH_QPICK2(RINGv, 2) BH_QPICK2(RINGv, 3)
    BH_QPICK(2) BH_QPICK(3) BH_QPICK(4) BH_QPICK(5)
#undef BH_QPICK
#undef BH_QPICK2
    if (io.attn_rec) {  // merging form: the o-projection shape (K = heads * 128 <= 4096: 8 elements per thread at most, ring <= 2)
        const int ne = (int)div_ceil(w.cols / 4, (size_t)512);  // 4-element slots per thread
        if (ln || nw != 8 || ring > 2 || ncp != 1 || w.cols % 128 != 0 || ne > 2 || !io.attn_pos || io.attn_chunks_max < 1) return hipErrorInvalidValue;
#define BH_QMRG(NEv)                                                                                                                   \
    if (ne <= NEv && !kfn) kfn = sc == 2 ? k_gemv_q<8, 2, 2, 0, 1, NEv> : sc == 1 ? k_gemv_q<8, 2, 1, 0, 1, NEv> : k_gemv_q<8, 2, 0, 0, 1, NEv>;
        kfn = nullptr;
        BH_QMRG(1) BH_QMRG(2)
#undef BH_QMRG
    }
    if (!kfn) return hipErrorInvalidValue;
    const int ring_t = ring <= 2 ? 2 : ring;
    const size_t lds = (size_t)ring_t * kQRec + (size_t)ncp * 16 * nw * 64 + (ln ? (size_t)nw * 64 * 16 : 0) + (size_t)nw * 16 * sizeof(float);
    hipLaunchKernelGGL(kfn, dim3(grid), dim3(nw * 64), lds, stream, a);
    return hipGetLastError();
}

}  // namespace bitnet_hip
