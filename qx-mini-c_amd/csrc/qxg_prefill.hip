// Batched prefill (CDNA4, gfx950): the T tokens of a prompt chunk go through each
// layer together.  The reference runs a prompt one token at a time through its
// decode step (src/qx_format.c:6250-6547 of the reference); here every projection
// and every expert matrix is one GEMM over the tokens (or over the tokens routed to
// that expert) on the matrix cores.
//
// Precision scheme of the GEMMs (fp16 MFMA, f32 accumulation).  Every weight of the
// formats used is, exactly,
//     IQ2_XS   w = (d/8) * [(2s+1) * grid * sign]        |code| <= 31*43 = 1333
//     IQ3_XXS  w = (d/4) * [(2a+1) * grid * sign]        |code| <= 31*62 = 1922
//     IQ4_XS   w = (d*(ls-32)) * kvalue                  |code| <= 127
// (the f32 products the reference forms, src/qx_format.c:1914-2053, are exact), and
// each bracketed integer code is exact in fp16.  Each activation row is scaled by a
// power of two s (max |x*s| in [2^13, 2^14)) and split as x*s = hi + lo (+ e), hi and
// lo fp16, |e| <= 2^-22 |x*s|.  A code times an fp16 value is exact in f32; the matrix
// cores sum the products in f32 over one block (IQ2_XS, IQ3_XXS: 256 values) or one
// group (IQ4_XS: 32 values), that partial sum is multiplied by its f32 scale once, and
// the row result is divided by s.  The GEMMs are in qxg_pf_dense.hip (Q/K/V, O) and
// qxg_pf_experts.hip; here are the stages between them.
#include "qxg_pf.h"
#include <cfloat>

// ================================================================= element-wise stages
// Q4_K embedding rows of tokens[0..T) (src/qx_format.c:3759-3793); block per token.
extern "C" __global__ __launch_bounds__(256) void qxp_embed(const uint8_t *emb, uint64_t row_bytes,
                                                            const uint32_t *tokens, float *x) {
    embed_q4k_row(emb + (uint64_t)tokens[blockIdx.x] * row_bytes, x + (uint64_t)blockIdx.x * 2048);
}

// RMSNorm of each token's 2048-vector (qx_apply_f32_rmsnorm, src/qx_format.c:3358-3371);
// wave per token (the stage probes).
extern "C" __global__ __launch_bounds__(256) void qxp_norm(const float *x, const float *w, uint32_t T, float *y) {
    const int lane = threadIdx.x & 63;
    const uint32_t t = blockIdx.x * 4 + wave_id();
    if (t >= T) return;
    float v[32], ww[32];
    load32(x + (uint64_t)t * 2048 + 32 * lane, v);
    load32(w + 32 * lane, ww);
    rmsnorm32(v, ww);
    float4 *o = reinterpret_cast<float4 *>(y + (uint64_t)t * 2048 + 32 * lane);
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}

// ---- rows of a token, block per token: thread tid holds values 8 tid .. 8 tid + 7.  (A wave per
// token with 32 values a lane left these stages waiting on one chain of loads after another:
// adding up 8 parts of Q/K/V took 45 us for 8 tokens.)
namespace {
DEV float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }
DEV void load8(const float *p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
DEV void store8(float *p, const float (&v)[8]) {
    reinterpret_cast<float4 *>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4 *>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
// RMSNorm of the block's 2048 values (qx_apply_f32_rmsnorm, src/qx_format.c:3358-3371; rmsnorm32's
// arithmetic, the squares summed in another order, in double)
DEV void block_rmsnorm(float (&v)[8], const float (&w)[8], double *red) {
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += (double)v[i] * (double)v[i];
    ss = wave_total_d(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const double inv = 1.0 / sqrt(((red[0] + red[1]) + (red[2] + red[3])) / 2048.0 + 1.0e-6);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (float)((double)v[i] * inv) * w[i];
}
// shift sh of the power-of-two scale that takes the block's largest magnitude into [2^13, 2^14);
// false when a value is not finite (the row then packs zeros under a scale of 0)
template <int N>
DEV bool block_shift(const float (&v)[N], float *red, int &sh) {
    float mx = 0.0f;
    bool fin = true;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        fin = fin && isfinite(v[i]);
        mx = fmaxf(mx, fabsf(v[i]));
    }
    mx = block_max256(fin ? mx : INFINITY, red);
    sh = 140 - (int)(__float_as_uint(mx) >> 23);
    sh = sh > 100 ? 100 : sh < -100 ? -100 : sh;
    return mx < INFINITY;
}
// 8 values as fp16 hi + lo at their chunk's place; returns the scaled values' sum
DEV float pack8(const float *v, float sc, bool ok, uint8_t *at) {
    h8v hi, lo;
    float t = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float y = ok ? v[j] * sc : 0.0f;
        const _Float16 a = (_Float16)y;
        hi[j] = a;
        lo[j] = (_Float16)(y - (float)a);
        t += y;
    }
    *reinterpret_cast<uint4 *>(at) = __builtin_bit_cast(uint4, hi);
    *reinterpret_cast<uint4 *>(at + 32) = __builtin_bit_cast(uint4, lo);
    return t;
}
// chunk c (8 values) of a dense row (k-steps of 16 consecutive values) and its line's sum
DEV void pack_dense8(const float *v, float sc, bool ok, uint8_t *row, float *sums, uint32_t c) {
    float t = pack8(v, sc, ok, row + (c >> 2) * 128 + 64 * ((c >> 1) & 1) + 16 * (c & 1));
    t += dppf<DPP_XOR1>(t);
    t += dppf<DPP_XOR2>(t);
    if ((c & 3) == 0) sums[c >> 2] = t;
}
// v += rows k .. k + N - 1 of 8 values, stride floats apart, in order, all loaded at once
template <int N>
DEV void add_parts(const float *p, uint64_t stride, float (&v)[8]) {
    float q[N][8];
#pragma unroll
    for (int u = 0; u < N; ++u) load8(p + u * stride, q[u]);
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += q[u][i];
}
// v = the sum of `parts` (a power of two) rows of 8 values, stride floats apart, in order
DEV void sum_parts(const float *p, uint64_t stride, uint32_t parts, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = -0.0f;
    if (parts == 1) add_parts<1>(p, stride, v);
    else if (parts == 2) add_parts<2>(p, stride, v);
    else if (parts == 4) add_parts<4>(p, stride, v);
    else for (uint32_t k = 0; k < parts; k += 8) add_parts<8>(p + k * stride, stride, v);
}
// x1 + sum_r (float)(w_r * (double)y[8 t + r]), ranks in order (src/qx_format.c:5296-5309)
DEV void combine8(const float *x1, const float *y, const double *wts, uint32_t t, int tid, float (&v)[8], float *moe) {
    float q[QXG_TOPK][8];
    double w[QXG_TOPK];
#pragma unroll
    for (int r = 0; r < QXG_TOPK; ++r) {
        load8(y + ((uint64_t)t * 8 + r) * 2048 + 8 * tid, q[r]);
        w[r] = wts[t * 8 + r];
    }
    load8(x1 + (uint64_t)t * 2048 + 8 * tid, v);
    float m[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        m[i] = 0.0f;
#pragma unroll
        for (int r = 0; r < QXG_TOPK; ++r) m[i] += (float)(w[r] * (double)q[r][i]);
        v[i] += m[i];
    }
    if (moe) store8(moe + (uint64_t)t * 2048 + 8 * tid, m);
}
}  // namespace

// The layer's input and its RMSNorm packed as the Q/K/V GEMM's rows.  With y, the input is the
// layer before's combined experts (combine8 on its x1, y and weights), stored to x.
extern "C" __global__ __launch_bounds__(256) void qxp_norm_pack(float *x, const float *x1, const float *y, const double *wts,
        const float *w, uint8_t *xp, float *rscale, float *sums) {
    __shared__ double red[4];
    __shared__ float redf[4];
    const int tid = threadIdx.x;
    const uint32_t t = blockIdx.x;
    float v[8], ww[8];
    load8(w + 8 * tid, ww);
    if (y) {
        combine8(x1, y, wts, t, tid, v, nullptr);
        store8(x + (uint64_t)t * 2048 + 8 * tid, v);
    } else {
        load8(x + (uint64_t)t * 2048 + 8 * tid, v);
    }
    block_rmsnorm(v, ww, red);
    int sh;
    const bool ok = block_shift<8>(v, redf, sh);
    if (tid == 0) rscale[t] = ok ? ldexpf(1.0f, -sh) : 0.0f;
    pack_dense8(v, ldexpf(1.0f, sh), ok, xp + (uint64_t)t * PF_PITCH(2048), sums + (uint64_t)t * 64, tid);
}

// The O projection's rows from the 4096-value context rows; with several runs of positions,
// the context is sum_r 2^(m_r - M) acc_r over sum_r 2^(m_r - M) den_r, runs in order.
extern "C" __global__ __launch_bounds__(256) void qxp_pack_ctx(const float *src, const float2 *md, uint32_t runs, uint32_t T,
                                                               uint8_t *xp, float *rscale, float *sums) {
    __shared__ float redf[4];
    const int tid = threadIdx.x;
    const uint32_t t = blockIdx.x;
    float v[16];
    const float *p = src + (uint64_t)t * 4096 + 8 * tid;
    if (runs == 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) load8(p + 2048 * i, *reinterpret_cast<float(*)[8]>(v + 8 * i));
    } else {
        // four runs' states, then their values, at a time: the compiler issues the values in groups of
        // two to four loads, a wait behind each (37 tokens over 12 runs: 11.8 us a run at a time, now 8)
        constexpr int N = 4;
        const float2 *s = md + (uint64_t)t * 32 + (tid >> 4);   // heads tid / 16 and 16 + tid / 16
        float M[2] = {-INFINITY, -INFINITY}, L[2] = {0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = 0.0f;
        for (uint32_t r0 = 0; r0 < runs; r0 += N) {
            float b[N][2][8];
            float2 st[N][2];
#pragma unroll
            for (int u = 0; u < N; ++u) {
                const uint32_t r = min(r0 + u, runs - 1);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    st[u][i] = s[(uint64_t)r * T * 32 + 16 * i];
                    load8(p + (uint64_t)r * T * 4096 + 2048 * i, b[u][i]);
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float m = M[i];
#pragma unroll
                for (int u = 0; u < N; ++u) m = fmaxf(m, st[u][i].x);   // (a repeated last run changes nothing)
                const float f0 = M[i] == -INFINITY ? 0.0f : exp2_fast(M[i] - m);
                L[i] *= f0;
#pragma unroll
                for (int j = 0; j < 8; ++j) v[8 * i + j] *= f0;
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const float f = r0 + u >= runs || st[u][i].x == -INFINITY ? 0.0f : exp2_fast(st[u][i].x - m);
                    L[i] = fmaf(f, st[u][i].y, L[i]);
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[8 * i + j] = fmaf(f, b[u][i][j], v[8 * i + j]);
                }
                M[i] = m;
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) v[8 * i + j] *= 1.0f / L[i];
    }
    int sh;
    const bool ok = block_shift<16>(v, redf, sh);
    if (tid == 0) rscale[t] = ok ? ldexpf(1.0f, -sh) : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        pack_dense8(v + 8 * i, ldexpf(1.0f, sh), ok, xp + (uint64_t)t * PF_PITCH(4096), sums + (uint64_t)t * 128, tid + 256 * i);
}

// The attention half's residual x1 = x + O (the O projection's parts of K added in order, a
// non-finite result 0, src/qx_format.c:4284) and its RMSNorm as f32 rows for the router and
// as the gate/up GEMM's packed rows (k-step 16 b + s and lane half h hold K = 256 b + 128 h +
// 8 s + j).
extern "C" __global__ __launch_bounds__(256) void qxp_ffn_norm(const float *x, const float *parts, uint32_t nparts,
        const float *w, uint32_t T, float *x1, float *y, uint8_t *xp, float *rscale) {
    __shared__ double red[4];
    __shared__ float redf[4];
    const int tid = threadIdx.x;
    const uint32_t t = blockIdx.x;
    const uint64_t at = (uint64_t)t * 2048 + 8 * tid;
    float v[8], r[8], ww[8];
    load8(x + at, r);
    load8(w + 8 * tid, ww);
    sum_parts(parts + at, (uint64_t)T * 2048, nparts, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = r[i] + (isfinite(v[i]) ? v[i] : 0.0f);
    store8(x1 + at, v);
    block_rmsnorm(v, ww, red);
    store8(y + at, v);
    int sh;
    const bool ok = block_shift<8>(v, redf, sh);
    if (tid == 0) rscale[t] = ok ? ldexpf(1.0f, -sh) : 0.0f;
    const uint32_t c = tid;
    pack8(v, ldexpf(1.0f, sh), ok, xp + (uint64_t)t * PF_PITCH(2048) + (16 * (c >> 5) + (c & 15)) * 64 + ((c >> 4) & 1) * 16);
}

// Per token (block): the Q/K/V GEMM's parts of K added in order (non-finite results 0,
// src/qx_format.c:4284), q/k head RMSNorm (src/qx_format.c:3740-3757) and RoPE at position
// p0+t (4625-4641), INT8 quantization of K and V over all 512 values (4449-4463) into
// the cache row [layer][p0+t]; the roped q (f32) goes to qr for attention.  Ten waves: each
// thread adds 8 columns, then waves 0 to 7 take four q heads each, wave 8 K and wave 9 V.
// Latency bounds it.  (Four waves with three runs of adds and eight q heads each: 8.9 us for
// 37 tokens, now 6.8.)
extern "C" __global__ __launch_bounds__(640) void qxp_qk(const float *parts, uint32_t nparts, uint32_t rows, const float *q_norm,
        const float *k_norm, Tables T, int8_t *kc, int8_t *vc, float *ks, float *vs, uint32_t layer, uint32_t ctx, uint32_t p0,
        float *qr) {
    __shared__ float s_row[5120];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const uint32_t t = blockIdx.x, pos = p0 + t;
    const float *nw = wave == 8 ? k_norm : q_norm;
    const float w0 = nw[lane], w1 = nw[64 + lane];
    const double c = T.rope_cos[pos * 64 + lane], s = T.rope_sin[pos * 64 + lane];
    float v[8];
    sum_parts(parts + (uint64_t)t * 5120 + 8 * tid, (uint64_t)rows * 5120, nparts, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = isfinite(v[j]) ? v[j] : 0.0f;
    store8(s_row + 8 * tid, v);
    __syncthreads();
    const float *own = s_row + 512 * wave + lane;   // the wave's four heads
    float a[4][2];
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) {
        a[hh][0] = own[128 * hh];
        a[hh][1] = own[128 * hh + 64];
        if (wave < 9) head_norm_rope_wave(a[hh][0], a[hh][1], w0, w1, c, s);
    }
    if (wave < 8) {
#pragma unroll
        for (int hh = 0; hh < 4; ++hh) {
            float *q = qr + (uint64_t)t * 4096 + 512 * wave + 128 * hh + lane;
            q[0] = a[hh][0];
            q[64] = a[hh][1];
        }
        return;
    }
    float mx = 0.0f;
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) mx = fmaxf(mx, fmaxf(int8_mag(a[hh][0]), int8_mag(a[hh][1])));
    const float scale = int8_scale(wave_max_f(mx));
    const uint64_t slot = (uint64_t)layer * ctx + pos;
    int8_t *code = (wave == 8 ? kc : vc) + slot * 512 + lane;
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) {
        code[128 * hh] = int8_code(a[hh][0], scale);
        code[128 * hh + 64] = int8_code(a[hh][1], scale);
    }
    if (lane == 0) (wave == 8 ? ks : vs)[slot] = scale;
}

// Causal GQA attention of the chunk on the matrix cores (qx_rope_gqa_attention_partial,
// src/qx_format.c:5051-5196, for every token of the chunk at once).  A workgroup takes one KV
// head, 4 consecutive tokens and a run of 32-position chunks (gridDim.z of them, so that few
// tokens over a long cache still fill the GPU); the 8 q heads of the KV head x 4 tokens are
// the 32 columns of v_mfma_f32_32x32x16_f16 (column c: head c/4, token c%4).  Its 4 waves
// take every fourth chunk and keep, per column, a running maximum, denominator and context.
// Per chunk:
//   scores  S^T[pos][col] = K8[pos][:] . q[col][:]: A = the chunk's INT8 K codes (exact in
//           fp16; lane half h holds dims 64h .. 64h + 63 of a position), B = q split hi + lo
//           in fp16 after a power-of-two row scale (in LDS, the same for the four waves),
//           the hi and the lo products summed apart (two chains of matrix instructions);
//           times ks[pos]; positions past the token masked in the chunks that hold any;
//   weights e = 2^(score * scale - m), pv = e * vs[pos] split hi + lo under a power-of-two
//           scale of the column in this chunk (from its largest |pv|, so that a chunk of small
//           weights behind a large one keeps all its bits);
//   context C[dim][col] = V8^T[dim][pos] . pv[pos][col] (A = V codes from a transposed LDS copy
//           of the chunk), added to the running context at the scale's inverse.
// The result registers of the score product are exactly the k layout the context product's B
// operand needs (lane l: column l%32, positions 8(r/4) + 4(l/32) + r%4 of register r), so the
// weights never leave the lane.  The softmax's vector work bounds this kernel, about 17 issue
// slots a score against 64 matrix cycles per 32 of them, so: m is the running maximum only to
// within a factor 2^8, and the context is rescaled (64 multiplies) only in the chunks that leave
// that; the exponent is base 2; the next chunk's K and V rows are loaded while the current one is
// worked on.  (One scale of the column over all chunks spared the 64 additions, which measured
// the same: 112 us for 512 at 3500 either way, and lost the bits of later, smaller weights.)  The
// waves' states are merged in LDS, the runs' by qxp_pack_ctx.  (One run, the context rescaled at every
// chunk: 60 us for 37 tokens at position 2100, now 16; 139 for 512 at 3500, now 106 to 113.)
namespace {
constexpr int PA_TT = 4;   // tokens per workgroup

DEV uint4 i8x8_to_f16(uint32_t vx, uint32_t vy) {   // 8 int8 -> 8 exact fp16 (bias 0x64 trick: 1024 + (b ^ 0x80) - 1152)
    const h2v bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t x = vx ^ 0x80808080u, y = vy ^ 0x80808080u;
    const uint32_t c = 0x64646464u;
    auto cv = [&](uint32_t w) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2v, w) - bias); };
    return make_uint4(cv(perm(c, x, 0x04010400u)), cv(perm(c, x, 0x04030402u)), cv(perm(c, y, 0x04010400u)),
                      cv(perm(c, y, 0x04030402u)));
}
DEV void split8(const float *v, float sc, uint4 &hi, uint4 &lo) {   // v * sc = hi + lo (+ 2^-22 rel)
    h8v h, l;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float a = v[i] * sc;
        const _Float16 t = (_Float16)a;
        h[i] = t;
        l[i] = (_Float16)(a - (float)t);
    }
    hi = __builtin_bit_cast(uint4, h);
    lo = __builtin_bit_cast(uint4, l);
}
// 2^(k - e) with |v| = f * 2^e, f in [0.5, 1); 1 for zero, subnormal and non-finite v
DEV float pow2_scale(float v, int k) {
    const int e = (int)((__float_as_uint(v) >> 23) & 255u);
    const int s = 127 + k + 126 - e;   // exponent field of the result
    return e == 0 || e == 255 ? 1.0f : __uint_as_float((uint32_t)(s < 1 ? 1 : s > 254 ? 254 : s) << 23);
}
struct PaRows { uint4 k[4]; uint32_t v[16]; float ks, vs; };   // a chunk's rows as one lane loads them
}  // namespace

extern "C" __global__ __launch_bounds__(256, 2) void qxp_attn(const float *qr, const int8_t *kc, const int8_t *vc,
        const float *ks, const float *vs, uint32_t layer, uint32_t ctx, uint32_t p0, uint32_t T, float *ctx_out, float2 *md) {
    __shared__ uint4 s_q[8 * 2 * 64];           // [k-step][hi, lo][lane] q fragments
    __shared__ float s_sf[32];                  // per column: 1 / (q scale * sqrt(128)) * log2(e)
    __shared__ float s_ks[4][32], s_vs[4][32];
    __shared__ float s_m[2][32], s_den[2][32];
    __shared__ union { uint32_t vt[4][128 * 9]; float acc[2][32][129]; } u;   // per wave V^T rows of 36 bytes; the merge
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const int col = lane & 31, h = lane >> 5;
    const uint32_t kh = blockIdx.x, t0 = blockIdx.y * PA_TT;
    const uint32_t tt = t0 + (col & 3), qh = kh * 8 + (col >> 2);
    const bool tok_ok = tt < T;
    const uint32_t limit = p0 + (tok_ok ? tt : 0);              // last position of the column's token
    const uint32_t npos = p0 + min(t0 + PA_TT, T);              // positions the workgroup's tokens need
    const uint32_t nchunk = (npos + 31) / 32;
    const uint32_t c_lo = nchunk * blockIdx.z / gridDim.z, c_hi = nchunk * (blockIdx.z + 1) / gridDim.z;
    const uint64_t base = (uint64_t)layer * ctx;
    PaRows nx;
    auto load = [&](uint32_t ci) {   // (rows past the last position read it again)
        const uint32_t pb = ci * 32, pk = min(pb + col, npos - 1);
        const uint4 *krow = reinterpret_cast<const uint4 *>(kc + (base + pk) * 512 + kh * 128 + 64 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i) nx.k[i] = krow[i];
        nx.ks = ks[base + pk];
        nx.vs = vs[base + pk];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int bq = lane + 64 * i, pq = bq & 7, dq = bq >> 3;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                nx.v[4 * i + r] = *reinterpret_cast<const uint32_t *>(vc + (base + min(pb + 4 * pq + r, npos - 1)) * 512 + kh * 128 + 4 * dq);
        }
    };
    if (c_lo + wave < c_hi) load(c_lo + wave);
    // q: thread takes 16 dims of a column; k-step s of lane half hh holds dims 64 hh + 8 s + j
    {
        const int c = tid >> 3, seg = tid & 7;
        const uint32_t ct = t0 + (c & 3);
        float v[16], mx = 0.0f;
        bool fin = true;
        const float4 *qrow = reinterpret_cast<const float4 *>(qr + (uint64_t)(ct < T ? ct : 0) * 4096 + (kh * 8 + (c >> 2)) * 128 + 16 * seg);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 a = qrow[i];
            v[4 * i] = a.x; v[4 * i + 1] = a.y; v[4 * i + 2] = a.z; v[4 * i + 3] = a.w;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) { fin = fin && isfinite(v[i]); mx = fmaxf(mx, fabsf(v[i])); }
        mx = fin && ct < T ? mx : INFINITY;
        mx = fmaxf(mx, dppf<DPP_XOR1>(mx)); mx = fmaxf(mx, dppf<DPP_XOR2>(mx)); mx = fmaxf(mx, dppf<DPP_HALF_MIRROR>(mx));
        // a non-finite q makes every score non-finite, which the reference stores as 0
        const bool zero = !(mx < INFINITY);
        const float sc = pow2_scale(zero ? 0.0f : mx, 14);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = zero ? 0.0f : v[i];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint4 hi, lo;
            split8(v + 8 * i, sc, hi, lo);
            const int s = 2 * (seg & 3) + i, l = c + 32 * (seg >> 2);
            s_q[(s * 2 + 0) * 64 + l] = hi;
            s_q[(s * 2 + 1) * 64 + l] = lo;
        }
        if (seg == 0) s_sf[c] = (float)(1.4426950408889634 / ((double)sc * sqrt(128.0)));
    }
    __syncthreads();
    const float sf = s_sf[col], sf_most = wave_max_f(sf);
    float m = -INFINITY, den = 0.0f;
    f16x acc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[d] = zero16();
    uint32_t *vt = u.vt[wave];
#pragma unroll 1
    for (uint32_t ci = c_lo + wave; ci < c_hi; ci += 4) {
        const uint32_t pb = ci * 32;
        // this chunk's rows: scales and V^T to LDS (a wave's own), K stays in registers
        const uint4 kq[4] = {nx.k[0], nx.k[1], nx.k[2], nx.k[3]};
        // a score is a sum below 2^28 times ks and sf: beyond 2^20 the rounding of the maximum, which the
        // weights' fma does not repeat, would show, beyond 2^128 the score itself is lost
        const bool big = __ballot(!(fabsf(nx.ks) * fmaxf(sf_most, 0x1p-98f) < 0x1p-8f)) != 0;
        if (lane < 32) {
            s_ks[wave][lane] = nx.ks;
            s_vs[wave][lane] = nx.vs;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int bq = lane + 64 * i, pq = bq & 7, dq = bq >> 3;
            const uint32_t *w = nx.v + 4 * i;
            const uint32_t a0 = perm(w[1], w[0], 0x05010400u), a1 = perm(w[3], w[2], 0x05010400u);
            const uint32_t a2 = perm(w[1], w[0], 0x07030602u), a3 = perm(w[3], w[2], 0x07030602u);
            vt[(4 * dq + 0) * 9 + pq] = perm(a1, a0, 0x05040100u);
            vt[(4 * dq + 1) * 9 + pq] = perm(a1, a0, 0x07060302u);
            vt[(4 * dq + 2) * 9 + pq] = perm(a3, a2, 0x05040100u);
            vt[(4 * dq + 3) * 9 + pq] = perm(a3, a2, 0x07060302u);
        }
        if (ci + 4 < c_hi) load(ci + 4);
        // scores: S^T = K8 . q
        f16x sh = zero16(), sl = zero16();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint4 kw = kq[s >> 1];
            const uint4 kf = s & 1 ? i8x8_to_f16(kw.z, kw.w) : i8x8_to_f16(kw.x, kw.y);
            sh = mfma(kf, s_q[(s * 2 + 0) * 64 + lane], sh);
            sl = mfma(kf, s_q[(s * 2 + 1) * 64 + lane], sl);
            if (s & 1) asm volatile("" ::: "memory");   // later q reads stay below: hoisted together they spill
        }
        // register r: position pb + 8(r/4) + 4h + r%4
        float sc[16], cmax = -INFINITY, f = sf;   // scores, still to be multiplied by f
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f4x k4 = *reinterpret_cast<const f4x *>(&s_ks[wave][8 * q + 4 * h]);
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[4 * q + r] = (sh[4 * q + r] + sl[4 * q + r]) * k4[r];
        }
        if (big) {
            // rounded once, so that the largest has weight 1.  The reference's scores are doubles: one beyond
            // f32 stays the largest there is; where K itself is not finite it is 0 (src/qx_format.c:5137-5139)
            f = 1.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float k = s_ks[wave][8 * (r >> 2) + 4 * h + (r & 3)];
                const double v = (double)(sh[r] + sl[r]) * ((double)k * (double)sf);
                sc[r] = fabsf(k) <= FLT_MAX / 127.0f ? (float)fmin(fmax(v, -3.0e38), 3.0e38) : 0.0f;
            }
        }
        const bool tail = pb + 31 > p0 + t0;   // the chunk holds positions past the first token
        if (tail) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = pb + 8 * (r >> 2) + 4 * h + (r & 3) <= limit ? sc[r] : -INFINITY;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) cmax = fmaxf(cmax, sc[r]);
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32)) * f;
        f4x v4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v4[q] = *reinterpret_cast<const f4x *>(&s_vs[wave][8 * q + 4 * h]);
        const bool grow = cmax > m + 8.0f;
        if (__ballot(grow) != 0) {   // (whole wave)
            const float mn = fmaxf(m, cmax);
            const float alpha = mn == -INFINITY || m == -INFINITY ? (m == mn ? 1.0f : 0.0f) : exp2_fast(m - mn);
            m = mn;
            den *= alpha;
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[d][r] *= alpha;
        }
        const float mm = m == -INFINITY ? 0.0f : m;
        float e[16], pv[16], pmx = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            e[r] = exp2_fast(fmaf(sc[r], f, -mm));
            pv[r] = e[r] * v4[r >> 2][r & 3];
        }
        if (tail) {   // (a masked position's V scale does not count, whatever it is)
#pragma unroll
            for (int r = 0; r < 16; ++r) pv[r] = sc[r] == -INFINITY ? 0.0f : pv[r];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) pmx = fmaxf(pmx, fabsf(pv[r]));
        pmx = fmaxf(pmx, __shfl_xor(pmx, 32));
        const float psc = pow2_scale(pmx, 15), pinv = 1.0f / psc;   // (powers of two: exact)
#pragma unroll
        for (int r = 0; r < 16; ++r) den += e[r];
        uint4 phi[2], plo[2];
        split8(pv, psc, phi[0], plo[0]);
        split8(pv + 8, psc, phi[1], plo[1]);
        // context: per 32-dim tile, C[dim][col] = V8^T . pv
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            f16x c = zero16();
            const uint32_t *row = vt + (32 * d + col) * 9;
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                const uint4 vf = i8x8_to_f16(row[4 * s2 + h], row[4 * s2 + 2 + h]);
                c = mfma(vf, phi[s2], c);
                c = mfma(vf, plo[s2], c);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[d][r] = fmaf(c[r], pinv, acc[d][r]);
        }
    }
    // merge the 4 waves' (max, denominator, context) per column: 2+3 into 0+1, then 1 into 0
    den += __shfl_xor(den, 32);
    __syncthreads();   // the V^T rows are read: their space takes the merge
#pragma unroll 1
    for (int round = 0; round < 2; ++round) {
        const int nw = round == 0 ? 2 : 1;   // waves [nw, 2nw) hand over to [0, nw)
        if (wave >= nw && wave < 2 * nw) {
            const int slot = wave - nw;
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) u.acc[slot][col][32 * d + 8 * (r >> 2) + 4 * h + (r & 3)] = acc[d][r];
            if (h == 0) { s_m[slot][col] = m; s_den[slot][col] = den; }
        }
        __syncthreads();
        if (wave < nw) {
            const float mo = s_m[wave][col], dn = s_den[wave][col];
            const float m_new = fmaxf(m, mo);
            const float fa = m == -INFINITY ? 0.0f : exp2_fast(m - m_new);
            const float fb = mo == -INFINITY ? 0.0f : exp2_fast(mo - m_new);
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[d][r] = acc[d][r] * fa + u.acc[wave][col][32 * d + 8 * (r >> 2) + 4 * h + (r & 3)] * fb;
            den = den * fa + dn * fb;
            m = m_new;
        }
        __syncthreads();
    }
    if (wave == 0 && tok_ok) {
        // one run: the context itself; several: its sums, with their maximum and denominator
        const float inv = gridDim.z == 1 ? 1.0f / den : 1.0f;
        const uint64_t row = (uint64_t)blockIdx.z * T + tt;
        float *out = ctx_out + row * 4096 + qh * 128;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4 *>(out + 32 * d + 8 * q + 4 * h) =
                    make_float4(acc[d][4 * q] * inv, acc[d][4 * q + 1] * inv, acc[d][4 * q + 2] * inv, acc[d][4 * q + 3] * inv);
        if (h == 0) md[row * 32 + qh] = make_float2(m, den);
    }
}

// Router logits on the FP64 matrix cores: logit[t][e] = sum_i (double)W[e][i] *
// (double)xn[t][i] (src/qx_format.c:5254-5264: the same exact double products, summed in
// another order, within ~1e-15 relative of the reference's sequential sum; equal router
// rows still give equal logits).  A workgroup owns a 16 x 16 (token x expert) tile of one
// quarter of K; its 4 waves split that in 128s, and lane group g = lane / 16 of a wave feeds
// k-slot g of v_mfma_f64_16x16x4 with float4 g of each 16 k.  The waves' tiles are added in
// LDS in a fixed order, the quarters (planes of `logits`) by qxp_route.  Latency bounds it: the
// compiler keeps four of a wave's sixteen loads in flight, the next two issued behind each pair's
// products; a row's four lane groups read one 64-byte piece.  (A workgroup over all of K, loads four iterations at a time: 11.4 us
// for 37 tokens and 12.6 for 512; now 4.9 and 10.2.)
typedef double f64x4 __attribute__((ext_vector_type(4)));
extern "C" __global__ __launch_bounds__(256) void qxp_router(const float *xn, const float *router, uint32_t T,
                                                             uint32_t experts, double *logits, uint32_t *cnt) {
    __shared__ double part[4][16][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const int i = lane & 15, g = lane >> 4;
    if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && tid < 128) cnt[tid] = 0u;   // for qxp_route, the next launch
    const uint32_t t = blockIdx.x * 16 + i;   // < 512: xn holds QXP_MAX rows
    const uint32_t e = blockIdx.y * 16 + i, er = e < experts ? e : 0u;
    const uint32_t k0 = blockIdx.z * 512 + wave * 128 + g * 4;
    const float *xa = xn + (uint64_t)t * 2048 + k0, *wb = router + (uint64_t)er * 2048 + k0;
    float4 a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        a[j] = *reinterpret_cast<const float4 *>(xa + 16 * j);
        b[j] = *reinterpret_cast<const float4 *>(wb + 16 * j);
    }
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[j].x, (double)b[j].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[j].y, (double)b[j].y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[j].z, (double)b[j].z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[j].w, (double)b[j].w, acc, 0, 0, 0);
    }
    // result r of lane l: token row l / 16 + 4 * r, expert column l % 16 (the f64 16x16
    // layout, unlike the f32 ones' 4 * (l / 16) + r)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][g + 4 * r][i] = acc[r];
    __syncthreads();
    const int row = tid >> 4, col = tid & 15;
    const double v = (part[0][row][col] + part[1][row][col]) + (part[2][row][col] + part[3][row][col]);
    const uint32_t tt = blockIdx.x * 16 + row, ee = blockIdx.y * 16 + col;
    if (tt < T && ee < experts) logits[((uint64_t)blockIdx.z * QXP_MAX + tt) * 128 + ee] = v;
}

// Top-8 experts and renormalised weights per token (the decode path's selection,
// src/qx_format.c:5265-5285), and the experts' pairs.  A workgroup takes 16 tokens, one a wave, and
// writes its word of every expert's set (bit p % 128 of pair p = 8 t + rank) and adds the words'
// bits to the counts.  The sets come out the same whatever the order of the workgroups; the expert
// GEMMs take the pairs in token order.  (Lists whose places were claimed by atomics put a pair into
// another pass from run to run, and a pass of at most 16 rows rounds differently.)
extern "C" __global__ __launch_bounds__(1024) void qxp_route(const double *logits, uint32_t T, uint32_t experts,
                                                             double *wts, uint32_t *cnt, uint4 *sets) {
    __shared__ uint4 s_set[128];
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < 128) s_set[tid] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    const int E = (int)experts;
    const uint32_t t = blockIdx.x * 16 + wave_id();
    if (t < T) {   // whole wave
        double q[4][2];   // the quarters of K
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double *lg = logits + ((uint64_t)k * QXP_MAX + t) * 128;
            q[k][0] = lane < E ? lg[lane] : 0.0;
            q[k][1] = lane + 64 < E ? lg[lane + 64] : 0.0;
        }
        const double l0 = (q[0][0] + q[1][0]) + (q[2][0] + q[3][0]), l1 = (q[0][1] + q[1][1]) + (q[2][1] + q[3][1]);
        uint32_t id[QXG_TOPK];
        double w[QXG_TOPK];
        wave_top8(l0, l1, E, id, w);
        double wl = 0.0;
        uint32_t e = 0;
#pragma unroll
        for (int q = 0; q < QXG_TOPK; ++q)
            if (lane == q) {
                e = id[q] < experts ? id[q] : 0u;
                wl = w[q];
            }
        if (lane < QXG_TOPK) {
            wts[t * 8 + lane] = wl;
            const uint32_t bit = 8 * wave_id() + lane;
            atomicOr(reinterpret_cast<uint32_t *>(&s_set[e]) + (bit >> 5), 1u << (bit & 31));
        }
    }
    __syncthreads();
    if (tid < 128) {
        const uint4 m = s_set[tid];
        sets[tid * QXP_SET + blockIdx.x] = m;
        const uint32_t n = __popc(m.x) + __popc(m.y) + __popc(m.z) + __popc(m.w);
        if (n) atomicAdd(&cnt[tid], n);
    }
}

// The last layer's output x = x1 + its combined experts (moe_dump: the expert sum alone)
extern "C" __global__ __launch_bounds__(256) void qxp_combine(const float *x1, const float *y, const double *wts, float *x,
                                                              float *moe_dump) {
    float v[8];
    combine8(x1, y, wts, blockIdx.x, threadIdx.x, v, moe_dump);
    store8(x + (uint64_t)blockIdx.x * 2048 + 8 * threadIdx.x, v);
}
