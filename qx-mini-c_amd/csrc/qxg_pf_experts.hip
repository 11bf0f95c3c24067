// Routed-expert GEMMs of the batched prefill (CDNA4, gfx950).
//
// Precision is that of qxg_prefill.hip: a weight is an f32 block scale times an integer
// code that fp16 holds exactly, an activation row is scaled by a power of two and split
// into fp16 hi + lo, the matrix cores accumulate in f32.  Here:
//
// Rows.  qxp_route forms each expert's set of (token, rank) pairs, p = 8 * token + rank; a
// workgroup takes up to 32 or 64 of one expert's pairs, in token order, and a range of its weight
// rows, and forms each code once for them.  Activations are packed per token
// (gate/up, gathered through the pairs while they are staged) and per pair (down, written
// by gate/up's epilogue); no copy of them is sorted or padded by expert.
//
// Order of K.  Which 8 values a lane half holds is free as long as A and B agree: a lane
// takes its part of a weight block whole, and the rows are packed (qxg_pf.h) with
//     gate/up: K = 256 b + 128 h + 8 s + j, k-step 16 b + s    (sub-blocks 4h .. 4h + 3)
//     down:    K = 128 q + 64 h + 8 s + j, k-step 8 q + s      (two sub-blocks of a half block)
//     down in IQ4_XS: K = 32 i + 8 h + 4 t + j / 2 + 16 (j % 2), k-step 2 i + t   (a scale per 32)
//
// Codes.  The codebooks are bytes in LDS, 8 or 4 magnitudes an entry, with a second table
// of sign bytes (0x80 where negative).  A magnitude byte and its sign byte side by side are
// a subnormal fp16 number, sign * mag * 2^-24, so one v_perm forms two of them and one
// v_pk_mul by (2 s + 1) * 2^11 makes the codes, exactly, at 2^-13 (11 significant bits; the
// block scale takes the 2^13).  Random 16-byte reads of ready fp16 entries and fp16 sign masks
// kept the LDS busy for most of the kernel; these take about 6 cycles each.
//
// What bounds them: the matrix instructions (twice the algorithmic work, for hi and lo) and the about 16
// vector instructions per 8 codes, which share a SIMD's time nearly without overlap (counted on 128
// random rows of gate/up: 49k and 59k of 120k cycles).
#include "qxg_pf.h"

namespace {
enum { FMT_IQ2 = 0, FMT_IQ2S = 1, FMT_IQ3 = 2, FMT_IQ3S = 3, FMT_IQ4 = 4 };

// two signed codes (sign byte over magnitude byte, a subnormal fp16) times m
DEV uint32_t code2(uint32_t mag, uint32_t sgn, uint32_t sel, h2v m) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2v, perm(sgn, mag, sel)) * m);
}
struct Codes { uint32_t m0, m1; uint2 sg; };   // 8 magnitude bytes and their sign bytes
DEV uint4 conv(const Codes &c, h2v m) {
    return make_uint4(code2(c.m0, c.sg.x, 0x05010400u, m), code2(c.m0, c.sg.x, 0x07030602u, m),
                      code2(c.m1, c.sg.y, 0x05010400u, m), code2(c.m1, c.sg.y, 0x07030602u, m));
}
DEV h2v odd_mul(uint32_t n) {   // (2 n + 1) * 2^11, n < 16: exact
    const _Float16 f = (_Float16)(uint16_t)((n << 12) | 2048u);
    return h2v{f, f};
}
constexpr float CODE_SCALE = 8192.0f;   // 2^13: the codes above are at 2^-13

// the sum of v over lanes 0 .. lane
DEV uint32_t wave_prefix(uint32_t v) {
    int s = (int)v;
    s += __builtin_amdgcn_update_dpp(0, s, 0x111, 0xf, 0xf, false);   // row_shr 1, 2, 4, 8
    s += __builtin_amdgcn_update_dpp(0, s, 0x112, 0xf, 0xf, false);
    s += __builtin_amdgcn_update_dpp(0, s, 0x114, 0xf, 0xf, false);
    s += __builtin_amdgcn_update_dpp(0, s, 0x118, 0xf, 0xf, false);
    s += __builtin_amdgcn_update_dpp(0, s, 0x142, 0xa, 0xf, false);   // row 0's and 2's sum to the row above
    s += __builtin_amdgcn_update_dpp(0, s, 0x143, 0xc, 0xf, false);   // the lower half's to the upper
    return (uint32_t)s;
}
// Pairs m0 .. m0 + n - 1 of expert e in token order (n at most R), the last repeated up to R.  One whole
// wave; lane l looks at tokens 8 l .. 8 l + 7.
template <int R>
DEV void pass_pairs(const PfExperts &a, uint32_t e, uint32_t m0, uint32_t n, uint32_t *s_pair) {
    const uint32_t lane = threadIdx.x & 63;
    uint2 m = make_uint2(0u, 0u);
    if (lane < 2 * a.words) m = reinterpret_cast<const uint2 *>(a.sets + e * QXP_SET)[lane];
    const uint32_t c = __popc(m.x) + __popc(m.y);
    uint32_t at = wave_prefix(c) - c - m0;   // (wraps below m0)
#pragma unroll 1
    for (uint64_t w = (uint64_t)m.y << 32 | m.x; w; w &= w - 1, ++at)
        if (at < n) s_pair[at] = 64 * lane + (uint32_t)__builtin_ctzll(w);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane >= n && lane < R) s_pair[lane] = s_pair[n - 1];
}

DEV uint32_t word_at(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }
DEV uint32_t byte_at(const uint4 &v, int i) { return (word_at(v, i >> 2) >> (8 * (i & 3))) & 255u; }
DEV uint32_t ldu16(const void *p) { return *reinterpret_cast<const uint16_t *>(p); }
DEV uint32_t ldu32(const void *p) { return *reinterpret_cast<const uint32_t *>(p); }
DEV uint2 ldu64(const void *p) { return *reinterpret_cast<const uint2 *>(p); }
DEV uint4 ldu128(const void *p) { return *reinterpret_cast<const uint4 *>(p); }

// ---------------------------------------------------------------- gate/up weights
template <int F> struct GuBlk;                                               // the lane's half of a block
template <> struct GuBlk<FMT_IQ2> { uint4 q[2]; uint32_t sc, d; };           // 16 grid/sign words, 4 scale bytes
template <> struct GuBlk<FMT_IQ2S> { uint4 q, sg; uint32_t qh, sc, d; };     // 16 grid bytes, sign bytes, 4 x 8 high bits
// load instructions of gu_load: a wait counts on them (the listing's test holds the built code to it)
template <int F> constexpr int GU_LOADS = F == FMT_IQ2 ? 4 : 5;
DEV void gu_load(GuBlk<FMT_IQ2> &w, const PfMat &m, uint32_t bi, int h) {
    w.q[0] = ldu128(m.qs + bi * 64u + 32 * h);
    w.q[1] = ldu128(m.qs + bi * 64u + 32 * h + 16);
    w.sc = ldu32(m.p1 + bi * 8u + 4 * h);
    w.d = ldu16(m.d + bi);
}
DEV void gu_load(GuBlk<FMT_IQ2S> &w, const PfMat &m, uint32_t bi, int h) {
    w.q = ldu128(m.qs + bi * 64u + 16 * h);
    w.sg = ldu128(m.qs + bi * 64u + 32 + 16 * h);
    w.qh = ldu32(m.p2 + bi * 8u + 4 * h);
    w.sc = ldu32(m.p1 + bi * 8u + 4 * h);
    w.d = ldu16(m.d + bi);
}
// IQ2_XS (src/qx_format.c:1914-1933): entry 16h + s is grid word q & 511, sign index q >> 9,
// scaled by the nibble s / 2 of the lane's four scale bytes
DEV Codes gu_look(const GuBlk<FMT_IQ2> &w, int s, const uint2 *grid, const uint2 *sgn) {
    const uint32_t q = word_at(w.q[s >> 3], (s >> 1) & 3) >> (16 * (s & 1));
    const uint2 m = grid[q & 511u];
    return Codes{m.x, m.y, sgn[(q >> 9) & 127u]};
}
// IQ2_S (src/qx_format.c:1961-1984): grid byte with two high bits, explicit sign byte
DEV Codes gu_look(const GuBlk<FMT_IQ2S> &w, int s, const uint2 *grid, const uint2 *sgn) {
    const uint2 m = grid[byte_at(w.q, s) | (((w.qh >> (2 * s)) & 3u) << 8)];
    return Codes{m.x, m.y, sgn[byte_at(w.sg, s)]};
}

// k-steps 8 half .. 8 half + 7 of a block: gate (tile 0) and up (1) of the wave's 32 columns.
// Tile i's codes are looked up two tiles ahead and formed one ahead.
template <int F, int R>
DEV void gu_half(const GuBlk<F> (&w)[2], int half, const uint4 *buf, const ALane &at, f16x (&G)[2], const uint2 *grid,
                 const uint2 *sgn) {
    Codes c0 = gu_look(w[0], 8 * half, grid, sgn), c1 = gu_look(w[1], 8 * half, grid, sgn);
    uint4 ah[1], al[1];
    a_read<R, 1>(ah, al, buf, at, 0);
    h2v m[2] = {odd_mul((w[0].sc >> (16 * half)) & 15u), odd_mul((w[1].sc >> (16 * half)) & 15u)};
    uint4 b = conv(c0, m[0]);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int s = i >> 1, f = i & 1, sn = (i + 1) >> 1, fn = (i + 1) & 1;
        uint4 bn = b, nh[1], nl[1];
        if (i < 15) {
            if (sn && !(sn & 1)) m[fn] = odd_mul((w[fn].sc >> (16 * half + 4 * (sn >> 1))) & 15u);
            bn = conv(c1, m[fn]);
        }
        if (i < 14) c1 = gu_look(w[f], 8 * half + s + 1, grid, sgn);
        if (f == 1 && s < 7) a_read<R, 1>(nh, nl, buf, at, s + 1);
        G[f] = mfma(ah[0], b, G[f]);
        if (R > 16) G[f] = mfma(al[0], b, G[f]);
        b = bn;
        if (f == 1 && s < 7) {
            ah[0] = nh[0];
            if (R > 16) al[0] = nl[0];
        }
    }
}

DEV float exp2i(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }   // 2^e, -126 <= e <= 127

template <int F, int R>
DEV void gu_pass(const PfExperts &a, uint32_t e, uint32_t cg, uint32_t m0, uint32_t n, const uint2 *grid,
                 const uint2 *sgn, uint4 *buf, uint32_t *s_pair, float *s_xs) {
    constexpr int NR = R > 16 ? 16 : 8;   // result registers of a tile, hi and lo added
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), h = lane >> 5, col = lane & 31;
    const uint32_t bi = (e * QXG_FFN + 128 * cg + 32 * wave + col) * 8;   // tiles 0 and 1: this row of gate and of up
    GuBlk<F> cur[2], nxt[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) gu_load(cur[f], a.w[f], bi, h);
    if (wave == 0) pass_pairs<R>(a, e, m0, n, s_pair);
    __syncthreads();   // the pairs, and the tables
    uint32_t off[R / 8];
    stage_offsets<R, 3>(off, s_pair, PF_PITCH(2048), lane);
    stage_rows<R>(a.xp, off, 0, buf, wave);
    if (tid < R) s_xs[tid] = a.xs[s_pair[tid] >> 3];   // (read behind the loop's barriers)
    const ALane at = a_lane<R>(lane);
    f16x acc[2] = {zero16(), zero16()};
#pragma unroll 1
    for (uint32_t b = 0; b < 8; ++b) {
        f16x G[2] = {zero16(), zero16()};
        wait_loads<0>();
        __syncthreads();   // the block's first half is staged; every wave is past the last block's second half
        stage_rows<R>(a.xp, off, 8 * b + 4, buf + STAGE<R>, wave);
        __builtin_amdgcn_sched_barrier(0);   // the weights' loads stay the youngest: the wait below leaves them in flight
        const uint32_t bn = b < 7 ? b + 1 : 7;
#pragma unroll
        for (int f = 0; f < 2; ++f) gu_load(nxt[f], a.w[f], bi + bn, h);
        __builtin_amdgcn_sched_barrier(0);
        gu_half<F, R>(cur, 0, buf, at, G, grid, sgn);
        wait_loads<2 * GU_LOADS<F>>();
        __syncthreads();
        if (b < 7) stage_rows<R>(a.xp, off, 8 * b + 8, buf, wave);
        gu_half<F, R>(cur, 1, buf + STAGE<R>, at, G, grid, sgn);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const float d = fp16_exact(cur[f].d) * (0.125f * CODE_SCALE);
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[f][r] = fmaf(d, R > 16 ? G[f][r] : G[f][r] + G[f][(r + 8) & 15], acc[f][r]);
            cur[f] = nxt[f];
        }
    }
    // SwiGLU (qx_silu, src/qx_format.c:2511-2513, in f32: relative error ~1e-7 against the
    // reference's double) into LDS, rows of 128 values
    __syncthreads();
    float *hs = reinterpret_cast<float *>(buf);
    constexpr int LD = 132;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const uint32_t row = 8 * (r >> 2) + 4 * h + (r & 3);
        const float rs = s_xs[row];
        float gv = acc[0][r] * rs, uv = acc[1][r] * rs;
        gv = isfinite(gv) ? gv : 0.0f;   // (src/qx_format.c:4284)
        uv = isfinite(uv) ? uv : 0.0f;
        hs[row * LD + 32 * wave + col] = gv / (1.0f + expf(-gv)) * uv;   // (correctly rounded quotient)
    }
    __syncthreads();
    // each row's 128 values become the down projection's packed operand, 16 lanes a row with 8
    // values each, under a power-of-two scale of their own; a non-finite value makes the
    // scale a NaN, which zeroes the pair's down row (its own non-finite rule)
#pragma unroll
    for (int i = 0; i < R / 16; ++i) {
        const uint32_t row = 16 * i + (tid >> 4), c = tid & 15;
        // chunk c of the 128 values: k-step and lane half of the down operand's order
        const uint32_t ks = 8 * cg + (a.h_pairs ? 2 * (c >> 2) + ((c >> 1) & 1) : c & 7), hh = a.h_pairs ? c & 1 : c >> 3;
        const float *src = hs + row * LD + (a.h_pairs ? 32 * (c >> 2) + 8 * (c & 1) + 4 * ((c >> 1) & 1) : 8 * c);
        const float4 p = *reinterpret_cast<const float4 *>(src);
        const float4 q = *reinterpret_cast<const float4 *>(src + (a.h_pairs ? 16 : 4));
        float v[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
        if (a.h_pairs) { v[1] = q.x; v[2] = p.y; v[3] = q.y; v[4] = p.z; v[5] = q.z; v[6] = p.w; }
        float mx = 0.0f;
        bool fin = true;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            fin = fin && isfinite(v[j]);
            mx = fmaxf(mx, fabsf(v[j]));
        }
        mx = fin ? mx : INFINITY;   // the 16 lanes' largest, infinite where a value is not finite
        mx = fmaxf(mx, dppf<DPP_XOR1>(mx)); mx = fmaxf(mx, dppf<DPP_XOR2>(mx));
        mx = fmaxf(mx, dppf<DPP_ROR4>(mx)); mx = fmaxf(mx, dppf<DPP_ROR8>(mx));
        const bool ok = mx < INFINITY;
        int sh = 140 - (int)(__float_as_uint(mx) >> 23);   // mx 2^sh in [2^13, 2^14) (zero and subnormal: 2^100)
        sh = sh > 100 ? 100 : sh < -100 ? -100 : sh;
        if (row < n) {
            const uint32_t pr = s_pair[row];
            const float sc = exp2i(sh);
            h8v hi, lo;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float y = ok ? v[j] * sc : 0.0f;
                const _Float16 t = (_Float16)y;
                hi[j] = t;
                lo[j] = (_Float16)(y - (float)t);
            }
            uint8_t *o = a.hp + (uint64_t)pr * PF_PITCH(768) + (ks >> 1) * 128 + (ks & 1) * 64 + hh * 16;
            *reinterpret_cast<uint4 *>(o) = __builtin_bit_cast(uint4, hi);
            *reinterpret_cast<uint4 *>(o + 32) = __builtin_bit_cast(uint4, lo);
            if (c == 0) a.hs[(uint64_t)pr * 8 + cg] = ok ? exp2i(-sh) : __builtin_nanf("");
        }
    }
}

// ---------------------------------------------------------------- down weights
template <int F> struct DnHalf;                                             // the lane's part of a half block (128 values)
template <> struct DnHalf<FMT_IQ3> { uint4 q; uint2 aux; uint32_t d; };     // 16 grid bytes, signs and scales
template <> struct DnHalf<FMT_IQ3S> { uint4 q; uint2 sg; uint32_t qh, sc, d; };   // 16 grid bytes, 8 sign bytes, high bits, scales
template <> struct DnHalf<FMT_IQ4> { uint2 q[4]; uint2 m; };                // 8 bytes of each of the half's sub-blocks, meta
DEV void dn_load(DnHalf<FMT_IQ3> &w, const PfMat &m, uint32_t bi, int half, int h) {
    w.q = ldu128(m.qs + bi * 64u + 32 * half + 16 * h);
    w.aux = ldu64(m.p1 + bi * 32u + 16 * half + 8 * h);
    w.d = ldu16(m.d + bi);
}
DEV void dn_load(DnHalf<FMT_IQ3S> &w, const PfMat &m, uint32_t bi, int half, int h) {
    w.q = ldu128(m.qs + bi * 64u + 32 * half + 16 * h);
    w.sg = ldu64(m.p1 + bi * 32u + 16 * half + 8 * h);
    w.qh = ldu16(m.p2 + bi * 16u + 4 * half + 2 * h);
    w.sc = m.p2[bi * 16u + 8 + 2 * half + h];
    w.d = ldu16(m.d + bi);
}
DEV void dn_load(DnHalf<FMT_IQ4> &w, const PfMat &m, uint32_t bi, int half, int h) {
#pragma unroll
    for (int i = 0; i < 4; ++i) w.q[i] = ldu64(m.qs + bi * 128u + 64 * half + 16 * i + 8 * h);
    w.m = ldu64(m.p1 + bi * 8u);
}
// k-step s of the half: entry s of the lane's 8 (sub-block s / 4 of its two)
// IQ3_XXS (src/qx_format.c:1935-1959)
DEV Codes dn_look(const DnHalf<FMT_IQ3> &w, int s, const uint32_t *grid, const uint2 *sgn) {
    return Codes{grid[byte_at(w.q, 2 * s)], grid[byte_at(w.q, 2 * s + 1)], sgn[((s < 4 ? w.aux.x : w.aux.y) >> (7 * (s & 3))) & 127u]};
}
DEV h2v dn_mul(const DnHalf<FMT_IQ3> &w, int sub) { return odd_mul((sub ? w.aux.y : w.aux.x) >> 28); }
// IQ3_S (src/qx_format.c:1986-2030): high index bits in qh, explicit sign bytes, nibble scales
DEV Codes dn_look(const DnHalf<FMT_IQ3S> &w, int s, const uint32_t *grid, const uint2 *sgn) {
    const uint32_t i0 = byte_at(w.q, 2 * s) | (((w.qh >> (2 * s)) & 1u) << 8);
    const uint32_t i1 = byte_at(w.q, 2 * s + 1) | (((w.qh >> (2 * s + 1)) & 1u) << 8);
    return Codes{grid[i0], grid[i1], sgn[((s < 4 ? w.sg.x : w.sg.y) >> (8 * (s & 3))) & 255u]};
}
DEV h2v dn_mul(const DnHalf<FMT_IQ3S> &w, int sub) { return odd_mul((w.sc >> (4 * sub)) & 15u); }
// IQ4_XS (src/qx_format.c:2032-2053): a byte is the codes of values j and 16 + j of a sub-block
DEV Codes dn_look(const DnHalf<FMT_IQ4> &w, int s, const uint32_t *kv2, const uint2 *) {
    const uint32_t q = s & 1 ? w.q[s >> 1].y : w.q[s >> 1].x;
    return Codes{kv2[q & 255u], kv2[(q >> 8) & 255u], make_uint2(kv2[(q >> 16) & 255u], kv2[q >> 24])};
}
DEV h2v dn_mul(const DnHalf<FMT_IQ4> &, int) { return h2v{0, 0}; }
DEV float dn_scale(const DnHalf<FMT_IQ3> &w, int, int) { return fp16_exact(w.d) * (0.25f * CODE_SCALE); }
DEV float dn_scale(const DnHalf<FMT_IQ3S> &w, int, int) { return fp16_exact(w.d) * CODE_SCALE; }
DEV float dn_scale(const DnHalf<FMT_IQ4> &w, int half, int i) {   // sub-block i of the half
    const int ib = 4 * half + i;
    const uint32_t sh = w.m.x >> 16, sl = (w.m.y >> (8 * (ib >> 1))) & 255u;
    const int ls = (int)(((sl >> (4 * (ib & 1))) & 15u) | (((sh >> (2 * ib)) & 3u) << 4));
    return fp16_exact(w.m.x & 0xffffu) * (float)(ls - 32);
}

template <int F, int R>
DEV void dn_pass(const PfExperts &a, uint32_t e, uint32_t cg, uint32_t m0, uint32_t n, const uint32_t *grid,
                 const uint2 *sgn, uint4 *buf, uint32_t *s_pair, float *s_hs) {
    constexpr int MT = R > 32 ? 2 : 1, NR = R > 16 ? 16 : 8;   // tiles; result registers of a tile, hi and lo added
    // half blocks loaded at once: both where the registers allow it (read apart, a block's lines came
    // twice from beyond L2: 98 MB for 47 of weights; IQ4_XS has whole lines per half)
    constexpr int NH = MT == 1 && F != FMT_IQ4 ? 2 : 1;
    constexpr bool PER32 = F == FMT_IQ4;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), h = lane >> 5, col = lane & 31;
    uint32_t bi[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) bi[f] = (e * 2048u + 256 * cg + 64 * wave + 32 * f + col) * 3;
    DnHalf<F> cur[2][NH], nxt[2][NH];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int i = 0; i < NH; ++i) dn_load(cur[f][i], a.w[2], bi[f], i, h);
    if (wave == 0) pass_pairs<R>(a, e, m0, n, s_pair);
    __syncthreads();   // the pairs, and the tables
    uint32_t off[R / 8];
    stage_offsets<R, 0>(off, s_pair, PF_PITCH(768), lane);
    stage_rows<R>(a.hp, off, 0, buf, wave);
    const ALane at = a_lane<R>(lane);
    for (int i = tid; i < 6 * R; i += 256)   // the rows' scales of each 128 values
        s_hs[i] = a.hs[(uint64_t)s_pair[i % R] * 8 + i / R];
    f16x acc[2][MT];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[f][mt] = zero16();
#pragma unroll 1
    for (int st0 = 0; st0 < 6; st0 += NH)
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
        const int st = st0 + hf;
        wait_loads<0>();
        __syncthreads();   // stage st is in; every wave is past stage st - 1
        const int sn = st < 5 ? st + 1 : 5;
        if (st < 5) stage_rows<R>(a.hp, off, 4 * sn, buf + (sn & 1) * STAGE<R>, wave);
        if (NH == 1 || hf == 0)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int i = 0; i < NH; ++i)
                    dn_load(nxt[f][i], a.w[2], bi[f] + (NH == 1 ? sn >> 1 : min(st / 2 + 1, 2)), NH == 1 ? sn & 1 : i, h);
        const uint4 *sb = buf + (st & 1) * STAGE<R>;
        f16x G[2][MT];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) G[f][mt] = zero16();
        // the column's scale (of the block or of sub-block i) times the rows' scales, onto acc
        auto flush = [&](int f, int i) {
            const float d = dn_scale(cur[f][hf], st & 1, i);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int q = 0; q < NR / 4; ++q) {
                    const f4x hsr = *reinterpret_cast<const f4x *>(s_hs + st * R + 32 * mt + 8 * q + 4 * h);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int k = 4 * q + r;
                        acc[f][mt][k] = fmaf(d * hsr[r], R > 16 ? G[f][mt][k] : G[f][mt][k] + G[f][mt][(k + 8) & 15], acc[f][mt][k]);
                        if (PER32) {
                            G[f][mt][k] = 0.0f;
                            if (R == 16) G[f][mt][(k + 8) & 15] = 0.0f;
                        }
                    }
                }
        };
        auto form = [&](const Codes &c, int f, int s) {
            return PER32 ? make_uint4(c.m0, c.m1, c.sg.x, c.sg.y) : conv(c, dn_mul(cur[f][hf], s >> 2));
        };
        Codes c1 = dn_look(cur[1][hf], 0, grid, sgn);
        uint4 ah[MT], al[MT];
        a_read<R, MT>(ah, al, sb, at, 0);
        uint4 b = form(dn_look(cur[0][hf], 0, grid, sgn), 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int s = i >> 1, f = i & 1;
            uint4 bn = b, nh[MT], nl[MT];
            if (i < 15) bn = form(c1, (i + 1) & 1, (i + 1) >> 1);
            if (i < 14) c1 = dn_look(cur[f][hf], s + 1, grid, sgn);
            if (f == 1 && s < 7) a_read<R, MT>(nh, nl, sb, at, s + 1);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) G[f][mt] = mfma(ah[mt], b, G[f][mt]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) if (R > 16) G[f][mt] = mfma(al[mt], b, G[f][mt]);
            if (PER32 && (s & 1)) flush(f, s >> 1);
            b = bn;
            if (f == 1 && s < 7) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) { ah[mt] = nh[mt]; al[mt] = nl[mt]; }
            }
        }
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            if (!PER32) flush(f, 0);
            if (hf == NH - 1)
#pragma unroll
                for (int i = 0; i < NH; ++i) cur[f][i] = nxt[f][i];
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const uint32_t row = 32 * mt + 8 * (r >> 2) + 4 * h + (r & 3);
            if (row >= n) continue;
            float *o = a.y + (uint64_t)s_pair[row] * 2048 + 256 * cg + 64 * wave + col;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const float y = acc[f][mt][r];
                o[32 * f] = isfinite(y) ? y : 0.0f;   // (src/qx_format.c:4284)
            }
        }
}
}  // namespace

namespace {
// The work items are (expert, pass) pairs in expert order: an expert with c pairs has
// ceil(c / R) passes of evenly many row tiles (real prompts crowd onto a few experts: every
// pass is its own workgroup, so one expert's passes run side by side).  Every wave finds its
// workgroup's item from the 128 counts (two a lane, a scan over the wave).
template <int R>
DEV bool expert_item(const uint32_t *cnt, uint32_t item, uint32_t &e, uint32_t &m0, uint32_t &n) {
    const int lane = threadIdx.x & 63;
    const uint2 c = reinterpret_cast<const uint2 *>(cnt)[lane];   // (zero past the last expert)
    const uint32_t p0 = (c.x + R - 1) / R, p1 = (c.y + R - 1) / R;
    const uint32_t incl = wave_prefix(p0 + p1);
    const uint64_t past = __ballot(incl > item);
    if (!past) return false;
    const int l = __builtin_ctzll(past);
    const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)(incl - p0 - p1), l);
    const uint32_t q0 = (uint32_t)__builtin_amdgcn_readlane((int)p0, l), q1 = (uint32_t)__builtin_amdgcn_readlane((int)p1, l);
    const bool second = item - before >= q0;
    const uint32_t cc = (uint32_t)__builtin_amdgcn_readlane((int)(second ? c.y : c.x), l);
    const uint32_t pass = item - before - (second ? q0 : 0u), passes = second ? q1 : q0;
    const uint32_t tiles = (cc + 31) / 32, rows = (tiles + passes - 1) / passes * 32;
    e = 2u * l + second;
    m0 = pass * rows;
    n = m0 < cc ? min(rows, cc - m0) : 0u;
    return n != 0;
}
}  // namespace

// Workgroup L of the grid (XCD L % 8, round-robin): the column groups of an item run on one
// XCD, so the item's gathered rows are fetched into one L2.
#define EXPERT_TILE(GROUPS, R)                                                                     \
    const uint32_t j_ = blockIdx.x >> 3, cg = j_ % (GROUPS);                                       \
    uint32_t e, m0, n;                                                                             \
    if (!expert_item<R>(a.cnt, (j_ / (GROUPS)) * 8 + (blockIdx.x & 7u), e, m0, n)) return;

// Rows of a pass.  Gate/up takes 32: its about 16 vector instructions per 8 codes do not hide behind the
// matrix instructions of another tile, and twice the workgroups fill the chip (512 tokens of a
// prompt 81 us with 64 rows, 80 with 32; 149 tokens 66 and 55; 128 random rows 58 and 53; 64 rows of one
// expert each 37 and 27).  At most 16 pairs run as one tile of hi and lo rows, half the matrix
// work (128 random rows, 8 pairs an expert: 69 -> 58 us).
constexpr int GU_ROWS = 32;
template <int F>
__global__ __launch_bounds__(256, 2) void qxp_gate_up(PfExperts a, PfTables P) {
    EXPERT_TILE(6u, GU_ROWS)
    constexpr int NG = F == FMT_IQ2 ? 512 : 1024, NS = F == FMT_IQ2 ? 128 : 256;
    __shared__ uint2 s_grid[NG], s_sgn[NS];
    __shared__ uint4 s_buf[2 * STAGE<GU_ROWS>];   // two stages; the epilogue's rows of 132 floats
    __shared__ uint32_t s_pair[GU_ROWS];
    __shared__ float s_xs[GU_ROWS];
    for (int i = threadIdx.x; i < NG; i += 256) s_grid[i] = (F == FMT_IQ2 ? P.g2 : P.g2s)[i];
    for (int i = threadIdx.x; i < NS; i += 256) s_sgn[i] = (F == FMT_IQ2 ? P.sg7 : P.sg8)[i];
    if (n <= 16) gu_pass<F, 16>(a, e, cg, m0, n, s_grid, s_sgn, s_buf, s_pair, s_xs);
    else gu_pass<F, 32>(a, e, cg, m0, n, s_grid, s_sgn, s_buf, s_pair, s_xs);
}

// Down takes up to R = 32 or 64 (see down_rows)
template <int F, int R>
__global__ __launch_bounds__(256, 2) void qxp_down(PfExperts a, PfTables P) {
    EXPERT_TILE(8u, R)
    constexpr int NG = F == FMT_IQ3S ? 512 : 256, NS = F == FMT_IQ3 ? 128 : F == FMT_IQ3S ? 256 : 1;
    __shared__ uint32_t s_grid[NG];
    __shared__ uint2 s_sgn[NS];
    __shared__ uint4 s_buf[2 * STAGE<R>];
    __shared__ uint32_t s_pair[R];
    __shared__ float s_hs[6 * R];
    for (int i = threadIdx.x; i < NG; i += 256) s_grid[i] = (F == FMT_IQ3 ? P.g3 : F == FMT_IQ3S ? P.g3s : P.kv2)[i];
    if (NS > 1) for (int i = threadIdx.x; i < NS; i += 256) s_sgn[i] = (F == FMT_IQ3 ? P.sg7 : P.sg8)[i];
    if (n <= 16) dn_pass<F, 16>(a, e, cg, m0, n, s_grid, s_sgn, s_buf, s_pair, s_hs);
    else if (n <= 32) dn_pass<F, 32>(a, e, cg, m0, n, s_grid, s_sgn, s_buf, s_pair, s_hs);
    else if constexpr (R == 64) dn_pass<F, 64>(a, e, cg, m0, n, s_grid, s_sgn, s_buf, s_pair, s_hs);
}

extern "C" {
// gate/up (IQ2_XS or IQ2_S) and down (IQ3_XXS, IQ3_S or IQ4_XS) of T tokens; the grid holds
// the most items T tokens can make with R rows a pass
static uint32_t item_bound(const PfExperts &a, uint32_t T, uint32_t R) {
    const uint32_t pairs = T * QXG_TOPK, most = pairs / R + (a.experts < pairs ? a.experts : pairs);
    return (most + 7) / 8 * 8;
}
void qxp_launch_gate_up(hipStream_t s, uint32_t type, const PfExperts &a, const PfTables &P, uint32_t T, Timer tm) {
    const dim3 grid(6 * item_bound(a, T, GU_ROWS));
    if (type == 22) qx_launch(qxp_gate_up<FMT_IQ2S>, grid, dim3(256), 0, s, tm, a, P);
    else qx_launch(qxp_gate_up<FMT_IQ2>, grid, dim3(256), 0, s, tm, a, P);
}
// Rows of down's passes: with up to 128 tokens, 32 spread a crowded expert over more workgroups (64 rows
// of one expert each 20 -> 16 us, 37 tokens of a mixed model 20.6 -> 17.8); with more tokens the chip
// is full and two tiles share the codes (300 tokens 33.6 us, 37.7 with 32 rows).  Between them, random
// rows over 128 experts, launch included, 32 rows against 64 in IQ3_XXS, IQ4_XS and IQ3_S: 96 tokens
// 36.7/37.3, 47.4/45.3, 42.9/44.2 us; 128 tokens 37.6/37.7, 49.9/46.0, 43.5/47.1; 149 tokens 37.7/37.8,
// 48.1/45.7, 51.0/47.8; 220 tokens 39.8/41.2, 54.2/52.1, 53.4/51.7.  (What counts is pairs an expert:
// with 32 experts 64 rows win from 96 tokens on, 128 tokens 23.0/21.8.)  With 64 rows IQ4_XS spills 7
// registers and IQ3_XXS one.
static uint32_t down_rows(uint32_t T) { return T <= 128 ? 32 : 64; }
void qxp_launch_down(hipStream_t s, uint32_t type, const PfExperts &a, const PfTables &P, uint32_t T, Timer tm) {
    const uint32_t R = down_rows(T);
    const dim3 grid(8 * item_bound(a, T, R));
    auto *k = type == 21 ? (R == 32 ? qxp_down<FMT_IQ3S, 32> : qxp_down<FMT_IQ3S, 64>)
              : type == 23 ? (R == 32 ? qxp_down<FMT_IQ4, 32> : qxp_down<FMT_IQ4, 64>)
                           : (R == 32 ? qxp_down<FMT_IQ3, 32> : qxp_down<FMT_IQ3, 64>);
    qx_launch(k, grid, dim3(256), 0, s, tm, a, P);
}
}
