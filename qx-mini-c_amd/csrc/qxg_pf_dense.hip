// Dense GEMMs of the batched prefill (CDNA4, gfx950): Q/K/V and the O projection.
//
// Weights.  qxp_dense_plane lays a matrix out once, before the first batched prefill of a bound
// model: one byte per weight, its integer code + 128 (IQ4_XS kvalue, Q5_K 5-bit code), in the order
// the matrix instruction reads, [32-row tile][line of 32 K][lane][16 codes], and per row and 32 values
// the f32 scale (d * (ls - 32) or d * sc) and, for Q5_K, the offset dmin * m: 1.13 or 1.25 bytes a
// weight, 21.2 to 23.6 MB a layer.  A code becomes fp16 as bits(1024 + byte) - 1152, two a v_perm and
// v_pk_add.  From the file's nibbles the same codes took a random LDS read per byte, for every
// row tile again, which bounded the kernel (56 us for Q/K/V and 49 for O of 512 tokens, now 36 and 27; 25 and
// 48 of 37, now 10 and 9).  The matrix instructions bound it, about 20 us of the 36.
//
// Tiles.  A workgroup takes up to 64 rows x 128 columns (4 waves of 32 columns) over a run of K;
// the rows are staged in LDS, the codes go straight to registers.  The matrix cores sum 32
// values of K in f32 (hi and lo), that sum times the scale joins the f32 accumulators, less the
// offset times the row's sum over the same 32 values (packed with the row).  K is split over
// gridDim.z so that about 320 workgroups run whatever the number of rows (two fit a CU): the
// consumers add the parts, [part][row][column], in order.
#include "qxg_pf.h"

namespace {
DEV uint32_t biased2(uint32_t q, uint32_t sel) {   // two biased bytes to fp16 codes
    const h2v k = {(_Float16)1152.0f, (_Float16)1152.0f};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2v, perm(0x64646464u, q, sel)) - k);
}
DEV uint4 biased8(uint32_t x, uint32_t y) {
    return make_uint4(biased2(x, 0x04010400u), biased2(x, 0x04030402u), biased2(y, 0x04010400u), biased2(y, 0x04030402u));
}
struct DnsStage { uint4 q[4]; float4 sc, of; };   // four lines of the lane's column
template <bool OFS>
DEV void dns_load(DnsStage &w, const PfDense &g, uint32_t ct, uint32_t line, int lane, bool ofs) {
    const uint8_t *q = g.codes + ((uint64_t)ct * g.lines + line) * 1024 + 16 * lane;
#pragma unroll
    for (int i = 0; i < 4; ++i) w.q[i] = *reinterpret_cast<const uint4 *>(q + 1024 * i);
    const uint64_t at = ((uint64_t)ct * g.lines + line) * 32 + 4 * (lane & 31);
    w.sc = *reinterpret_cast<const float4 *>(g.scale + at);
    if (OFS && ofs) w.of = *reinterpret_cast<const float4 *>(g.ofs + at);
}

template <int MT, bool OFS>
DEV void dns_tile(const PfDense &g, uint4 *buf, float *s_sum) {
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), h = lane >> 5, col = lane & 31;
    const uint32_t ct = blockIdx.x * 4 + wave, row0 = blockIdx.y * (32 * MT);
    const uint32_t l0 = blockIdx.z * g.part_lines, stages = g.part_lines / 4;
    // (wave-uniform: the matrices meet at multiples of 32 columns)
    const bool ofs = OFS && ((g.ofs_segs >> (ct >= g.seg2 ? 2 : ct >= g.seg1 ? 1 : 0)) & 1u);
    uint32_t off[4 * MT];
#pragma unroll
    for (int i = 0; i < 4 * MT; ++i)
        off[i] = min(row0 + 8 * i + (lane >> 3), g.rows - 1) * g.row_bytes + stage_chunk(i, lane);
    const uint32_t srow = min(row0 + (uint32_t)(tid & (32 * MT - 1)), g.rows - 1);
    auto stage = [&](uint32_t st) {
        stage_rows<32 * MT>(g.rows_packed, off, l0 + 4 * st, buf + (st & 1) * STAGE<32 * MT>, wave);
    };
    // the rows' sums of the stage's four lines, for the offsets
    auto load_sum = [&](uint32_t st) {
        return tid < 4 * 32 * MT ? g.sums[(uint64_t)srow * g.lines + l0 + 4 * st + tid / (32 * MT)] : 0.0f;
    };
    DnsStage cur, nxt;
    dns_load<OFS>(cur, g, ct, l0, lane, ofs);
    stage(0);
    float sum = OFS ? load_sum(0) : 0.0f;
    const ALane at = a_lane<32 * MT>(lane);
    f16x acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = zero16();
#pragma unroll 1
    for (uint32_t st = 0; st < stages; ++st) {
        if (OFS && tid < 4 * 32 * MT) s_sum[(st & 1) * 4 * ROWS + (tid / (32 * MT)) * ROWS + (tid & (32 * MT - 1))] = sum;
        wait_loads<0>();
        __syncthreads();   // the stage is in; every wave is past the one before
        const uint32_t sn = st + 1 < stages ? st + 1 : st;
        if (sn != st) stage(sn);
        dns_load<OFS>(nxt, g, ct, l0 + 4 * sn, lane, ofs);
        if (OFS) sum = load_sum(sn);
        const uint4 *sb = buf + (st & 1) * STAGE<32 * MT>;
        // line l's sums times the column's scale, less its offset times the rows' sums
        auto add = [&](f16x (&acc)[MT], const f16x (&G)[MT], int l) {
            const float sc = l == 0 ? cur.sc.x : l == 1 ? cur.sc.y : l == 2 ? cur.sc.z : cur.sc.w;
            const float of = l == 0 ? cur.of.x : l == 1 ? cur.of.y : l == 2 ? cur.of.z : cur.of.w;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[mt][r] = fmaf(sc, G[mt][r], acc[mt][r]);
            if (OFS && ofs) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const f4x s = *reinterpret_cast<const f4x *>(s_sum + (st & 1) * 4 * ROWS + l * ROWS + 32 * mt + 8 * q + 4 * h);
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[mt][4 * q + r] = fmaf(-of, s[r], acc[mt][4 * q + r]);
                    }
            }
        };
        // a line's rows are read while the line before is multiplied, and a line's sums join the
        // accumulators behind the next line's products: one wave a SIMD has to overlap both itself
        uint4 ah[2][MT], al[2][MT], nh[2][MT], nl[2][MT];
        a_read<32 * MT, MT>(ah[0], al[0], sb, at, 0);
        a_read<32 * MT, MT>(ah[1], al[1], sb, at, 1);
        f16x P[MT];   // the previous line's sums, still unscaled
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            if (l < 3) {
                a_read<32 * MT, MT>(nh[0], nl[0], sb, at, 2 * l + 2);
                a_read<32 * MT, MT>(nh[1], nl[1], sb, at, 2 * l + 3);
            }
            __builtin_amdgcn_sched_barrier(0);
            const uint4 b0 = biased8(cur.q[l].x, cur.q[l].y), b1 = biased8(cur.q[l].z, cur.q[l].w);
            f16x G[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) G[mt] = mfma(ah[0][mt], b0, zero16());
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) G[mt] = mfma(al[0][mt], b0, G[mt]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) G[mt] = mfma(ah[1][mt], b1, G[mt]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) G[mt] = mfma(al[1][mt], b1, G[mt]);
            if (l) add(acc, P, l - 1);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) P[mt] = G[mt];
            if (l < 3) {
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) { ah[k][mt] = nh[k][mt]; al[k][mt] = nl[k][mt]; }
            }
        }
        add(acc, P, 3);
        cur = nxt;
    }
    // through LDS, so that a row's 128 columns leave as 16-byte stores
    __syncthreads();
    float *o = reinterpret_cast<float *>(buf);
    constexpr int LD = 132;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[(32 * mt + 8 * (r >> 2) + 4 * h + (r & 3)) * LD + 32 * wave + col] = acc[mt][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4 * MT; ++i) {
        const uint32_t r = 8 * i + (tid >> 5), row = row0 + r;
        if (row >= g.rows) continue;
        const float rs = g.rscale[row];
        const float4 v = *reinterpret_cast<const float4 *>(o + r * LD + 4 * (tid & 31));
        *reinterpret_cast<float4 *>(g.out + ((uint64_t)blockIdx.z * g.rows + row) * g.cols + 128 * blockIdx.x + 4 * (tid & 31)) =
            make_float4(v.x * rs, v.y * rs, v.z * rs, v.w * rs);
    }
}

template <int MT, bool OFS>
__global__ __launch_bounds__(256, 2) void qxp_dense(PfDense g) {
    __shared__ uint4 s_buf[2 * STAGE<32 * MT>];
    __shared__ float s_sum[OFS ? 2 * 4 * ROWS : 1];
    dns_tile<MT, OFS>(g, s_buf, s_sum);
}
}  // namespace

// One matrix (repacked IQ4_XS or Q5_K planes, K = 32 * lines) as the dense layout, from 32-row
// tile ct0 on; thread per row and line.  Decoding as src/qx_format.c:2032-2053 and 2112-2145.
extern "C" __global__ __launch_bounds__(256) void qxp_dense_plane(uint32_t type, const uint8_t *qs, const uint8_t *meta,
        const uint8_t *qh, uint32_t rows, uint32_t lines, uint32_t ct0, uint8_t *codes, float *scale, float *ofs) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * lines) return;
    const uint32_t r = i / lines, line = i % lines, ib = line & 7u;
    const uint64_t bi = (uint64_t)r * (lines / 8) + (line >> 3);
    uint8_t c[32];
    float sc, of = 0.0f;
    if (type == 23) {
        const uint2 m = *reinterpret_cast<const uint2 *>(meta + bi * 8);
        const uint32_t sh = m.x >> 16, sl = (m.y >> (8 * (ib >> 1))) & 255u;
        const int ls = (int)(((sl >> (4 * (ib & 1))) & 15u) | (((sh >> (2 * ib)) & 3u) << 4));
        sc = fp16_exact(m.x & 0xffffu) * (float)(ls - 32);
        for (int j = 0; j < 16; ++j) {
            const uint8_t q = qs[bi * 128 + 16 * ib + j];
            c[j] = (uint8_t)(KV[q & 15] + 128);
            c[16 + j] = (uint8_t)(KV[q >> 4] + 128);
        }
    } else {
        const uint4 m = *reinterpret_cast<const uint4 *>(meta + bi * 16);
        auto sb = [&](int k) { return ((k < 4 ? m.y : k < 8 ? m.z : m.w) >> (8 * (k & 3))) & 255u; };
        uint32_t s6, m6;   // get_scale_min_k4, src/qx_format.c:2079-2087
        if (ib < 4) { s6 = sb(ib) & 63u; m6 = sb(ib + 4) & 63u; }
        else { s6 = (sb(ib + 4) & 15u) | ((sb(ib - 4) >> 6) << 4); m6 = (sb(ib + 4) >> 4) | ((sb(ib) >> 6) << 4); }
        sc = fp16_exact(m.x & 0xffffu) * (float)s6;
        of = fp16_exact(m.x >> 16) * (float)m6;
        for (int j = 0; j < 32; ++j) {
            const uint32_t q = qs[bi * 128 + 32 * (ib >> 1) + j];
            c[j] = (uint8_t)((((ib & 1) ? q >> 4 : q & 15u) | (((qh[bi * 32 + j] >> ib) & 1u) << 4)) + 128u);
        }
    }
    const uint32_t ct = ct0 + r / 32, col = r & 31;
    uint8_t *o = codes + ((uint64_t)ct * lines + line) * 1024 + 16 * col;
    for (int t = 0; t < 2; ++t)
        for (int h = 0; h < 2; ++h)
            for (int j = 0; j < 8; ++j) o[512 * h + 8 * t + j] = c[16 * t + 8 * h + j];
    // scales: [tile][line / 4][column][line % 4]
    const uint64_t at = ((uint64_t)ct * lines + (line & ~3u)) * 32 + 4 * col + (line & 3u);
    scale[at] = sc;
    if (ofs) ofs[at] = of;
}

extern "C" void qxp_launch_dense(hipStream_t s, const PfDense &g, uint32_t parts, Timer tm) {
    const uint32_t gx = g.cols / 128;
    if (g.rows > 32) {
        const dim3 grid(gx, (g.rows + 63) / 64, parts);
        if (g.ofs_segs) qx_launch(qxp_dense<2, true>, grid, dim3(256), 0, s, tm, g);
        else qx_launch(qxp_dense<2, false>, grid, dim3(256), 0, s, tm, g);
    } else {
        const dim3 grid(gx, 1, parts);
        if (g.ofs_segs) qx_launch(qxp_dense<1, true>, grid, dim3(256), 0, s, tm, g);
        else qx_launch(qxp_dense<1, false>, grid, dim3(256), 0, s, tm, g);
    }
}
