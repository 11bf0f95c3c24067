// Shared by the prefill's GEMMs: the matrix instruction, the packed activation rows and their
// staging.  Header-only (internal linkage).
//
// Tiles.  v_mfma_f32_32x32x16_f16: lane l holds, for A, row l%32 and, for B, column l%32,
// each 8 values of K at lane half h = l/32; result register r of lane l is row
// 8*(r/4) + 4*h + r%4, column l%32.  (With one wave on a SIMD the 16x16x32 form reaches 1.2
// PFLOP/s here, this one 1.6.)  Rows are tokens or pairs, columns weight rows.
//
// Packed rows.  A row of K values is K / 32 lines of 128 bytes: line k / 2 holds k-steps k and
// k + 1, [k % 2][hi, lo][h][8 fp16].
//
// Staging.  A stage is four lines of a workgroup's rows, copied to LDS by load-to-LDS
// instructions of 8 rows x one whole line; the 16-byte chunk c of row r lies at place
// c ^ (r / 2 % 8) of its line, so 16 rows' chunks (two rows span the 64 banks) lie in 16
// different bank groups: a column-wise read takes 4 cycles (with c ^ (r % 8) it took 8).
#pragma once
#include "qxg_dev.h"

namespace {
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f4x __attribute__((ext_vector_type(4)));
typedef float f16x __attribute__((ext_vector_type(16)));

DEV f16x mfma(uint4 a, uint4 b, f16x c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, a), __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}
DEV f16x zero16() {
    f16x z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}
// lane i's 16 bytes at base + off land at lds + 16 i (lds the same in every lane).  The copy needs one
// wait state after the write of M0 and five after a vector instruction (readfirstlane) that wrote
// its base; the compiler adds none inside the assembly.
DEV void dma16(const void *base, uint32_t off, const void *lds) {
    const uint32_t l = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)lds);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(l) : "memory", "m0");
}
// waits until at most N of the wave's loads (the youngest) are outstanding
template <int N>
DEV void wait_loads() {
    static_assert(N < 16, "the wait's low counter bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | N);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

constexpr int RT = 2;                    // 32-row tiles of a workgroup, at most
constexpr int ROWS = 32 * RT;
template <int R> constexpr int STAGE = 4 * R * 8;   // uint4 per stage of R rows: 4 lines of 8 chunks a row

// The four lines from line0 on of the workgroup's rows: wave w copies line w, 8 rows an
// instruction; off[i] is the lane's row 8 i + lane / 8 and its chunk of the line.
template <int R>
DEV void stage_rows(const void *rows, const uint32_t (&off)[R / 8], uint32_t line0, uint4 *buf, int wave) {
#pragma unroll
    for (int i = 0; i < R / 8; ++i) dma16(rows, off[i] + (line0 + wave) * 128, buf + (wave * R + 8 * i) * 8);
}
// byte offset in its line of the chunk that lane copies in instruction i
DEV uint32_t stage_chunk(int i, int lane) { return ((lane ^ (4 * i + (lane >> 4))) & 7) << 4; }
// of the rows of pairs s_pair[], a row for 2^SHIFT pairs
template <int R, int SHIFT>
DEV void stage_offsets(uint32_t (&off)[R / 8], const uint32_t *s_pair, uint32_t row_bytes, int lane) {
#pragma unroll
    for (int i = 0; i < R / 8; ++i) off[i] = (s_pair[8 * i + (lane >> 3)] >> SHIFT) * row_bytes + stage_chunk(i, lane);
}
// A fragments of k-step s of the stage: lane's row l%32 of each tile, lane half l/32.  Of 16
// rows there is one fragment, tile rows 0 .. 15 their hi and 16 .. 31 their lo halves: one
// matrix instruction does both products, and register r + 8 of a result is the lo part of r's.
struct ALane { uint32_t at[4]; };   // byte offset of chunk 2 i + h in the lane's row of line 0
template <int R>
DEV ALane a_lane(int lane) {
    ALane a;
    const int row = lane & (R == 16 ? 15 : 31), lo = R == 16 ? (lane >> 4) & 1 : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) a.at[i] = row * 128 + ((((2 * (i | lo) + (lane >> 5)) ^ (row >> 1)) & 7) << 4);
    return a;
}
template <int R, int MT>
DEV void a_read(uint4 (&ah)[MT], uint4 (&al)[MT], const uint4 *buf, const ALane &a, int s) {
    const uint8_t *p = reinterpret_cast<const uint8_t *>(buf) + (s >> 1) * (R * 128);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        ah[mt] = *reinterpret_cast<const uint4 *>(p + mt * 4096 + a.at[2 * (s & 1)]);
        if (R > 16) al[mt] = *reinterpret_cast<const uint4 *>(p + mt * 4096 + a.at[2 * (s & 1) + 1]);
    }
}
}  // namespace
