// q4k_mfma.h -- the Q4_K GEMV for several activation columns on the matrix
// cores: v_mfma_i32_16x16x64_i8 forms the int32 sub-block sums of a tile of
// 16 weight rows against up to 8 columns, the VALU only unpacks nibbles and
// applies the per-(row, column, sub-block) scales.
//
// Operands of one MFMA.  Product m = 2h + p of super-block kb takes the low
// (p = 0) or high (p = 1) nibbles of qs bytes [64h, 64h + 64) of each row,
// i.e. sub-blocks 4h + p and 4h + 2 + p.  The instruction's 64 k-slots are
// lane group g = lane/16, byte t; A row i and B column j of lane l are
// l % 16, and D element v of lane l is D[4(l/16) + v][l % 16] (checked on the
// device).  Here
//   k-slots   lane group g: the 16 nibbles of bytes [64h + 16g, +16): g = 0, 1
//             sub-block 4h + p, g = 2, 3 sub-block 4h + 2 + p;
//   A row i   activation column i % 8 for sub-block 4h + p (i < 8) or
//             4h + 2 + p (i >= 8): its q8 in the slots of its own sub-block,
//             zeros in the other two lane groups (read from a zero area of
//             LDS);
//   B col r   weight row r of the tile.  A lane's 16 bytes serve two
//             products, so it reads 32 of the row's 128 qs bytes;
//   D         D[i][r] = the int32 sum S_qq of row r, column i % 8, sub-block
//             4h + p + 2(i/8): every output is one the product needs.
// So lane l ends up with one weight row (l % 16), one sub-block parity
// (hid = l / 32: sub-blocks 2hid, 2hid + 1, 4 + 2hid, 5 + 2hid) and four
// columns (4((l/16) & 1) + v): the row's scales are unpacked once per lane
// and used for four columns.  The products start from 1.5 * 2^23 as an
// integer, so their bits read as a float are 1.5 * 2^23 + S, and one fma with
// (sc, -1.5 * 2^23 * sc) gives sc * S, exact: no conversion.
//
// The min term of a super-block, the sum over its sub-blocks s of
// m_s * (d8 sum q8)_s, is a product over s, so it runs on the f32 matrix
// instruction 16x16x4 (a fused multiply-add per k in 32 bits), twice: A row
// i, lane group g: d8 * sum of the q8 of column i % 8, block {0, 1, 4, 5}[g] +
// 2(i/8); B col r: m of row r, of blocks {0, 1, 4, 5}[g] (first product, A's
// rows i >= 8 zero) and {2, 3, 6, 7}[g] (second, the rows i < 8 zero).  So a
// lane gets the min sums of its own four sub-blocks, as it gets their S.
//
// Work split: tiles of 16 rows, split evenly over the workgroups (one per
// CU, 8 or, by override, 16 waves).  The waves of a workgroup form groups of KS
// (8/KS groups of 8 waves); in
// each round every group takes one tile and its KS waves take equal shares
// of the tile's super-blocks.  At the end of a round each wave leaves its
// partial results in LDS and, after a barrier, the workgroup combines the KS
// partials of each tile and writes the outputs.
//
// A operand from the Q8_1 buffer (GA variants, pre-quantised activation):
// instead of an LDS copy of the whole activation, each item's activation --
// super-block kb of the NC columns, 8 AoS block_q8_1 of 36 bytes (288
// contiguous bytes) per column -- arrives with the item's weights, in three
// 64-lane x 16-byte loads (chunk c = lane + 64i is bytes [16 (c % 18), +16)
// of column c / 18), goes to a second LDS slot of the wave as it lies in
// memory, and the MFMA lanes read their A operands from there.  The LDS
// holds only the d8 of every (block, column) besides, so the length of the
// rows is not bounded by the LDS (staged, eight columns end at 14336 values,
// 163456 of its 163840 bytes).  The sums of the blocks' q8, which the staged
// layout keeps times d8, come from MFMAs of the same registers as the B
// operand against an A of ones (D[i][j] = the sum of column j % 8's block
// 4h + p + 2(j/8), in every row i); d8 * that sum is the staged product, so
// both variants compute the same bits.
//
// Summation order: a row's super-blocks form S = min(8, 2^floor(log2 nb))
// segments [s nb/S, (s+1) nb/S), each summed in order; the segment sums are
// combined in a fixed balanced binary tree.  A wave owns an aligned run of
// S/KS segments and forms that subtree itself; the reduction completes the
// tree across the KS waves.  So the result depends on K alone -- not on the
// number of rows, the tiles per workgroup or KS -- and row slices of a
// product reproduce it bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include "q4k_stage_units.h"
#include "q4k_tile.h"

namespace q4k {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int kMfmaRows = 16;   // weight rows per tile
constexpr int kMfmaCols = 8;    // activation columns of one MFMA (padded)
constexpr int kMfmaMaxSegs = 8; // summation segments of a row, at most
constexpr int kMfmaZeroBytes = 512;
// per-wave partial results of a round: 32 lanes x 4 columns, two buffers
__host__ __device__ constexpr int mfma_part_bytes(int waves) { return 2 * waves * 32 * 16; }

// LDS layout (bytes from the start): NC q8 columns of qcol = K + 16 bytes
// (the 16-byte skew puts the eight columns' reads of one lane octet in
// different banks), then d8 of every 32-value block for 8 columns
// ([block][column], half precision, as Q8_1 defines it), their d8 * sum q8
// ([block][column], float), the zero area, the partials and one weight slot
// per wave.
__host__ __device__ constexpr int mfma_qcol(int K) { return K + 16; }
__host__ __device__ constexpr int mfma_dk_off(int K, int nc) { return nc * mfma_qcol(K); }
__host__ __device__ constexpr int mfma_km_off(int K, int nc) { return mfma_dk_off(K, nc) + (K / 32) * kMfmaCols * 2; }
__host__ __device__ constexpr int mfma_zero_off(int K, int nc) { return mfma_km_off(K, nc) + (K / 32) * kMfmaCols * 4; }
__host__ __device__ constexpr int mfma_part_off(int K, int nc) { return mfma_zero_off(K, nc) + kMfmaZeroBytes; }
// Weight staging: an item (16 rows x one super-block, 2304 bytes) arrives
// with three contiguous 64-lane x 16-byte loads (chunk c = lane + 64i is
// bytes [16 (c % 9), +16) of row c / 9; loads that each touch one or two
// rows stream as fast as the tile kernel's, where loads touching all 16 rows
// reached half that), goes to the wave's LDS slot as it lies in memory (row
// pitch 144 bytes = 36 dwords: the 16-byte reads of 16 rows at one offset
// fall in distinct banks, and the writes are one contiguous run) and the
// MFMA operands are read from there.
constexpr int kMfmaSlotPitch = kBlockBytes;
constexpr int kMfmaSlotBytes = kMfmaRows * kMfmaSlotPitch;
constexpr int kMfmaChunks = kMfmaRows * kBlockBytes / 16;  // 144
__host__ __device__ constexpr int mfma_slot_off(int K, int nc, int waves) {
    return mfma_part_off(K, nc) + mfma_part_bytes(waves);
}
__host__ __device__ constexpr int mfma_lds_bytes(int K, int nc, int waves) {
    return mfma_slot_off(K, nc, waves) + waves * kMfmaSlotBytes;
}
// GA variants: d8 of every (block, column) ([block][8 columns], half: K / 2
// bytes), a zero area, the partials, one weight slot and one activation
// slot (8 columns x 288 bytes) per wave.
constexpr int kGaZeroBytes = 256;
constexpr int kGaSuperBytes = 8 * kQ81Bytes;  // one super-block of one Q8_1 column
constexpr int kGaSlotBytes = kMfmaCols * kGaSuperBytes;
__host__ __device__ constexpr int mfma_ga_zero_off(int K) { return K / 2; }
__host__ __device__ constexpr int mfma_ga_part_off(int K) { return K / 2 + kGaZeroBytes; }
__host__ __device__ constexpr int mfma_ga_slot_off(int K, int waves) { return mfma_ga_part_off(K) + mfma_part_bytes(waves); }
__host__ __device__ constexpr int mfma_ga_aslot_off(int K, int waves) {
    return mfma_ga_slot_off(K, waves) + waves * kMfmaSlotBytes;
}
__host__ __device__ constexpr int mfma_ga_lds_bytes(int K, int waves) {
    return mfma_ga_aslot_off(K, waves) + waves * kGaSlotBytes;
}

// One super-block's weights as the MFMA lane needs them: the header of row
// l % 16 and the lane group's 16 qs bytes of each 64.
struct MfmaRegs {
    u32x4 h;
    u32x4 q[2];
};

// One item in flight: the lane's three 16-byte chunks of the contiguous loads.
struct MfmaLoad {
    u32x4 v[3];
};

// Per-lane constants.
struct MfmaLane {
    int lane;
    int wrow;         // weight row in the tile (B column, D column)
    int grp;          // lane group: which 16 of 64 qs bytes the lane reads
    int hid;          // D: sub-block parity of the lane's outputs (lane / 32)
    int c0;           // D: first of the lane's four columns
    int a_off;        // LDS byte offset of the lane's A operand for super-block 0
    int a_inc;        // per super-block: 256 (data lanes) or 0 (zero lanes)
    int dk_off;       // LDS byte offset of its four columns' d8, block 2 hid of super-block 0
    int km_off;       // LDS byte offset of its min term's d8 * sum q8 (GA: of d8), super-block 0
    uint32_t sels, selm;  // byte selectors of its scales and mins
    uint32_t g_off[3];    // its chunks of an item: byte offsets from the item's first row
    int s_off[3];         // and in the wave's slot
    uint32_t ya_off[3];   // GA: its chunks of an item's activation, byte offsets from the item's first block
    int ar_off;           // GA: its A operand of product 0 in the activation slot (data lanes)
    int ar_step;          // GA: per block in the slot: 36 (data lanes) or 0 (zero lanes)
    bool a_data;          // GA: the lane carries activation (else it reads the zero area)
};

template <int NC, bool GA = false>
__device__ __forceinline__ MfmaLane mfma_lane(int K, int64_t stride_col_y = 0) {
    MfmaLane m;
    const int l = threadIdx.x & (kWave - 1);
    const int g = l >> 4;
    m.lane = l;
    m.wrow = l & 15;
    m.grp = g;
    m.hid = l >> 5;
    m.c0 = 4 * (g & 1);
    // A: row i = l % 16 -> column i % 8, sub-block pair i / 8; it holds
    // data in the lane groups of its own sub-block, zeros elsewhere
    const int ca = l & 7, hia = (l >> 3) & 1;
    const bool data = (g >> 1) == hia && ca < NC;
    m.a_off = data ? ca * mfma_qcol(K) + 64 * hia + 16 * (g & 1) : mfma_zero_off(K, NC) + 16 * (l & 7);
    m.a_inc = data ? kQK : 0;
    m.dk_off = (GA ? 0 : mfma_dk_off(K, NC)) + (2 * m.hid * kMfmaCols + m.c0) * 2;
    const int bm = (g & 1) + 4 * (g >> 1) + 2 * hia;  // its block of the min term
    m.km_off = GA ? (bm * kMfmaCols + ca) * 2 : mfma_km_off(K, NC) + (bm * kMfmaCols + ca) * 4;
    const uint32_t h = 2u * (uint32_t)m.hid, e = (uint32_t)(g & 1);
    m.sels = h | ((h + 1u) << 8) | ((h + 4u) << 16) | ((h + 5u) << 24);
    m.selm = e | ((e + 2u) << 8) | ((e + 4u) << 16) | ((e + 6u) << 24);
    // GA: chunk c = l + 64i of an item's activation is bytes [16 (c % 18),
    // +16) of column c / 18 (kOOB past the NC columns); the A operand of
    // product 2h + p is q8 bytes 16 (g & 1) .. of block 4h + p + 2 hia of
    // column ca
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int c = l + 64 * i, col = c / 18, o = c - 18 * col;
        m.ya_off[i] = col < NC ? (uint32_t)(col * stride_col_y) * (uint32_t)kQ81Bytes + 16u * (uint32_t)o : kOOB;
    }
    m.a_data = data;
    m.ar_off = ca * kGaSuperBytes + 2 * hia * kQ81Bytes + 4 + 16 * (g & 1);
    m.ar_step = data ? kQ81Bytes : 0;
    return m;
}

// The lane's chunk offsets of an item (rows row_stride bytes apart); chunks
// past the item's 144 get no offset (their loads read zeros, nothing is
// written).
__device__ __forceinline__ void mfma_chunks(MfmaLane &m, int64_t row_stride) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int c = m.lane + 64 * i, r = c / 9, o = c - 9 * (c / 9);
        m.g_off[i] = c < kMfmaChunks ? (uint32_t)(r * row_stride) + 16u * (uint32_t)o : kOOB;
        m.s_off[i] = r * kMfmaSlotPitch + 16 * o;
    }
}

// Loads one item: one super-block of 16 rows whose first row's block
// starts at byte offset off of the workgroup's buffer, or zeros when off is
// kOOB.  The sums need no selects: the buffer is under 2^31 bytes and off
// under 2^31 or kOOB, so off + kOOB and kOOB + g_off (g_off < 2^31) fall
// outside it and read zeros; kOOB + kOOB wraps to 0 and reads bytes, but
// only for chunks past the item's 144, which are never written to the slot.
__device__ __forceinline__ void mfma_load(__amdgpu_buffer_rsrc_t rs, uint32_t off, const MfmaLane &ln,
                                          MfmaLoad &w) {
#pragma unroll
    for (int i = 0; i < 3; ++i) w.v[i] = load16(rs, off + ln.g_off[i]);
}

__device__ __forceinline__ MfmaRegs mfma_read(const uint8_t *slot, const MfmaLane &ln) {
    MfmaRegs r;
    const uint8_t *row = slot + ln.wrow * kMfmaSlotPitch;
    r.h = *reinterpret_cast<const u32x4 *>(row);
#pragma unroll
    for (int h = 0; h < 2; ++h) r.q[h] = *reinterpret_cast<const u32x4 *>(row + 16 + 64 * h + 16 * ln.grp);
    return r;
}

// Writes an item to the wave's slot and reads the lane's operands back.
// The lanes read bytes other lanes wrote: a wave's LDS operations execute in
// order, so the compiler's order is enough (and the previous item's reads,
// issued before, are not overtaken by the writes).
__device__ __forceinline__ MfmaRegs mfma_stage(uint8_t *slot, const MfmaLane &ln, const MfmaLoad &w) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (i < 2 || ln.lane + 128 < kMfmaChunks) *reinterpret_cast<u32x4 *>(slot + ln.s_off[i]) = w.v[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return mfma_read(slot, ln);
}

// The lane's scales of sub-blocks 2hid, 2hid + 1, 4 + 2hid, 5 + 2hid, one per
// byte (the 4+2-bit fields of get_scale_min_k4).
__device__ __forceinline__ uint32_t mfma_scales(u32x4 h, const MfmaLane &ln) {
    const uint32_t x = __builtin_amdgcn_perm(h[3], h[1], ln.sels);
    return (x & 0x0f0f3f3fu) | ((x << 14) & 0x30300000u);
}

// The lane's mins of blocks b and b + 2, b = {0, 1, 4, 5}[lane group], in bytes
// 0 and 1.
__device__ __forceinline__ uint32_t mfma_mins(u32x4 h, const MfmaLane &ln) {
    const uint32_t x = __builtin_amdgcn_perm(h[3], h[2], ln.selm);
    const uint32_t low = x & 0x3f3fu;
    const uint32_t split = ((x >> 20) & 0x0f0fu) | ((x >> 2) & 0x3030u);
    return ln.grp < 2 ? low : split;
}

// The B operand of product m = 2h + p, and the start of the products.
__device__ __forceinline__ i32x4 mfma_b(const MfmaRegs &w, int m) {
    u32x4 b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = (m & 1 ? w.q[m >> 1][e] >> 4 : w.q[m >> 1][e]) & 0x0f0f0f0fu;
    return __builtin_bit_cast(i32x4, b);
}
constexpr int kMfmaMagic = 0x4B400000;  // 1.5 * 2^23 as a float

// The lane's d8 of its four columns and four sub-blocks, and its d8 * sum q8
// of the min term.
struct MfmaAux {
    f16x4 d8[4];
    float km;
};

// d8 from pd, the lane's of product 0.
__device__ __forceinline__ void mfma_d8(const uint8_t *pd, MfmaAux &x) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
        x.d8[m] = *reinterpret_cast<const f16x4 *>(pd + 2 * kMfmaCols * (4 * (m >> 1) + (m & 1)));
}

// The scaling of an item's four products s and its min term into acc.
// SUMS: also stores the int32 sums.
template <int NC, bool SUMS>
__device__ __forceinline__ void mfma_scale(const GemvParams &p, const MfmaLane &ln, const MfmaAux &aux, int kb,
                                           u32x4 h, const i32x4 (&s)[4], float (&acc)[4], int row, bool row_ok) {
    const uint32_t sc = mfma_scales(h, ln), mm = mfma_mins(h, ln);
    const float d = half_bits_to_float(h[0]), dmin = half_bits_to_float(h[0] >> 16);
    const bool second = (ln.lane & 8) != 0;
    f32x4 u = __builtin_amdgcn_mfma_f32_16x16x4f32(second ? 0.0f : aux.km, (float)(mm & 0xffu),
                                                   f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
    u = __builtin_amdgcn_mfma_f32_16x16x4f32(second ? aux.km : 0.0f, (float)((mm >> 8) & 0xffu), u, 0, 0, 0);
    float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const float scf = (float)((sc >> (8 * m)) & 0xffu);
        const float off = scf * -__builtin_bit_cast(float, kMfmaMagic);
        // the whole vector is cast (this clang reads element 0 for every
        // element of a vector cast one by one)
        const f32x4 sf = __builtin_bit_cast(f32x4, s[m]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            // |S| <= 32*15*127 and sc <= 63: sc * S is exact in f32
            const float x = __builtin_fmaf(sf[v], scf, off);
            t[v] = __builtin_fmaf((float)aux.d8[m][v], x, t[v]);
        }
        if constexpr (SUMS) {
            if (row_ok) {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (ln.c0 + v < NC)
                        p.sums[((int64_t)(ln.c0 + v) * p.M + row) * (p.K / 32) + kb * 8 + 4 * (m >> 1) + (m & 1) + 2 * ln.hid] =
                            s[m][v] - kMfmaMagic;
            }
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        acc[v] = __builtin_fmaf(d, t[v], acc[v]);
        acc[v] = __builtin_fmaf(-dmin, u[v], acc[v]);
    }
}

// One item: four MFMAs and their scaling into acc (the lane's row, four
// columns).
template <int NC, bool SUMS>
__device__ __forceinline__ void mfma_item(const GemvParams &p, const MfmaLane &ln, const uint8_t *lds, int kb,
                                          const MfmaRegs &w, float (&acc)[4], int row, bool row_ok) {
    const uint8_t *pa = lds + ln.a_off + ln.a_inc * kb;
    // the four products first (independent), then their scaling
    i32x4 s[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const i32x4 av = *reinterpret_cast<const i32x4 *>(pa + 128 * (m >> 1) + 32 * (m & 1));
        s[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, mfma_b(w, m),
                                                     i32x4{kMfmaMagic, kMfmaMagic, kMfmaMagic, kMfmaMagic}, 0, 0, 0);
    }
    MfmaAux aux;
    aux.km = *reinterpret_cast<const float *>(lds + ln.km_off + kb * (8 * kMfmaCols * 4));
    mfma_d8(lds + ln.dk_off + kb * (8 * kMfmaCols * 2), aux);
    mfma_scale<NC, SUMS>(p, ln, aux, kb, w.h, s, acc, row, row_ok);
}

// GA: the lane's chunks of the activation of super-block kb (zeros past the
// NC columns: kOOB + 288 kb stays outside the buffer).
__device__ __forceinline__ void mfma_load_act(__amdgpu_buffer_rsrc_t ry, const MfmaLane &ln, int kb, MfmaLoad &a) {
    const uint32_t o = (uint32_t)kb * (uint32_t)kGaSuperBytes;
#pragma unroll
    for (int i = 0; i < 3; ++i) a.v[i] = load16(ry, o + ln.ya_off[i]);
}

// GA: an item's A operands, those of its four products.
struct MfmaAct {
    i32x4 a[4];
};

// GA: mfma_stage for an item's weights and activation through the wave's two
// slots.  pa: the lane's A operand of product 0 (in the activation slot,
// 4-byte aligned, or the zero area), pa + ar_step * blk that of the product
// of blk.
__device__ __forceinline__ MfmaRegs mfma_stage_ga(uint8_t *slot, uint8_t *aslot, const uint8_t *pa, const MfmaLane &ln,
                                                  const MfmaLoad &w, const MfmaLoad &a, int nc, MfmaAct &act) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if (i < 2 || ln.lane + 128 < kMfmaChunks) *reinterpret_cast<u32x4 *>(slot + ln.s_off[i]) = w.v[i];
        if (ln.lane + 64 * i < 18 * nc) *reinterpret_cast<u32x4 *>(aslot + 16 * (ln.lane + 64 * i)) = a.v[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const uint32_t *q = reinterpret_cast<const uint32_t *>(pa + ln.ar_step * (4 * (m >> 1) + (m & 1)));
        act.a[m] = i32x4{(int)q[0], (int)q[1], (int)q[2], (int)q[3]};
    }
    return mfma_read(slot, ln);
}

// mfma_item with the A operands in registers (GA): d8 from the LDS table,
// the blocks' sums of q8 from the products of ones.  SQ: also stores those
// (the lanes of the min term's block hold them).
template <int NC, bool SUMS>
__device__ __forceinline__ void mfma_item_ga(const GemvParams &p, const MfmaLane &ln, const uint8_t *lds, int kb,
                                             const MfmaRegs &w, const MfmaAct &act, float (&acc)[4], int row,
                                             bool row_ok, bool sq_ok) {
    i32x4 s[4], z[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        s[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(act.a[m], mfma_b(w, m),
                                                     i32x4{kMfmaMagic, kMfmaMagic, kMfmaMagic, kMfmaMagic}, 0, 0, 0);
        z[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{0x01010101, 0x01010101, 0x01010101, 0x01010101}, act.a[m],
                                                     i32x4{0, 0, 0, 0}, 0, 0, 0);
    }
    const int z01 = ln.grp & 1 ? z[1][0] : z[0][0], z23 = ln.grp & 1 ? z[3][0] : z[2][0];
    const int zs = ln.grp < 2 ? z01 : z23;  // of block {0, 1, 4, 5}[lane group] + 2 hia
    MfmaAux aux;
    aux.km = (float)*reinterpret_cast<const _Float16 *>(lds + ln.km_off + kb * (8 * kMfmaCols * 2)) * (float)zs;
    mfma_d8(lds + ln.dk_off + kb * (8 * kMfmaCols * 2), aux);
    if constexpr (SUMS) {
        const int blk = (ln.grp & 1) + 4 * (ln.grp >> 1) + 2 * ((ln.lane >> 3) & 1);
        if (sq_ok && (ln.lane & 7) < NC) p.sq[(ln.lane & 7) * (p.K / 32) + kb * 8 + blk] = zs;
    }
    mfma_scale<NC, SUMS>(p, ln, aux, kb, w.h, s, acc, row, row_ok);
}

// Adds segment value v (the sum of one segment, local index t in the wave's
// run) into the wave's subtree: l1, l2, l4 hold the pending left subtrees of
// 1, 2 and 4 segments; returns the subtree that ends at t.
__device__ __forceinline__ void mfma_tree_push(int t, float (&v)[4], float (&l1)[4], float (&l2)[4],
                                               float (&l4)[4]) {
    if (t & 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = l1[k] + v[k];
        if (t & 2) {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = l2[k] + v[k];
            if (t & 4) {
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = l4[k] + v[k];
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) l4[k] = v[k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) l2[k] = v[k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) l1[k] = v[k];
    }
}

// A wave's position in its items: round r (tile group + ngroups * r) and
// super-block kb of the tile.
struct MfmaPos {
    int r, kb;
};

// What bounds it: with few tiles per workgroup the chain before the first
// product (the activation's loads, queued 1.3-1.9 us after the start, and its
// quantisation, to 5 us), then 0.7 us per item and wave of LDS and dependent
// arithmetic; over many tiles the weight stream (128256 x 4096 N=8 64 us, 4.6
// TB/s; a plain read in the same pattern 52).  The arithmetic takes about 100
// vector instructions an item against 170 with the min term, the int -> float
// conversions and a nibble mask and shift per product on the vector unit.
// With that, the staging on the scalar unit, the loads among the rounds, none
// past the end and 8 waves for 16: 14336 x 4096 N=8 14.9 -> 13.1 us, 13824 x
// 5120 N=6 17.5 -> 15.0; GA 4096 x 14336 N=8 19.3 -> 18.6 with its quantiser.
// The kernel.  rows_base / rows_extra are the tile split: each workgroup
// owns rows_base tiles of 16 rows, the first rows_extra one more;
// p.rpw: KS, the waves that share one tile (1, 2, 4 or 8, at most S);
// p.ntiles: S, the segments of a row.  GA: the A operand from the Q8_1
// buffer p.y (which the GA variants require).  NIF: items in flight per
// wave (2, or 4 in the GA variants).
template <int NC, int WAVES, bool SUMS = false, bool GA = false, int NIF = 2>
__global__ __launch_bounds__(kWave *WAVES) void gemv_q4k_mfma_kernel(Q4K_GEMV_KERNEL_ARGS) {
    static_assert(NC >= 1 && NC <= kMfmaCols, "up to 8 columns");
    static_assert(WAVES == 8 || WAVES == 16, "8 or 16 waves");
    constexpr int NT = kWave * WAVES;
    int32_t *const sq_out = SUMS ? p.sq : nullptr;
    p = with_head(p, Q4K_GEMV_HEAD_VALUES);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    int8_t *q8s = reinterpret_cast<int8_t *>(lds);
    void *aux = lds + mfma_dk_off(p.K, NC);

    constexpr int kLPB = stage_lpb(NC);
    constexpr int kPreR = GA ? 1 : pre_rounds(NC, NT);
    ActStage<kLPB, kPreR> xs;
    Q81Stage<kPreR> ys;
    if constexpr (!GA) {
        // first of all: everything waits for the activation
        if (p.x) unit_f32_issue<kLPB, NT>(p.x, p.ldx, p.K, NC, p.vec_ok != 0, p.stage_div, xs);
        else unit_q81_issue<NT>(p.y, p.stride_col_y, p.K, NC, p.stage_div, ys);
        __builtin_amdgcn_sched_barrier(0);
    }
    MfmaLane ln = mfma_lane<NC, GA>(p.K, p.stride_col_y);
    mfma_chunks(ln, p.row_stride);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // KS and S are powers of two
    const int KS = p.rpw, lks = __builtin_ctz(KS), S = p.ntiles, ls = __builtin_ctz(S);
    const int group = wave >> lks, ks = wave & (KS - 1);
    const int ngroups = WAVES >> lks;
    const int segs = S >> lks, seg0 = ks * segs;  // the wave's run of segments
    // this workgroup's tiles and this wave's super-blocks of each
    const int b = (int)blockIdx.x;
    const int t0 = b * p.rows_base + min(b, p.rows_extra);
    const int nt = p.rows_base + (b < p.rows_extra ? 1 : 0);
    const int rounds = (nt + ngroups - 1) * KS / WAVES;
    const int kb0 = seg0 * p.nb >> ls, kb1 = (seg0 + segs) * p.nb >> ls;  // kb1 > kb0 (S <= nb)
    const int items = rounds * (kb1 - kb0);
    const int row0 = t0 * kMfmaRows;
    const int nrows = min(nt * kMfmaRows, p.M - row0);
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(p.w + (int64_t)row0 * p.row_stride, nrows > 0 ? (uint32_t)(nrows * p.row_stride) : 0u);

    if constexpr (!GA) __syncthreads();  // all activation loads of this CU are queued first
    // GA: the Q8_1 columns as one buffer (columns stride_col_y blocks apart;
    // the host keeps it under 2^31 bytes)
    const __amdgpu_buffer_rsrc_t ry =
        make_rsrc(p.y, GA ? (uint32_t)((int64_t)(NC - 1) * p.stride_col_y * kQ81Bytes + (p.K / 32) * kQ81Bytes) : 0u);

    // items in order: rounds, and super-blocks kb0..kb1-1 of each; loads of
    // positions past the wave's last round or the workgroup's tiles read zeros
    auto next = [&](MfmaPos q) -> MfmaPos { return q.kb + 1 < kb1 ? MfmaPos{q.r, q.kb + 1} : MfmaPos{q.r + 1, kb0}; };
    auto item_off = [&](MfmaPos q) -> uint32_t {
        const int tile = group + ngroups * q.r;
        if (q.r >= rounds || tile >= nt) return kOOB;
        return (uint32_t)(tile * kMfmaRows * p.row_stride) + (uint32_t)q.kb * kBlockBytes;
    };
    static_assert(NIF >= 2 && NIF <= 4, "items in flight");
    MfmaPos cur{0, kb0};
    MfmaPos ahead = cur;
    MfmaLoad w[NIF];
    MfmaLoad av[GA ? NIF : 1];
    auto issue = [&](int k) {
        mfma_load(rs, item_off(ahead), ln, w[k]);
        if constexpr (GA) mfma_load_act(ry, ln, ahead.kb, av[GA ? k : 0]);
        ahead = next(ahead);
    };

    if constexpr (GA) {
#pragma unroll
        for (int k = 0; k < NIF; ++k) issue(k);
        // d8 of every (block, column); the padding columns' outputs are dropped
        uint16_t *d8s = reinterpret_cast<uint16_t *>(lds);
        for (int q = (int)threadIdx.x; q < (p.K / 32) * kMfmaCols; q += NT) {
            const int blk = q >> 3, c = q & 7;
            if (c < NC)
                d8s[q] = *reinterpret_cast<const uint16_t *>(p.y + ((int64_t)c * p.stride_col_y + blk) * kQ81Bytes);
        }
        // the zero area the A operand's zero lanes read
        if (threadIdx.x < kGaZeroBytes / 16)
            reinterpret_cast<u32x4 *>(lds + mfma_ga_zero_off(p.K))[threadIdx.x] = u32x4{0u, 0u, 0u, 0u};
    } else {
        // the items' loads among the rounds of the quantisation: issued
        // together ahead of it, the waves whose requests queued last stood
        // still until most of the others' data had arrived
        stage_interleaved<kLayoutMfma, kLPB, NT, NIF>(p.x, p.ldx, p.y, p.stride_col_y, p.K, NC, p.vec_ok != 0, p.stage_div,
                                                      xs, ys, __builtin_amdgcn_readfirstlane(mfma_qcol(p.K)), q8s, aux,
                                                      sq_out, issue);
        // the zero area of the A operand (the padding columns' d8 stay
        // unwritten: their outputs are dropped)
        if (threadIdx.x < kMfmaZeroBytes / 16)
            reinterpret_cast<u32x4 *>(lds + mfma_zero_off(p.K, NC))[threadIdx.x] = u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();

    float acc[4] = {}, l1[4] = {}, l2[4] = {}, l4[4] = {};
    float *part = reinterpret_cast<float *>(lds + (GA ? mfma_ga_part_off(p.K) : mfma_part_off(p.K, NC)));
    uint8_t *slot =
        lds + (GA ? mfma_ga_slot_off(p.K, WAVES) : mfma_slot_off(p.K, NC, WAVES)) + wave * kMfmaSlotBytes;
    uint8_t *aslot = lds + mfma_ga_aslot_off(p.K, WAVES) + wave * kGaSlotBytes;  // GA only
    const uint8_t *pa = GA && ln.a_data ? aslot + ln.ar_off : lds + mfma_ga_zero_off(p.K);
    int t = 0;                            // local segment of the current item
    int seg_end = (seg0 + 1) * p.nb >> ls;  // its end (super-block)
    // One item, held in registers k; reload: then the loads of the item NIF
    // further on, into the same.
    auto item = [&](int k, bool reload) {
        const int tile = group + ngroups * cur.r;
        const int row = row0 + tile * kMfmaRows + ln.wrow;
        const bool row_ok = SUMS && tile < nt && row < p.M;
        if constexpr (GA) {
            MfmaAct act;
            const MfmaRegs wr = mfma_stage_ga(slot, aslot, pa, ln, w[k], av[GA ? k : 0], NC, act);
            if (reload) issue(k);
            // sq: the group of waves holding tile 0 of workgroup 0 covers
            // every super-block once
            mfma_item_ga<NC, SUMS>(p, ln, lds, cur.kb, wr, act, acc, row, row_ok,
                                   SUMS && blockIdx.x == 0 && group == 0 && cur.r == 0);
        } else {
            const MfmaRegs wr = mfma_stage(slot, ln, w[k]);
            if (reload) issue(k);
            mfma_item<NC, SUMS>(p, ln, lds, cur.kb, wr, acc, row, row_ok);
        }
        const MfmaPos done = cur;
        cur = next(cur);
        if (done.kb + 1 != seg_end) return;
        // segment end: its value is the sum of the two sub-block parities of
        // each (row, column), in lanes l and l + 32
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float hi = acc[c];
            permlane32_swap(acc[c], hi);
            v[c] = acc[c] + hi;
            acc[c] = 0.0f;
        }
        mfma_tree_push(t, v, l1, l2, l4);
        ++t;
        if (t < segs) {
            seg_end = (seg0 + t + 1) * p.nb >> ls;
            return;
        }
        // round end: v is the wave's subtree of the tile
        t = 0;
        seg_end = (seg0 + 1) * p.nb >> ls;
        const int buf = done.r & 1;
        if (ln.lane < 32)
            *reinterpret_cast<float4 *>(part + ((buf * WAVES + wave) * 32 + ln.lane) * 4) =
                make_float4(v[0], v[1], v[2], v[3]);
        __syncthreads();
        // outputs of this round: tile group q, column c, row rr; consecutive
        // threads write consecutive rows of a column.  The KS subtrees
        // combine in the same balanced tree.
        for (int o = (int)threadIdx.x; o < ngroups * kMfmaRows * kMfmaCols; o += NT) {
            const int rr = o & 15, c = (o >> 4) & 7, q = o >> 7;
            const int otile = q + ngroups * done.r;
            const int orow = row0 + otile * kMfmaRows + rr;
            if (c < NC && otile < nt && orow < p.M) {
                const int l32 = rr + 16 * (c >> 2);
                const float *src = part + ((buf * WAVES + q * KS) * 32 + l32) * 4 + (c & 3);
                float pv[kMfmaMaxSegs];
#pragma unroll
                for (int j = 0; j < kMfmaMaxSegs; ++j) pv[j] = j < KS ? src[j * 32 * 4] : 0.0f;
#pragma unroll
                for (int wdt = 1; wdt < kMfmaMaxSegs; wdt *= 2)
#pragma unroll
                    for (int j = 0; j + wdt < kMfmaMaxSegs; j += 2 * wdt)
                        if (j + wdt < KS) pv[j] = pv[j] + pv[j + wdt];
                p.dst[(int64_t)c * p.ld_dst + orow] = pv[0];
            }
        }
    };
    // The main loop's items all have one to reload, so its waits count exactly
    // the loads in flight; the last ones (NIF, or up to one less than two
    // rounds of the loop) are apart, without loads past the wave's items:
    // those read zeros, but each of their instructions takes the CU's address
    // path some 17 ns all the same (4096 x 4096 N=8: 0.4 us per item in
    // flight and wave).
    int it = 0;
    for (; it + 2 * NIF <= items; it += NIF) {
#pragma unroll
        for (int k = 0; k < NIF; ++k) item(k, true);
    }
#pragma unroll
    for (int k = 0; k < 2 * NIF - 1; ++k) {
        if (it + k >= items) return;  // uniform; the last barrier is behind
        item(k % NIF, k < NIF && it + k + NIF < items);
    }
}

}  // namespace q4k
