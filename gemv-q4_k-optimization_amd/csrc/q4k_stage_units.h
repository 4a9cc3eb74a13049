// q4k_stage_units.h -- the staging of the matrix-core kernels (q4k_mfma.h,
// q6k_mfma.h): F32 columns quantised to Q8_1, or Q8_1 columns, into linear q8
// columns in LDS with their d8 (and d8 * sum q8) per [block][column].
//
// The other kernels stage lane by lane (q4k_device.h, stage_f32_issue and what
// follows), each lane with the address and place of its own block.  Here a
// round's column and super-block are wave-uniform.  It suits these kernels
// (14336 x 4096 N=8 14.9 -> 13.2 us together with the loads among the rounds)
// and not those: with it the tile kernel's pre-quantised launches took up to
// 14 % longer (MI355X, us, units against lanes: 1548 x 13568 N=8 15.9 / 14.0,
// 640 x 768 N=7 5.05 / 4.50, 1613 x 14592 N=5 12.1 / 11.0) and its F32 ones up
// to 11 % (4635 x 4864 N=1 5.92 / 5.36).
#pragma once

#include <hip/hip_runtime.h>

#include "q4k_device.h"

namespace q4k {

// The super-blocks that a staging round of a wave covers: a unit of SPW = 8 /
// LPB super-blocks of one column (kb and kb + 1 with kb even where SPW is 2:
// the wave's lanes below 32 take the first, the others the second, which a
// column with an odd number lacks in its last unit).  The units of all
// columns in order are dealt to the workgroup's waves, round by round.  So
// what depends on the super-block (column, address, LDS places) is
// wave-uniform and computed on the scalar unit, and the lanes add constants:
// each vector instruction before the first load costs a 16-wave workgroup 16
// cycles per SIMD, and with a division and three products per lane and round
// the loads of 14336 x 4096 N=8 were queued only 2.4 us after the start.
// With several columns the workgroups of an XCD (blockIdx % 8) start at
// different units: all of them read the whole activation, and in one order
// all would wait for the first fetch of the same lines.
template <int LPB, int NT>
struct StageMap {
    static constexpr int kSPW = 8 / LPB;
    static constexpr bool kRotate = kSPW == 2;
    static constexpr int kWaves = NT / kWave;
    int wave, upc, units, rot, nb;
    int e, s;        // lane: part of its block, block of its super-block
    int second;      // lane: 1 in the unit's second super-block
};

// One round: the unit's column and (first) super-block.
struct StagePlace {
    int c, kb;
    bool half;       // the unit has no second super-block
};

// Units per column of K values at LPB 4: what FastDiv arguments divide by.
__host__ __device__ constexpr int stage_units(int K) { return (K / kQK + 1) / 2; }

template <int LPB, int NT>
__device__ __forceinline__ StageMap<LPB, NT> stage_map(int K, int ncols) {
    typedef StageMap<LPB, NT> Map;
    Map m;
    m.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    m.nb = K / kQK;
    m.upc = Map::kSPW == 2 ? stage_units(K) : m.nb;
    m.units = ncols * m.upc;
    m.rot = Map::kRotate ? (int)(((blockIdx.x >> 3) & 31u) * (uint32_t)m.units >> 5) : 0;
    const int lane = threadIdx.x & (kWave - 1);
    m.e = lane & (LPB - 1);
    m.s = (lane / LPB) & 7;
    m.second = Map::kSPW == 2 ? lane >> 5 : 0;
    return m;
}

// The wave has a round j.
template <int LPB, int NT>
__device__ __forceinline__ bool stage_has(const StageMap<LPB, NT> &m, int j) {
    return m.wave + j * m.kWaves < m.units;
}

// The place of the wave's round j (a round past the last: the last).
template <int LPB, int NT>
__device__ __forceinline__ StagePlace stage_place(const StageMap<LPB, NT> &m, int j, int ncols, const FastDiv &fd) {
    typedef StageMap<LPB, NT> Map;
    int u = min(m.wave + j * Map::kWaves, m.units - 1);
    if (Map::kRotate) {
        u += m.rot;
        if (u >= m.units) u -= m.units;
    }
    StagePlace p;
    p.c = ncols == 1 ? 0 : (int)fastdiv((uint32_t)u, fd);
    p.kb = Map::kSPW * (u - p.c * m.upc);
    p.half = Map::kSPW == 2 && p.kb + 1 == m.nb;
    return p;
}

// Where a lane's part of a round goes in LDS: its values' byte offset in the
// q8 columns; its d8 (half) at d8[a0] of the auxiliary area and, with the sums
// (kLayoutMfma), its d8 * sum q8 (float) at index a1 from the area's start; the
// block's index qb = c*K/32 + b.
struct StageDst {
    int q8, a0, a1, qb;
};

template <int LPB, int NT>
__device__ __forceinline__ StageDst stage_dst(const StageMap<LPB, NT> &m, const StagePlace &p, int qcol, int e4) {
    const int nblk = m.nb * 8;
    // the lane's block of the unit, 0..15
    const int blk = m.s + 8 * m.second;
    StageDst d;
    d.q8 = __builtin_amdgcn_readfirstlane(p.c * qcol + p.kb * kQK) + (blk * 32 + e4 * 4);
    d.a0 = __builtin_amdgcn_readfirstlane(p.kb * 64 + p.c) + 8 * blk;
    d.a1 = __builtin_amdgcn_readfirstlane(nblk * 4 + p.kb * 64 + p.c) + 8 * blk;
    d.qb = p.c * nblk + p.kb * 8 + blk;
    return d;
}

// Stores a block's auxiliary terms from its first lane: d8 = half(d) widened,
// qsum = sum of all 32 q8.
template <int LAYOUT>
__device__ __forceinline__ void unit_store_aux(void *aux, const StageDst &at, float d8, int qsum) {
    static_assert(LAYOUT == kLayoutMfma || LAYOUT == kLayoutMfmaQ6, "the matrix-core kernels' layouts");
    reinterpret_cast<_Float16 *>(aux)[at.a0] = (_Float16)d8;
    if (LAYOUT == kLayoutMfma) reinterpret_cast<float *>(aux)[at.a1] = d8 * (float)qsum;
}

// sq_out (parity variants only; a literal null in the product kernels, so the
// store compiles away): the int32 sum of the block's 32 q8 at sq_out[qb].
// live: the lane has a block (only the stores are left out without one).
template <int LAYOUT, int LPB>
__device__ __forceinline__ void unit_quantize(const float (&v)[32 / LPB], int e, bool live, const StageDst &at,
                                                    int8_t *q8s, void *aux, int32_t *sq_out = nullptr) {
    constexpr int V = 32 / LPB;
    float d;
    uint32_t word[V / 4];
    quantize_lanes(v, d, word);
    int hsum, fsum;
    block_sums<LPB>(packed_sum(word), hsum, fsum);
    if (!live) return;
    int8_t *dst = q8s + at.q8;
    if (V == 4) *reinterpret_cast<uint32_t *>(dst) = word[0];
    else *reinterpret_cast<uint2 *>(dst) = make_uint2(word[0], word[V / 4 - 1]);
    const float d8 = (float)(_Float16)d;
    if (e == 0) unit_store_aux<LAYOUT>(aux, at, d8, fsum);
    if (sq_out && e == 0) sq_out[at.qb] = fsum;
}

// The lane's values of a round; lanes without a super-block re-read the
// unit's first.
template <int LPB, int NT>
__device__ __forceinline__ const float *stage_src(const StageMap<LPB, NT> &m, const StagePlace &p, const float *x,
                                                  int64_t ldx) {
    const uint32_t lane = (uint32_t)(m.s * 32 + m.e * (32 / LPB));
    return x + (p.c * ldx + p.kb * kQK) + (p.half ? lane : lane + (uint32_t)m.second * kQK);
}

template <int LPB, int NT, int PRE>
__device__ __forceinline__ void unit_f32_issue(const float *__restrict__ x, int64_t ldx, int K,
                                                int ncols, bool vec_ok, const FastDiv &fd,
                                                ActStage<LPB, PRE> &st) {
    const auto m = stage_map<LPB, NT>(K, ncols);
#pragma unroll
    for (int j = 0; j < PRE; ++j) {
        if (j >= 4 && j * m.kWaves >= m.units) break;  // uniform: rounds past the values are not loaded
        load_xv<32 / LPB>(stage_src(m, stage_place(m, j, ncols, fd), x, ldx), vec_ok, st.v[j]);
    }
}

// Values that were loaded and are not needed: the compiler waits for their
// loads here (they are older than any weight's) and not, by waiting for
// everything, where it next uses their registers.
template <typename T, int V>
__device__ __forceinline__ void stage_use(const T (&v)[V]) {
#pragma unroll
    for (int k = 0; k < V; ++k) asm volatile("" ::"v"(v[k]));
}

// Every load has arrived (the wave's newest were just used): tells the
// compiler, which merges the paths with and without further rounds.
__device__ __forceinline__ void stage_loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0) alone

// Quantises the wave's round j, values v (nothing when it has none).
template <int LAYOUT, int LPB, int NT>
__device__ __forceinline__ void unit_f32_round(const StageMap<LPB, NT> &m, int j, const float (&v)[32 / LPB],
                                                int ncols, const FastDiv &fd, int qcol, int8_t *q8s, void *aux,
                                                int32_t *sq_out) {
    if (!stage_has(m, j)) {  // uniform
        stage_use(v);
        return;
    }
    const StagePlace p = stage_place(m, j, ncols, fd);
    unit_quantize<LAYOUT, LPB>(v, m.e, !(p.half && m.second),
                                     stage_dst(m, p, qcol, m.e * (8 / LPB)), q8s, aux,
                                     sq_out);
}

// Rounds [j0, j1) of those in registers.
template <int LAYOUT, int LPB, int NT, int PRE>
__device__ __forceinline__ void unit_f32_span(const StageMap<LPB, NT> &m, int j0, int j1,
                                               const ActStage<LPB, PRE> &st, int ncols, const FastDiv &fd, int qcol,
                                               int8_t *q8s, void *aux, int32_t *sq_out) {
#pragma unroll
    for (int j = j0; j < j1; ++j) unit_f32_round<LAYOUT>(m, j, st.v[j], ncols, fd, qcol, q8s, aux, sq_out);
}

// The rounds from PRE on.
template <int LAYOUT, int LPB, int NT, int CHUNK, int PRE>
__device__ __forceinline__ void unit_f32_rest(const StageMap<LPB, NT> &m, const float *__restrict__ x, int64_t ldx,
                                               int ncols, bool vec_ok, const FastDiv &fd, int qcol, int8_t *q8s,
                                               void *aux, int32_t *sq_out) {
    constexpr int V = 32 / LPB;
    // A chunk of rounds at a time: all their loads first, then their
    // quantisation, so a chunk costs one memory round trip rather than one
    // per round.
    constexpr int kChunk = CHUNK;
    for (int j0 = PRE; stage_has(m, j0); j0 += kChunk) {
        float v[kChunk][V];
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
            if (j > 0 && !stage_has(m, j0 + j)) break;
            load_xv<V>(stage_src(m, stage_place(m, j0 + j, ncols, fd), x, ldx), vec_ok, v[j]);
        }
#pragma unroll
        for (int j = 0; j < kChunk; ++j)
            unit_f32_round<LAYOUT>(m, j0 + j, v[j], ncols, fd, qcol, q8s, aux, sq_out);
        stage_loads_done();
    }
}

// The lane's 8 of a block's 32 q8 and the block's ds.
template <int NT>
__device__ __forceinline__ void load_q81(const StageMap<4, NT> &m, const StagePlace &p,
                                         const uint8_t *__restrict__ y, int64_t stride_col_y, uint32_t (&w)[2],
                                         uint32_t &ds) {
    const uint32_t lane = (uint32_t)(m.s * kQ81Bytes);
    const uint8_t *blk = y + (p.c * stride_col_y + p.kb * 8) * kQ81Bytes +
                         (p.half ? lane : lane + (uint32_t)(m.second * 8 * kQ81Bytes));
    w[0] = *reinterpret_cast<const uint32_t *>(blk + 4 + m.e * 8);
    w[1] = *reinterpret_cast<const uint32_t *>(blk + 8 + m.e * 8);
    ds = *reinterpret_cast<const uint32_t *>(blk);
}

template <int NT, int PRE>
__device__ __forceinline__ void unit_q81_issue(const uint8_t *__restrict__ y, int64_t stride_col_y,
                                                int K, int ncols, const FastDiv &fd, Q81Stage<PRE> &st) {
    const auto m = stage_map<4, NT>(K, ncols);
#pragma unroll
    for (int j = 0; j < PRE; ++j) {
        if (j >= 4 && j * m.kWaves >= m.units) break;  // uniform, as above
        load_q81(m, stage_place(m, j, ncols, fd), y, stride_col_y, st.w[j], st.ds[j]);  // unconditional, as above
    }
}

template <int LAYOUT>
__device__ __forceinline__ void unit_q81_store(uint32_t w0, uint32_t w1, uint32_t ds, int quarter, bool live,
                                               const StageDst &at, int8_t *q8s, void *aux,
                                               int32_t *sq_out = nullptr) {
    int hsum, fsum;
    block_sums<4>(__builtin_amdgcn_sdot4((int)w0, 0x01010101, __builtin_amdgcn_sdot4((int)w1, 0x01010101, 0, false),
                                         false),
                  hsum, fsum);
    if (!live) return;
    *reinterpret_cast<uint2 *>(q8s + at.q8) = make_uint2(w0, w1);
    if (quarter == 0) unit_store_aux<LAYOUT>(aux, at, half_bits_to_float(ds), fsum);
    if (sq_out && quarter == 0) sq_out[at.qb] = fsum;
}

template <int LAYOUT, int NT>
__device__ __forceinline__ void unit_q81_round(const StageMap<4, NT> &m, int j, const uint32_t (&w)[2], uint32_t ds,
                                                int ncols, const FastDiv &fd, int qcol, int8_t *q8s, void *aux,
                                                int32_t *sq_out) {
    if (!stage_has(m, j)) {  // uniform
        stage_use(w);
        asm volatile("" ::"v"(ds));
        return;
    }
    const StagePlace p = stage_place(m, j, ncols, fd);
    unit_q81_store<LAYOUT>(w[0], w[1], ds, m.e, !(p.half && m.second),
                           stage_dst(m, p, qcol, 2 * m.e), q8s, aux, sq_out);
}

template <int LAYOUT, int NT, int CHUNK, int PRE>
__device__ __forceinline__ void unit_q81_rest(const StageMap<4, NT> &m, const uint8_t *__restrict__ y,
                                               int64_t stride_col_y, int ncols, const FastDiv &fd, int qcol,
                                               int8_t *q8s, void *aux, int32_t *sq_out) {
    // CHUNK rounds at a time, loads first, as in unit_f32_rest
    constexpr int kChunk = CHUNK;
    for (int j0 = PRE; stage_has(m, j0); j0 += kChunk) {
        uint32_t w[kChunk][2], ds[kChunk];
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
            if (j > 0 && !stage_has(m, j0 + j)) break;
            load_q81(m, stage_place(m, j0 + j, ncols, fd), y, stride_col_y, w[j], ds[j]);
        }
#pragma unroll
        for (int j = 0; j < kChunk; ++j)
            unit_q81_round<LAYOUT>(m, j0 + j, w[j], ds[j], ncols, fd, qcol, q8s, aux, sq_out);
        stage_loads_done();
    }
}

// The whole activation into LDS, from F32 or (x null) from Q8_1 columns, with N
// other steps among the rounds: issue(k) before the k-th N-th of those in
// registers (which unit_f32_issue or unit_q81_issue loaded).
template <int LAYOUT, int LPB, int NT, int N, int PRE, typename F>
__device__ __forceinline__ void stage_interleaved(const float *__restrict__ x, int64_t ldx,
                                                  const uint8_t *__restrict__ y, int64_t stride_col_y, int K,
                                                  int ncols, bool vec_ok, const FastDiv &fd,
                                                  const ActStage<LPB, PRE> &xs, const Q81Stage<PRE> &ys, int qcol,
                                                  int8_t *q8s, void *aux, int32_t *sq_out, F issue) {
    if (x) {
        const auto m = stage_map<LPB, NT>(K, ncols);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            issue(k);
            unit_f32_span<LAYOUT>(m, k * PRE / N, (k + 1) * PRE / N, xs, ncols, fd, qcol, q8s, aux, sq_out);
        }
        unit_f32_rest<LAYOUT, LPB, NT, kFinishRounds, PRE>(m, x, ldx, ncols, vec_ok, fd, qcol, q8s, aux, sq_out);
    } else {
        const auto m = stage_map<4, NT>(K, ncols);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            issue(k);
#pragma unroll
            for (int j = k * PRE / N; j < (k + 1) * PRE / N; ++j)
                unit_q81_round<LAYOUT>(m, j, ys.w[j], ys.ds[j], ncols, fd, qcol, q8s, aux, sq_out);
        }
        unit_q81_rest<LAYOUT, NT, kFinishRounds, PRE>(m, y, stride_col_y, ncols, fd, qcol, q8s, aux, sq_out);
    }
}

}  // namespace q4k
