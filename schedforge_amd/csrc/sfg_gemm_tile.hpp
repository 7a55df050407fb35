// sfg_gemm_tile.hpp -- what the tiled MFMA GEMM kernels share: their argument
// block, the tile order, the instruction-interleaving helpers and the store
// epilogues (residual, GLU, QKV split + RoPE).
#pragma once

#include <type_traits>

#include "sfg_gemm_plan.hpp"
#include "sfg_kernels.hpp"

namespace sfg {


template <int EPI>
struct EpiTraits {
    static constexpr bool glu = (EPI == SFG_EPI_SWIGLU || EPI == SFG_EPI_GLU_SILU_UP);
};

__device__ __forceinline__ float glu_combine(int epi, float g, float u) {
    return epi == SFG_EPI_SWIGLU ? silu(g) * u : g * silu(u);
}

__device__ __forceinline__ void store_out(void* c, int c_dtype, int64_t idx, float v) {
    if (c_dtype == SFG_F32) static_cast<float*>(c)[idx] = v;
    else static_cast<uint16_t*>(c)[idx] = f32_to_bf16(v);
}


struct TiledArgs {
    const uint16_t* a; int64_t lda; const int32_t* a_rows; int64_t a_rows_limit;
    const void* b; int64_t ldb; const float* scales;
    int64_t b_group_stride, s_group_stride;
    void* c; int c_dtype; int64_t ldc;
    const float* residual; int64_t ldr;
    int64_t m, n, k;
    const int32_t* offsets;   // grouped: first row of each group
    int groups;
    QkvRopeOut qkv;           // kEpiQkvRope only
    int xcds;                 // XCDs the dispatcher deals workgroups over
    int b_tiled;              // gemm_ring_kernel: B in SFG_LAYOUT_TILED
};

// (sfg_gemm_ring.hip)
int launch_ring(const TiledArgs& a, const RingPlan& plan, int b_dtype, int epi, float* part, hipStream_t s);

// ===========================================================================
// QKV epilogue for the bf16 prefill (split_qkv + apply_rope,
// decoder_compiler.cpp:96-148, plus the transposed V the flash prefill reads):
// the [rows][H + 2 Hkv 128] product is never stored.  Column c of the
// accumulator lives in lane c % 32; RoPE pairs (2i, 2i+1) are neighbouring
// lanes of one row, so one lane exchange gives each lane its partner, and the
// rotation is split_rope_kernel's expression (same table, same float ops).
// Every 32-column block lies inside one head, so the Q / K / V choice is
// uniform per block.  A lane's four consecutive rows (r % 4) are four
// consecutive tokens of one sequence (S % 4 == 0, checked on the host), so
// V^T takes one 8-byte store per lane and block.  kAnySeq: sequences of any length
// of at least four rows, where a run of four rows may end one and begin the next,
// and V^T takes single stores unless S % 4 == 0.  (Wave blocks larger than 64 x 64
// have no registers for it.)
// ===========================================================================
template <int WM, int WN, bool kAnySeq>
__device__ __forceinline__ void qkv_rope_epilogue(const QkvRopeOut& o, const floatx16 (&acc)[WM][WN],
                                                  int64_t wave_row0, int64_t wave_col0, int64_t re,
                                                  int64_t n, int l32, int khalf) {
    const int64_t H = static_cast<int64_t>(o.q_heads) * 128;
    const int64_t kvd = static_cast<int64_t>(o.kv_heads) * 128;
    const int seq = static_cast<int>(o.seq);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        // One 32-row block: positions and (cos, sin) of all its rows and this
        // lane's columns are fetched first, so the block waits for the table
        // once instead of once per element.
        int bq[4], sq[4];
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            const int rr = static_cast<int>(wave_row0 + i * 32 + 8 * rq + 4 * khalf);
            bq[rq] = rr / seq;
            sq[rq] = rr - bq[rq] * seq;
        }
        // row e of a run of four: its (sequence, position), the run's own unless
        // a sequence ends inside it (sequences hold at least four rows)
        auto row_pos = [&](int rq, int e, int& b, int& sp) __attribute__((always_inline)) {
            const bool wrap = kAnySeq && sq[rq] + e >= seq;
            b = bq[rq] + (wrap ? 1 : 0);
            sp = sq[rq] + e - (wrap ? seq : 0);
        };
        float2 cs[WN][4][4];
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const int64_t col = wave_col0 + j * 32 + l32;
            const bool rot = col < H + kvd;  // uniform over the 32-column block
            const int pr = static_cast<int>(col & 127) >> 1;
#pragma unroll
            for (int rq = 0; rq < 4; ++rq)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    int b, sp;
                    row_pos(rq, e, b, sp);
                    cs[j][rq][e] = rot ? o.rope[static_cast<int64_t>(sp) * 64 + pr] : make_float2(1.f, 0.f);
                }
        }
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            const int64_t row = wave_row0 + i * 32 + 8 * rq + 4 * khalf;  // rows row .. row + 3
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const int64_t col = wave_col0 + j * 32 + l32;
                float v[4], pv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = acc[i][j][4 * rq + e];
                    pv[e] = __shfl_xor(v[e], 1, 64);
                }
                if (col >= n || row >= re) continue;
                const int d = static_cast<int>(col & 127);
                if (col < H + kvd) {
                    const bool isq = col < H;
                    uint16_t* const base = isq ? o.q : o.k;
                    const int64_t heads = isq ? o.q_heads : o.kv_heads;
                    const int64_t head = isq ? col >> 7 : (col - H) >> 7;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (kAnySeq && row + e >= re) break;
                        int b, sp;
                        row_pos(rq, e, b, sp);
                        const float2 c = cs[j][rq][e];
                        // (even, odd) -> (even c - odd s, odd c + even s), the same
                        // fused operations as qkv_rope_epilogue_staged
                        const float r0 = (d & 1) ? fmaf(v[e], c.x, pv[e] * c.y) : fmaf(v[e], c.x, -(pv[e] * c.y));
                        base[((static_cast<int64_t>(b) * heads + head) * seq + sp) * 128 + d] = f32_to_bf16(r0);
                    }
                } else {
                    const int64_t hv = (col - H - kvd) >> 7;
                    if (!kAnySeq || seq % 4 == 0) {  // four positions of one sequence, 8-byte aligned
                        uint2 pk;
                        pk.x = pack_bf16x2(v[0], v[1]);
                        pk.y = pack_bf16x2(v[2], v[3]);
                        *reinterpret_cast<uint2*>(o.vt + ((static_cast<int64_t>(bq[rq]) * o.kv_heads + hv) * 128 + d) * o.ld_vt + sq[rq]) = pk;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (kAnySeq && row + e >= re) break;
                            int b, sp;
                            row_pos(rq, e, b, sp);
                            o.vt[((static_cast<int64_t>(b) * o.kv_heads + hv) * 128 + d) * o.ld_vt + sp] = f32_to_bf16(v[e]);
                        }
                    }
                }
            }
        }
    }
}

// The same epilogue for a wave's block of a four-wave tile (128 x 128 of a
// 256 x 256 tile, or 64 x 64 of a 128 x 128 one), through the wave's own LDS
// stage array: for each 32-row block the accumulators go to LDS as fp32
// [32][kCols] (column c of row r at c ^ ((r & 4) << 3), so the two row halves
// of a write use different banks), then every lane reads 8 consecutive
// columns of one row, rotates its 4 pairs with a 32-byte read of the
// (cos, sin) table (issued one row block ahead) and writes 16 bytes of Q or K.
// A V^T block is staged transposed and leaves as 16-byte runs of positions; a
// block past the last column, or V^T when the sequence length is not a
// multiple of 8, takes the per-lane path.
template <int WM, int WN, bool kAnySeq>
__device__ __forceinline__ void qkv_rope_epilogue_staged(const QkvRopeOut& o, const floatx16 (&acc)[WM][WN],
                                                         int64_t wave_row0, int64_t wave_col0, int64_t re,
                                                         int64_t n, int lane, float* stage) {
    static_assert((WM == 4 && WN == 4) || (WM == 2 && WN == 2), "128 x 128 or 64 x 64 per wave");
    constexpr int kCols = 32 * WN;          // columns of the wave block (within one head)
    constexpr int kPos = 32 * WM;           // rows (positions) of the wave block
    const int l32 = lane & 31, khalf = lane >> 5;
    const int64_t H = static_cast<int64_t>(o.q_heads) * 128;
    const int64_t kvd = static_cast<int64_t>(o.kv_heads) * 128;
    const int64_t seq = o.seq;
    if (wave_col0 + kCols > n || (wave_col0 >= H + kvd && seq % 8 != 0)) {
        qkv_rope_epilogue<WM, WN, kAnySeq>(o, acc, wave_row0, wave_col0, re, n, l32, khalf);
        return;
    }
    const int col_in_head = static_cast<int>(wave_col0 & 127);  // 0, or 64 for 64-column blocks
    if (wave_col0 >= H + kvd) {
        // V^T block: bf16 [kCols d][kPos s] in LDS; 8-byte granule g of row d
        // sits at g ^ x(d), which spreads the 32 rows of a write over distinct
        // bank pairs (rows are 256 B apart for kPos 128, 128 B for 64).
        // Then 16-byte runs of 8 positions of one d row go out whole.
        constexpr int kGran = kPos / 4;
        auto swz = [](int d) { return kGran == 32 ? (d & 31) : ((d >> 1) & (kGran - 1)); };
        uint16_t* const st = reinterpret_cast<uint16_t*>(stage);
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int rq = 0; rq < 4; ++rq) {
                    const int d = j * 32 + l32;
                    const int g = i * 8 + 2 * rq + khalf;  // positions 4 g .. 4 g + 3
                    uint2 pk;
                    pk.x = cvt_pk_bf16(acc[i][j][4 * rq + 0], acc[i][j][4 * rq + 1]);
                    pk.y = cvt_pk_bf16(acc[i][j][4 * rq + 2], acc[i][j][4 * rq + 3]);
                    *reinterpret_cast<uint2*>(st + d * kPos + (g ^ swz(d)) * 4) = pk;
                }
        constexpr int kRunLanes = kPos / 8;         // lanes per d row (8 positions each)
        constexpr int kRowsPer = 64 / kRunLanes;    // d rows per instruction
        const int64_t hv = (wave_col0 - H - kvd) >> 7;
        const int c = lane % kRunLanes;             // positions 8 c .. 8 c + 7 of a d row
        const int64_t grow = wave_row0 + 8 * c;     // first of the 8 rows
        const int64_t b = static_cast<uint32_t>(grow) / static_cast<uint32_t>(seq);
        const int64_t sp = grow - b * seq;
        uint16_t* const dst0 = o.vt + ((b * o.kv_heads + hv) * 128 + col_in_head) * o.ld_vt + sp;
#pragma unroll
        for (int t = 0; t < kCols / kRowsPer; ++t) {
            const int d = kRowsPer * t + lane / kRunLanes;
            const int x = swz(d);
            uint4 v = *reinterpret_cast<const uint4*>(st + d * kPos + ((2 * c) ^ (x & ~1)) * 4);
            if (x & 1) v = make_uint4(v.z, v.w, v.x, v.y);  // the two granules of the run swapped
            uint16_t* const dst = dst0 + d * o.ld_vt;
            if (grow + 8 <= re && sp + 8 <= seq) {
                *reinterpret_cast<uint4*>(dst) = v;
            } else {
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int64_t r = grow + e;
                    if (r >= re) break;
                    const int64_t be = r / seq, se = r - be * seq;
                    o.vt[((be * o.kv_heads + hv) * 128 + col_in_head + d) * o.ld_vt + se] =
                        static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
                }
            }
        }
        return;
    }
    const bool isq = wave_col0 < H;
    uint16_t* const base = isq ? o.q : o.k;
    const int64_t heads = isq ? o.q_heads : o.kv_heads;
    const int64_t head = isq ? (wave_col0 >> 7) : ((wave_col0 - H) >> 7);
    constexpr int kChunkLanes = kCols / 8;        // lanes per row when reading back
    constexpr int kRowsPer = 64 / kChunkLanes;    // rows per read-back step
    constexpr int kSteps = 32 / kRowsPer;         // steps per 32-row block
    const int c8 = lane % kChunkLanes;            // this lane's 8-column chunk
    const int lrow = lane / kChunkLanes;
    // (sequence, position) of this lane's first row in block i.  Its rows are
    // kRowsPer t + lrow, so later ones advance the position by kRowsPer,
    // wrapping into the next sequence: one division per block (rows and the
    // sequence length fit 32 bits on this path) instead of one per row.
    const uint32_t useq = static_cast<uint32_t>(seq);
    auto block_pos = [&](int i, uint32_t& b, uint32_t& sp) {
        const uint32_t g = static_cast<uint32_t>(wave_row0 + i * 32 + lrow);
        b = g / useq;
        sp = g - b * useq;
    };
    auto next_pos = [&](uint32_t& b, uint32_t& sp) {
        sp += kRowsPer;
        if (sp >= useq) {  // a sequence boundary (several when seq < kRowsPer)
            const uint32_t q = sp / useq;
            b += q;
            sp -= q * useq;
        }
    };
    // (cos, sin) of this lane's 4 pairs for its rows of block i: all table
    // reads of a block are issued one block ahead, so the block never waits
    // for the table.  (Rows past the end read a valid row, unused.)
    const int pair0 = col_in_head / 2 + c8 * 4;
    auto table = [&](int i, float4 (&cs)[kSteps][2]) {
        uint32_t bt, sp;
        block_pos(i, bt, sp);
#pragma unroll
        for (int t = 0; t < kSteps; ++t) {
            if (t) next_pos(bt, sp);
            const float4* src = reinterpret_cast<const float4*>(o.rope + static_cast<int64_t>(sp) * 64 + pair0);
            cs[t][0] = src[0];
            cs[t][1] = src[1];
        }
    };
    float4 cs[2][kSteps][2];
    table(0, cs[0]);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        if (i + 1 < WM) table(i + 1, cs[(i + 1) & 1]);
        // LDS accesses of one wave complete in order: the reads below see
        // these writes, and the next block's writes follow these reads.
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 8 * (r >> 2) + 4 * khalf + (r & 3);
                stage[row * kCols + ((j * 32 + l32) ^ ((row & 4) << 3))] = acc[i][j][r];
            }
        uint32_t b, sp;
        block_pos(i, b, sp);
#pragma unroll
        for (int t = 0; t < kSteps; ++t) {
            if (t) next_pos(b, sp);
            const int row = kRowsPer * t + lrow;
            const float* src = stage + row * kCols + ((c8 * 8) ^ ((row & 4) << 3));
            const float4 v0 = *reinterpret_cast<const float4*>(src);
            const float4 v1 = *reinterpret_cast<const float4*>(src + 4);
            const int64_t grow = wave_row0 + i * 32 + row;
            if (grow >= re) continue;
            const float4 cs0 = cs[i & 1][t][0], cs1 = cs[i & 1][t][1];  // this lane's 4 pairs
            // hardware RNE pair conversion: the same bits as pack_bf16x2 for finite values
            auto rot = [](float e, float od, float c, float sn) {
                return cvt_pk_bf16(fmaf(e, c, -(od * sn)), fmaf(od, c, e * sn));
            };
            uint4 pk;
            pk.x = rot(v0.x, v0.y, cs0.x, cs0.y);
            pk.y = rot(v0.z, v0.w, cs0.z, cs0.w);
            pk.z = rot(v1.x, v1.y, cs1.x, cs1.y);
            pk.w = rot(v1.z, v1.w, cs1.z, cs1.w);
            *reinterpret_cast<uint4*>(base + ((static_cast<int64_t>(b) * heads + head) * seq + sp) * 128 +
                                      col_in_head + c8 * 8) = pk;
        }
    }
}

// GLU store epilogue of a wave's 128 x 64 output block in the four-wave
// 256 x 256 tile (bf16 out), through a 16 KB LDS region of its own: the
// silu-combined values go to LDS as bf16 [128 rows][64 columns] (column c of
// row r at c ^ ((r & 4) << 3), so the two row halves of a write hit different
// banks), then every lane stores 16-byte row chunks, instead of one 2-byte
// element per lane per store instruction.  The arithmetic is the generic
// epilogue's, value for value.
template <int EPI>
__device__ __forceinline__ void glu_epilogue_staged(const TiledArgs& p, const floatx16 (&acc)[4][4],
                                                    int64_t wrow0, int64_t wcol0, int64_t re,
                                                    const float* scales, int lane, uint16_t* stage) {
    const int l32 = lane & 31, khalf = lane >> 5;
    // wcol0: the first of this wave's 64 output columns
    float sc_lo[2], sc_hi[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int64_t cc = min(wcol0 + j * 32 + l32, p.n - 1);
        sc_lo[j] = scales ? scales[cc] : 1.f;
        sc_hi[j] = scales ? scales[p.n + cc] : 1.f;
    }
    // Two rows at a time through the hardware RNE converter (the same bits as
    // f32_to_bf16 for finite values); unscaled weights skip the multiplies.
    auto combine_rows = [&](auto scaled_c) __attribute__((always_inline)) {
        constexpr bool kScaled = decltype(scaled_c)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    float v[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float g = kScaled ? acc[i][2 * j][r + e] * sc_lo[j] : acc[i][2 * j][r + e];
                        const float u = kScaled ? acc[i][2 * j + 1][r + e] * sc_hi[j] : acc[i][2 * j + 1][r + e];
                        v[e] = glu_combine(EPI, g, u);
                    }
                    const uint32_t pk = cvt_pk_bf16(v[0], v[1]);
                    const int row = i * 32 + 8 * (r >> 2) + 4 * khalf + (r & 3);  // rows row, row + 1
                    const int col = j * 32 + l32;
                    stage[row * 64 + (col ^ ((row & 4) << 3))] = static_cast<uint16_t>(pk);
                    stage[(row + 1) * 64 + (col ^ (((row + 1) & 4) << 3))] = static_cast<uint16_t>(pk >> 16);
                }
    };
    if (scales) combine_rows(std::true_type{});
    else combine_rows(std::false_type{});
    // a wave's LDS accesses complete in order: the reads see the writes
    uint16_t* const out = static_cast<uint16_t*>(p.c);
    const int c8 = lane & 7;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const int row = t * 8 + (lane >> 3);
        const uint4 v = *reinterpret_cast<const uint4*>(stage + row * 64 + ((c8 * 8) ^ ((row & 4) << 3)));
        const int64_t grow = wrow0 + row, col = wcol0 + c8 * 8;
        if (grow >= re) continue;
        uint16_t* const dst = out + grow * p.ldc + col;
        if (col + 8 <= p.n) {
            *reinterpret_cast<uint4*>(dst) = v;
        } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (col + e < p.n) dst[e] = static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// Scheduling groups for one interleaved half slab: NM MFMAs; the NR LDS reads
// of the next half go one after each of the first MFMAs (so the last has most
// of the half to land before its MFMA needs it), and the NV VMEM loads are
// spread over the MFMAs after them.
template <int NM, int NR, int NV, int I = 0>
__device__ __forceinline__ void interleave_groups() {
    if constexpr (I < NM) {
        constexpr int kRest = NM - (NR < NM ? NR : NM);  // MFMAs after the reads
        constexpr int kJ = I - (NM - kRest);              // index among them
        constexpr int kLoadsHere = (NV == 0 || kJ < 0) ? 0
            : (kRest == 0 ? (I == NM - 1 ? NV : 0) : (kJ + 1) * NV / kRest - kJ * NV / kRest);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        if constexpr (I < NR) __builtin_amdgcn_sched_group_barrier(0x100, I == NM - 1 ? NR - I : 1, 0);  // DS read
        if constexpr (kLoadsHere > 0) __builtin_amdgcn_sched_group_barrier(0x020, kLoadsHere, 0);  // VMEM read
        interleave_groups<NM, NR, NV, I + 1>();
    }
}

// Scheduling groups for a run of NM MFMAs that also reads fragments and
// issues loads: one LDS fragment read after each of the first NR MFMAs, and NV
// VMEM instructions (LDS DMA) spread evenly over all NM, so the four waves of
// a CU never queue a burst of LDS reads or of DMA requests.
template <int NM, int NR, int NV, int I = 0>
__device__ __forceinline__ void spread_reads_loads() {
    if constexpr (I < NM) {
        constexpr int loads = (I + 1) * NV / NM - I * NV / NM;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          // MFMA
        if constexpr (I < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // DS read
        if constexpr (loads > 0) __builtin_amdgcn_sched_group_barrier(0x020, loads, 0);  // VMEM
        spread_reads_loads<NM, NR, NV, I + 1>();
    }
}

// Scheduling groups for NM MFMAs with NV VALU instructions spread over them.
template <int NM, int NV, int I = 0>
__device__ __forceinline__ void spread_valu() {
    if constexpr (I < NM) {
        constexpr int here = (I + 1) * NV / NM - I * NV / NM;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                        // MFMA
        if constexpr (here > 0) __builtin_amdgcn_sched_group_barrier(0x002, here, 0);  // VALU
        spread_valu<NM, NV, I + 1>();
    }
}

// Tile of this workgroup in a direct-to-LDS launch.  Grouped (p.offsets):
// blockIdx.x is the column tile, blockIdx.y walks the row tiles of the groups
// in order (group g: ceil(rows_g / BM) tiles; false past the last).  Dense: a
// 1-D grid of tiles_m x tiles_n tiles in the XCD-aware order.  Sets the group
// g, its row range [rb, re) and the tile (tm, tn).
template <int BM>
__device__ __forceinline__ bool dma_tile_coords(const TiledArgs& p, int tiles_m, int tiles_n, int& g,
                                                int64_t& rb, int64_t& re, int64_t& tm, int64_t& tn) {
    g = 0;
    rb = 0;
    re = p.m;
    if (p.offsets) {
        tn = blockIdx.x;
        int64_t t = blockIdx.y;
        auto bound = [&](int e) {
            return min(max(static_cast<int64_t>(p.offsets[e]), int64_t(0)), p.m);
        };
        g = -1;
        for (int e = 0; e < p.groups; ++e) {
            const int64_t rows = max(bound(e + 1) - bound(e), int64_t(0));
            const int64_t tiles = (rows + BM - 1) / BM;
            if (t < tiles) { g = e; break; }
            t -= tiles;
        }
        if (g < 0) return false;
        rb = bound(g);
        re = max(bound(g + 1), rb);
        tm = t;
    } else {
        // XCD-aware order: the dispatcher deals consecutive workgroup ids to
        // the XCDs in turn, so hand each XCD a contiguous run of tiles and
        // walk them in groups of 8 M-tiles (A and B tiles shared in one L2).
        const int64_t total = static_cast<int64_t>(tiles_m) * tiles_n;
        const int64_t i = blockIdx.x;
        const int64_t x = p.xcds;
        const int64_t full = total - total % x;
        int64_t L = i;
        if (i < full) L = (i % x) * (full / x) + i / x;
        constexpr int64_t kGroupM = 8;
        const int64_t group = L / (kGroupM * tiles_n);
        const int64_t first_m = group * kGroupM;
        const int64_t gsize = min(static_cast<int64_t>(tiles_m) - first_m, kGroupM);
        const int64_t in_group = L % (kGroupM * tiles_n);
        tm = first_m + in_group % gsize;
        tn = in_group / gsize;
    }
    return true;
}

// Store epilogue of one wave's (BM / 2) x (BN / (NW / 2)) block of a
// direct-to-LDS tile (wave (wm, wn) of the 2 x (NW / 2) wave grid), for every
// epilogue but the staged GLU one of the 64-k slab tile.  qkv_stage: this
// wave's own LDS region for the staged QKV epilogue (every wave calls this
// function: the staged path meets the others at a barrier first).
template <int BM, int BN, int NW, int EPI, bool PP, int kWavesM = 2, bool kAnySeq = false, int WM, int WN>
__device__ __forceinline__ void dma_tile_epilogue(const TiledArgs& p, const floatx16 (&acc)[WM][WN], int wm,
                                                  int wn, int64_t row0, int64_t ncol0, int64_t re,
                                                  const float* scales, float* qkv_stage) {
    constexpr bool kGlu = EpiTraits<EPI>::glu;
    constexpr int kWavesN = NW / kWavesM;
    static_assert(WM == BM / (32 * kWavesM) && WN == BN / (32 * kWavesN), "wave block shape");
    // The epilogues take the lane index again from the lane mask, so no
    // lane-derived value of the prologue has to live through the main loop.
    const int elane = static_cast<int>(__lane_id());
    const int el32 = elane & 31, ekhalf = elane >> 5;
    // Epilogue: 32x32 D layout, lane holds column (lane & 31) and rows
    // 8 (r / 4) + 4 (lane >> 5) + (r % 4).  The output dtype and the scales are
    // resolved once per tile, a lane's scales (its columns are fixed) are read
    // once, and the residual loads of a group of half blocks (at clamped,
    // always valid addresses) all precede the group's first store, so the
    // group waits for memory once instead of once per element; only the
    // stores are guarded.
    if constexpr (EPI != kEpiQkvRope) {
        constexpr int kCols = kGlu ? WN / 2 : WN;  // output columns per lane
        int64_t cols[kCols];
        float sc_lo[kCols], sc_hi[kCols];
#pragma unroll
        for (int j = 0; j < kCols; ++j) {
            cols[j] = kGlu ? ncol0 + (wn * WN / 2 + j) * 32 + el32 : ncol0 + wn * (BN / kWavesN) + j * 32 + el32;
            const int64_t cc = min(cols[j], p.n - 1);
            sc_lo[j] = scales ? scales[cc] : 1.f;
            sc_hi[j] = (kGlu && scales) ? scales[p.n + cc] : 1.f;
        }
        // Residual rows [0, m) addressable with 32-bit byte offsets: loads go
        // through a buffer resource (reads past its end return 0, and every
        // load of a column >= n feeds only an output that is not stored).
        const bool res_rsrc_ok = EPI == SFG_EPI_RESIDUAL && p.residual &&
                                 static_cast<uint64_t>(p.m) * p.ldr * 4 <= 0xFFFFFFFFull;
        const buf_rsrc res_rsrc = make_rsrc(p.residual, res_rsrc_ok ? static_cast<uint32_t>(p.m * p.ldr * 4) : 0u);
        auto store_tile = [&](auto* out) {
            using OutT = std::remove_pointer_t<decltype(out)>;
            // Residual epilogues load the residual of kGroup half blocks before
            // the first of their stores (each element is still read before it
            // is written, so an in-place residual stays correct): the tile
            // waits for memory 2 WM / kGroup times instead of 2 WM.
            // (four-wave 256 x 256 tiles only: the others have no registers for it).
            constexpr int kGroup = (EPI == SFG_EPI_RESIDUAL && NW == 4 && BM == 256 && BN == 256) ? 4 : 1;
#pragma unroll
            for (int g0 = 0; g0 < 2 * WM; g0 += kGroup) {
                float res[kGroup][8][kCols];
                if constexpr (EPI == SFG_EPI_RESIDUAL) {
                    if (kGroup > 1 && res_rsrc_ok) {
                        // 32-bit offsets through a buffer resource over the
                        // residual rows [0, m): one offset per row, the column
                        // blocks 128 B apart as immediate offsets
#pragma unroll
                        for (int h = 0; h < kGroup; ++h) {
                            const int ih = g0 + h, i = ih >> 1, r0 = (ih & 1) * 8;
                            const int64_t rbase = row0 + wm * (BM / kWavesM) + i * 32 + 4 * ekhalf;
#pragma unroll
                            for (int rr = 0; rr < 8; ++rr) {
                                const int r = r0 + rr;
                                const int64_t row = min(rbase + 8 * (r >> 2) + (r & 3), re - 1);
                                const uint32_t off = static_cast<uint32_t>((row * p.ldr + cols[0]) * 4);
#pragma unroll
                                for (int j = 0; j < kCols; ++j)
                                    res[h][rr][j] = __builtin_bit_cast(
                                        float, __builtin_amdgcn_raw_buffer_load_b32(res_rsrc, off + j * 128, 0, 0));
                            }
                        }
                    } else {
#pragma unroll
                        for (int h = 0; h < kGroup; ++h) {
                            const int ih = g0 + h, i = ih >> 1, r0 = (ih & 1) * 8;
                            const int64_t rbase = row0 + wm * (BM / kWavesM) + i * 32 + 4 * ekhalf;
#pragma unroll
                            for (int rr = 0; rr < 8; ++rr)
#pragma unroll
                                for (int j = 0; j < kCols; ++j) {
                                    const int r = r0 + rr;
                                    const int64_t row = min(rbase + 8 * (r >> 2) + (r & 3), re - 1);
                                    res[h][rr][j] = p.residual[row * p.ldr + min(cols[j], p.n - 1)];
                                }
                        }
                    }
                }
#pragma unroll
                for (int h = 0; h < kGroup; ++h) {  // half 32-row blocks: 8 accumulator rows each
                    const int ih = g0 + h, i = ih >> 1, r0 = (ih & 1) * 8;
                    const int64_t rbase = row0 + wm * (BM / kWavesM) + i * 32 + 4 * ekhalf;
#pragma unroll
                    for (int rr = 0; rr < 8; ++rr) {
                        const int r = r0 + rr;
                        const int64_t row = rbase + 8 * (r >> 2) + (r & 3);
#pragma unroll
                        for (int j = 0; j < kCols; ++j) {
                            float v;
                            if constexpr (kGlu) {
                                v = glu_combine(EPI, acc[i][2 * j][r] * sc_lo[j], acc[i][2 * j + 1][r] * sc_hi[j]);
                            } else {
                                v = acc[i][j][r] * sc_lo[j];
                                if constexpr (EPI == SFG_EPI_RESIDUAL) v += res[h][rr][j];
                            }
                            if (row < re && cols[j] < p.n) {
                                if constexpr (sizeof(OutT) == 4) out[row * p.ldc + cols[j]] = v;
                                else out[row * p.ldc + cols[j]] = f32_to_bf16(v);
                            }
                        }
                    }
                }
            }
        };
        if (p.c_dtype == SFG_F32) store_tile(static_cast<float*>(p.c));
        else store_tile(static_cast<uint16_t*>(p.c));
    }
    if constexpr (EPI == kEpiQkvRope) {
        // four-wave tiles with square wave blocks stage through LDS (a wave's
        // own stage array holds its fp32 32-row block and its V^T block)
        constexpr bool kStaged = (NW == 4 || kWavesM == 4) && !PP && ((WM == 4 && WN == 4) || (WM == 2 && WN == 2));
        if constexpr (kStaged) {
            // every wave's reads of the last slabs are done before any wave
            // reuses its array as staging (the DMA drained above)
            wait_lds();
            barrier_no_fence();
            qkv_rope_epilogue_staged<WM, WN, kAnySeq>(p.qkv, acc, row0 + wm * (BM / kWavesM), ncol0 + wn * (BN / kWavesN),
                                             re, p.n, elane, qkv_stage);
        } else {
            const int64_t wrow0 = row0 + wm * (BM / kWavesM), wcol0 = ncol0 + wn * (BN / kWavesN);
            qkv_rope_epilogue<WM, WN, kAnySeq>(p.qkv, acc, wrow0, wcol0, re, p.n, el32, ekhalf);
        }
    }
}

}  // namespace sfg
