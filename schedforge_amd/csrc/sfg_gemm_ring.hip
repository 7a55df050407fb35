// sfg_gemm_ring.hip -- the MFMA GEMM from 65 rows up: bf16 or int8 weights, dense
// or grouped, optionally split over K; and the fp32 GEMM.
#include "sfg_gemm_tile.hpp"

namespace sfg {

// ===========================================================================
// Ring GEMM: BM x BN output tile, NW waves (four or eight) two abreast, K in slabs
// of 64 through a ring of NS LDS stages filled by DMA (global -> LDS, no registers).
//
// With 65 .. ~1000 rows a launch has one or two tiles per CU, so nothing else
// on the CU hides a slab's latency: what bounds the tile is how many bytes it
// keeps in flight.  The ring holds most of the CU's 160 KB for one workgroup
// (NS - 1 slabs of 12 - 48 KB in flight), one barrier per 64 k.  (int8: the
// conversion bounds it; a slab of half the bytes takes as long.)
//
// B rows come from [N][K] or from the fragment-tiled layout (the DMA lanes pick
// their chunks).  A rows are 128 B with 16-byte chunk c of row r in slot c ^ ((r >> 1) & 7);
// bf16 B rows the same; int8 B rows are 64 B with chunk c in slot
// c ^ ((r >> 2) & 3), converted to bf16 (exactly) between the LDS read and the
// MFMA, under the matrix pipe.  The MFMA k order is free as long as A and B
// agree: int8 step j of a slab takes k = 32 (j / 2) + 16 half + 8 (j % 2) + [0, 8),
// so one 16-byte read feeds two steps.
// fp32 operands (slabs of 32 k, the same 128 bytes) run on
// v_mfma_f32_32x32x2_f32, where the matrix pipe bounds the tile.
// The last slab's chunks past K are loaded from past the end of the buffer
// resource, which returns zeros (K is a whole number of 16-byte chunks).
//
// SPLIT: blockIdx.y takes a contiguous range of slabs and the fp32 sums go to
// part [split][m][B rows]; gemm_splitk_reduce_kernel adds them in split order.
// ===========================================================================
template <int BDT, int BM, int BN>
constexpr int kRingStageElems = BM * 64 + BN * (BDT == SFG_I8 ? 32 : 64);  // uint16 units

// k per slab: 128 bytes of an A row
template <int BDT>
constexpr int kRingSlabK = BDT == SFG_F32 ? 32 : 64;

template <int BDT, int BM, int BN, int NW, int NS, int EPI, bool SPLIT>
__global__ __launch_bounds__(NW * 64) void gemm_ring_kernel(TiledArgs p, int tiles_m, int tiles_n, float* part) {
    constexpr bool kGlu = EpiTraits<EPI>::glu;
    constexpr bool kI8 = BDT == SFG_I8, kF32 = BDT == SFG_F32;
    constexpr int kSlabK = kRingSlabK<BDT>;
    constexpr int kAElem = kF32 ? 4 : 2, kBElem = kI8 ? 1 : kAElem;
    constexpr int kWavesM = NW / 2;
    constexpr int WM = BM / (32 * kWavesM), WN = BN / 64;  // 32 x 32 tiles per wave
    constexpr int kStage = kRingStageElems<BDT, BM, BN>;
    constexpr int kBRow = kI8 ? 32 : 64;                 // uint16 units per B row in LDS
    constexpr int kLoadsA = BM / (8 * NW), kLoadsB = BN / ((kI8 ? 16 : 8) * NW);  // DMA instructions per wave per slab
    constexpr int kLoads = kLoadsA + kLoadsB;
    static_assert(NS >= 3 && NS <= 6 && (NS - 2) * kLoads < 64, "ring depth");
    static_assert(!kGlu || WN % 2 == 0, "GLU tiles pair gate and up blocks");
    // one array per stage: the compiler tells loads in flight from the stage
    // being read by the array
    __shared__ __attribute__((aligned(1024))) uint16_t s0[kStage];
    __shared__ __attribute__((aligned(1024))) uint16_t s1[kStage];
    __shared__ __attribute__((aligned(1024))) uint16_t s2[kStage];
    __shared__ __attribute__((aligned(1024))) uint16_t s3[NS > 3 ? kStage : 8];
    __shared__ __attribute__((aligned(1024))) uint16_t s4[NS > 4 ? kStage : 8];
    __shared__ __attribute__((aligned(1024))) uint16_t s5[NS > 5 ? kStage : 8];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    constexpr int kOutCols = kGlu ? BN / 2 : BN;

    int g;
    int64_t rb, re, tm, tn;
    if (!dma_tile_coords<BM>(p, tiles_m, tiles_n, g, rb, re, tm, tn)) return;
    const int64_t row0 = rb + tm * BM;
    if (row0 >= re) return;
    const int64_t ncol0 = tn * kOutCols;
    const float* scales = p.scales ? p.scales + static_cast<int64_t>(g) * p.s_group_stride : nullptr;

    // slabs of this workgroup
    const int64_t all_slabs = (p.k + kSlabK - 1) / kSlabK;
    int64_t slab0 = 0, slab1 = all_slabs;
    if constexpr (SPLIT) {
        slab0 = all_slabs * blockIdx.y / gridDim.y;
        slab1 = all_slabs * (blockIdx.y + 1) / gridDim.y;
    }
    // 16-byte chunks of a row the last slab holds (0: all)
    const int tail_a = static_cast<int>(p.k % kSlabK) * kAElem / 16, tail_b = static_cast<int>(p.k % kSlabK) * kBElem / 16;

    // DMA sources.  A: instruction i fills rows 8 (4 i + wave) + lane / 8, slot
    // lane % 8.  Rows past the tile read its first row (never stored); a
    // gathered id outside A starts past A's resource and reads zeros.
    const uint32_t a_bytes = static_cast<uint32_t>(p.a_rows_limit * p.lda * kAElem);
    const buf_rsrc ra = make_rsrc(p.a, a_bytes);
    uint32_t a_off[kLoadsA];
    const int a_row = lane >> 3, a_slot = lane & 7;
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) {
        const int local = (NW * i + wave) * 8 + a_row;
        const int64_t r = row0 + local;
        int64_t src = r < re ? r : row0;
        if (p.a_rows) src = p.a_rows[src];
        const int chunk = a_slot ^ ((local >> 1) & 7);
        a_off[i] = (src < 0 || src >= p.a_rows_limit) ? a_bytes
                                                      : static_cast<uint32_t>(src * p.lda * kAElem + chunk * 16);
    }
    const uint32_t b_bytes = static_cast<uint32_t>((kGlu ? 2 : 1) * p.n * p.ldb * kBElem);
    const buf_rsrc rbs = make_rsrc(static_cast<const char*>(p.b) + static_cast<int64_t>(g) * p.b_group_stride * kBElem,
                                   b_bytes);
    uint32_t b_off[kLoadsB];
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) {
        const int local = kI8 ? (NW * i + wave) * 16 + (lane >> 2) : (NW * i + wave) * 8 + (lane >> 3);
        const int chunk = kI8 ? (lane & 3) ^ ((local >> 2) & 3) : (lane & 7) ^ ((local >> 1) & 7);
        int64_t brow;
        if (kGlu) {
            const int block = local >> 5;
            const int64_t col = ncol0 + (block >> 1) * 32 + (local & 31);
            brow = col < p.n ? ((block & 1) ? p.n + col : col) : 0;
        } else {
            const int64_t col = ncol0 + local;
            brow = col < p.n ? col : 0;
        }
        if constexpr (!kF32) {
            if (p.b_tiled) {
                // 16-row x 128-k tiles: 16-byte chunk c of a row's 64-k half sits
                // in (bf16) fragment c / 4, lane group c % 4; (int8) fragment
                // c % 2, lane group c / 2
                const int64_t at = (brow / 16) * (p.k / 128) * (2048 * kBElem) + (brow % 16) * 16 +
                                   (kI8 ? (chunk & 1) * 1024 + (chunk >> 1) * 256 : (chunk >> 2) * 1024 + (chunk & 3) * 256);
                b_off[i] = static_cast<uint32_t>(at);
                continue;
            }
        }
        b_off[i] = static_cast<uint32_t>((brow * p.ldb) * kBElem + chunk * 16);
    }
    // DMA instructions [i0, i1) of slab s into stage st (A's first, then B's).
    // Slabs past the end re-fetch the last one.
    auto issue = [&](uint16_t* st, int64_t s, int i0, int i1) __attribute__((always_inline)) {
        const int64_t sl = min(s, slab1 - 1);
        const bool tail = tail_a != 0 && sl == all_slabs - 1;  // wave-uniform
        const uint32_t ka = static_cast<uint32_t>(sl * 128), kb = !kF32 && p.b_tiled ? static_cast<uint32_t>((sl >> 1) * (2048 * kBElem) + (sl & 1) * (kI8 ? 512 : 2048))
                                                                                      : static_cast<uint32_t>(sl * kSlabK * kBElem);
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
            if (i < i0 || i >= i1) continue;
            const int local = (NW * i + wave) * 8 + a_row;
            const uint32_t off = tail && (a_slot ^ ((local >> 1) & 7)) >= tail_a ? a_bytes : a_off[i];
            lds_dma16_buf(ra, off, ka, st + (NW * i + wave) * 8 * 64);
        }
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) {
            if (i + kLoadsA < i0 || i + kLoadsA >= i1) continue;
            const int local = kI8 ? (NW * i + wave) * 16 + (lane >> 2) : (NW * i + wave) * 8 + (lane >> 3);
            const bool up = (kI8 ? (lane & 3) ^ ((local >> 2) & 3) : (lane & 7) ^ ((local >> 1) & 7)) >= tail_b;
            const uint32_t off = tail && up ? b_bytes : b_off[i];
            lds_dma16_buf(rbs, off, kb, st + BM * 64 + (NW * i + wave) * (kI8 ? 16 : 8) * kBRow);
        }
    };

    floatx16 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const int l32 = lane & 31, khalf = lane >> 5;
    const int asw = (l32 >> 1) & 7, bsw = kI8 ? (l32 >> 2) & 3 : asw;
    // A and B fragments of step J, a quarter of the slab (int8: raw, both steps
    // of the 32-k group at even J)
    uint4 fa[2][WM], fb[2][WN], fq[2][kI8 ? WN : 1];
    auto frags = [&](const uint16_t* st, auto j_c) __attribute__((always_inline)) {
        constexpr int J = decltype(j_c)::value;
        const int ca = kI8 ? 4 * (J >> 1) + 2 * khalf + (J & 1) : 2 * J + khalf;
#pragma unroll
        for (int i = 0; i < WM; ++i)
            fa[J & 1][i] = *reinterpret_cast<const uint4*>(st + (wm * (BM / kWavesM) + i * 32 + l32) * 64 + (ca ^ asw) * 8);
        const uint16_t* sb = st + BM * 64;
        if constexpr (kI8) {
            if constexpr ((J & 1) == 0) {
#pragma unroll
                for (int i = 0; i < WN; ++i)
                    fq[(J >> 1) & 1][i] = *reinterpret_cast<const uint4*>(
                        sb + (wn * (BN / 2) + i * 32 + l32) * kBRow + (((J & 2) + khalf) ^ bsw) * 8);
            }
        } else {
#pragma unroll
            for (int i = 0; i < WN; ++i)
                fb[J & 1][i] = *reinterpret_cast<const uint4*>(
                    sb + (wn * (BN / 2) + i * 32 + l32) * kBRow + ((2 * J + khalf) ^ bsw) * 8);
        }
    };
    // int8: the bf16 fragments of step J from the raw ones
    auto convert = [&](auto j_c) __attribute__((always_inline)) {
        constexpr int J = decltype(j_c)::value;
        if constexpr (kI8) {
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const uint4 q = fq[(J >> 1) & 1][j];
                fb[J & 1][j] = (J & 1) ? i8x8_to_bf16x8(q.z, q.w) : i8x8_to_bf16x8(q.x, q.y);
            }
        }
    };
    // MFMAs [q0, q1) of step J, row-major over the wave's tiles
    auto mfmas = [&](auto j_c, int q0, int q1) __attribute__((always_inline)) {
        constexpr int J = decltype(j_c)::value;
        if constexpr (kF32) {
            // a lane's four consecutive k feed four MFMAs of two k each
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j) {
                        const uint4 a = fa[J & 1][i], b = fb[J & 1][j];
                        const uint32_t av = t == 0 ? a.x : t == 1 ? a.y : t == 2 ? a.z : a.w;
                        const uint32_t bv = t == 0 ? b.x : t == 1 ? b.y : t == 2 ? b.z : b.w;
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(av), __uint_as_float(bv), acc[i][j], 0, 0, 0);
                    }
        } else {
#pragma unroll
            for (int q = 0; q < WM * WN; ++q) {
                if (q < q0 || q >= q1) continue;
                acc[q / WN][q % WN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(fa[J & 1][q / WN]), as_bf16x8(fb[J & 1][q % WN]),
                                                                              acc[q / WN][q % WN], 0, 0, 0);
            }
        }
    };
    using J0 = std::integral_constant<int, 0>;
    using J1 = std::integral_constant<int, 1>;
    using J2 = std::integral_constant<int, 2>;
    using J3 = std::integral_constant<int, 3>;
    // Step J's MFMAs with the next step's fragments (of stage st) read and DMA
    // instructions [I0, I1) issued under them; int8 fragments of the next step
    // are converted under the second half.
    auto step = [&](auto j_c, auto next_c, const uint16_t* st, uint16_t* prev, int64_t s, auto i0_c, auto i1_c)
                    __attribute__((always_inline)) {
        constexpr int I0 = decltype(i0_c)::value, I1 = decltype(i1_c)::value;
        constexpr int kM = WM * WN * (kF32 ? 4 : 1), kR = WM + WN;
        frags(st, next_c);
        issue(prev, s + NS - 1, I0, I1);
        if constexpr (kI8) {
            constexpr int kH = kM / 2;
            mfmas(j_c, 0, kH);
            spread_reads_loads<kH, (kR + 1) / 2 * 2 <= kH ? kR : kH, I1 - I0>();
            __builtin_amdgcn_sched_barrier(0);
            convert(next_c);
            mfmas(j_c, kH, kM);
            spread_valu<kM - kH, 12 * WN>();
        } else {
            mfmas(j_c, 0, kM);
            spread_reads_loads<kM, kR, I1 - I0>();
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // One slab: each step's fragments are read under the step before it.  The
    // barrier that publishes slab s + 1 also retires every read of slab s, so
    // the next slab's DMA may overwrite that stage.  Every slab issues the same
    // number of loads (past the end it re-fetches the last one), so the wait is
    // always for all but the newest NS - 2 groups.
    auto slab = [&](int64_t s, const uint16_t* cur, uint16_t* prev, const uint16_t* next) __attribute__((always_inline)) {
        constexpr int kL1 = (kLoads + 2) / 3, kL2 = (2 * kLoads + 2) / 3;
        step(J0{}, J1{}, cur, prev, s, std::integral_constant<int, 0>{}, std::integral_constant<int, kL1>{});
        step(J1{}, J2{}, cur, prev, s, std::integral_constant<int, kL1>{}, std::integral_constant<int, kL2>{});
        step(J2{}, J3{}, cur, prev, s, std::integral_constant<int, kL2>{}, std::integral_constant<int, kLoads>{});
        wait_vmem_lds<(NS - 2) * kLoads>();
        barrier_no_fence();
        step(J3{}, J0{}, next, prev, s, std::integral_constant<int, kLoads>{}, std::integral_constant<int, kLoads>{});
    };
    issue(s0, slab0, 0, kLoads);
    issue(s1, slab0 + 1, 0, kLoads);
    if constexpr (NS > 3) issue(s2, slab0 + 2, 0, kLoads);
    if constexpr (NS > 4) issue(s3, slab0 + 3, 0, kLoads);
    if constexpr (NS > 5) issue(s4, slab0 + 4, 0, kLoads);
    wait_vmem_lds<(NS - 2) * kLoads>();
    barrier_no_fence();
    frags(s0, J0{});
    convert(J0{});
    int64_t s = slab0;
    if constexpr (NS == 3) {
        for (; s + 3 <= slab1; s += 3) {
            slab(s, s0, s2, s1);
            slab(s + 1, s1, s0, s2);
            slab(s + 2, s2, s1, s0);
        }
        if (s < slab1) slab(s, s0, s2, s1);
        if (s + 1 < slab1) slab(s + 1, s1, s0, s2);
    } else if constexpr (NS == 4) {
        for (; s + 4 <= slab1; s += 4) {
            slab(s, s0, s3, s1);
            slab(s + 1, s1, s0, s2);
            slab(s + 2, s2, s1, s3);
            slab(s + 3, s3, s2, s0);
        }
        if (s < slab1) slab(s, s0, s3, s1);
        if (s + 1 < slab1) slab(s + 1, s1, s0, s2);
        if (s + 2 < slab1) slab(s + 2, s2, s1, s3);
    } else if constexpr (NS == 5) {
        for (; s + 5 <= slab1; s += 5) {
            slab(s, s0, s4, s1);
            slab(s + 1, s1, s0, s2);
            slab(s + 2, s2, s1, s3);
            slab(s + 3, s3, s2, s4);
            slab(s + 4, s4, s3, s0);
        }
        if (s < slab1) slab(s, s0, s4, s1);
        if (s + 1 < slab1) slab(s + 1, s1, s0, s2);
        if (s + 2 < slab1) slab(s + 2, s2, s1, s3);
        if (s + 3 < slab1) slab(s + 3, s3, s2, s4);
    } else {
        for (; s + 6 <= slab1; s += 6) {
            slab(s, s0, s5, s1);
            slab(s + 1, s1, s0, s2);
            slab(s + 2, s2, s1, s3);
            slab(s + 3, s3, s2, s4);
            slab(s + 4, s4, s3, s5);
            slab(s + 5, s5, s4, s0);
        }
        if (s < slab1) slab(s, s0, s5, s1);
        if (s + 1 < slab1) slab(s + 1, s1, s0, s2);
        if (s + 2 < slab1) slab(s + 2, s2, s1, s3);
        if (s + 3 < slab1) slab(s + 3, s3, s2, s4);
        if (s + 4 < slab1) slab(s + 4, s4, s3, s5);
    }
    wait_vmem<0>();

    if constexpr (SPLIT) {
        // fp32 sums of this slab range, B row order
        const int64_t nb = (kGlu ? 2 : 1) * p.n;
        float* const out = part + static_cast<int64_t>(blockIdx.y) * p.m * nb;
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * (BM / kWavesM) + i * 32 + 8 * (r >> 2) + 4 * khalf + (r & 3);
                if (row >= re) continue;
#pragma unroll
                for (int j = 0; j < WN; ++j) {
                    const int block = wn * WN + j;
                    const int64_t col = kGlu ? ncol0 + (block >> 1) * 32 + l32 : ncol0 + block * 32 + l32;
                    if (col < p.n) out[row * nb + (kGlu && (block & 1) ? p.n + col : col)] = acc[i][j][r];
                }
            }
    } else {
        if constexpr (kGlu && WM == 4 && WN == 4) {
            if (p.c_dtype == SFG_BF16) {
                // 16 KB of staging per wave; every wave's reads of the last
                // slab are done before any wave reuses its stage
                constexpr int kPer16 = kStage / 8192;
                static_assert(NW <= 2 * kPer16, "staging fits two stage arrays");
                wait_lds();
                barrier_no_fence();
                glu_epilogue_staged<EPI>(p, acc, row0 + wm * (BM / kWavesM), ncol0 + wn * (BN / 4), re, scales, lane,
                                         (wave < kPer16 ? s0 : s1) + (wave % kPer16) * 8192);
                return;
            }
        }
        if constexpr (EPI == kEpiQkvRope && kI8) {
            // the QKV epilogue takes finished products
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const float sc = scales[min(ncol0 + wn * (BN / 2) + j * 32 + l32, p.n - 1)];
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] *= sc;
            }
        }
        // 8 KB of staging per wave for the QKV epilogue of 64 x 64 wave blocks
        constexpr int kPer = kStage / 4096;  // waves' regions per stage array
        static_assert(EPI != kEpiQkvRope || WM != 2 || WN != 2 || NW <= 3 * kPer, "staging fits three stage arrays");
        float* const qkv_stage = reinterpret_cast<float*>((wave < kPer ? s0 : wave < 2 * kPer ? s1 : s2) + (wave % kPer) * 4096);
        dma_tile_epilogue<BM, BN, NW, EPI, false, kWavesM, true>(p, acc, wm, wn, row0, ncol0, re, scales, qkv_stage);
    }
}

// ===========================================================================
// fp32 GEMM for products that fill few 64 x 64 tiles (short prompts, decode
// rows): a 32 x 32 output tile per workgroup (GLU: 32 gate and 32 up columns)
// whose four waves take every fourth 32-k slab, each through an LDS ring of its
// own filled by its own DMA.  No barrier until the four partial sums meet in
// LDS, in wave order: what bounds such a product is the length of one chain of
// dependent slabs, and this one is a quarter of a tile kernel's, with
// 4 x (NS - 1) slabs of 8 KB in flight.  128 rows, gate|up 2 x 688 x 256: 13.3 us
// on the VALU tiles, 7.8 here; down 256 x 688: 15.8, 8.1.
// ===========================================================================
template <int EPI>
__global__ __launch_bounds__(256) void gemm_f32_small_kernel(TiledArgs p, int tiles_m, int tiles_n) {
    constexpr bool kGlu = EpiTraits<EPI>::glu;
    constexpr int NT = kGlu ? 2 : 1;             // 32-column B blocks
    constexpr int kWaveStage = (32 + 32 * NT) * 32;  // floats
    constexpr int kLoads = 4 + 4 * NT;
    constexpr int NS = kGlu ? 3 : 4;
    __shared__ __attribute__((aligned(1024))) float s0[4 * kWaveStage];
    __shared__ __attribute__((aligned(1024))) float s1[4 * kWaveStage];
    __shared__ __attribute__((aligned(1024))) float s2[4 * kWaveStage];
    __shared__ __attribute__((aligned(1024))) float s3[NS > 3 ? 4 * kWaveStage : 8];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    int g;
    int64_t rb, re, tm, tn;
    if (!dma_tile_coords<32>(p, tiles_m, tiles_n, g, rb, re, tm, tn)) return;
    const int64_t row0 = rb + tm * 32;
    if (row0 >= re) return;
    const int64_t ncol0 = tn * 32;
    const int64_t all_slabs = (p.k + 31) / 32;
    const int tail = static_cast<int>(p.k % 32) / 4;  // 16-byte chunks of the last slab (0: all)
    const int64_t mine = all_slabs > wave ? (all_slabs - wave + 3) / 4 : 0;  // slabs wave, wave + 4, ...

    const uint32_t a_bytes = static_cast<uint32_t>(p.a_rows_limit * p.lda * 4);
    const uint32_t b_bytes = static_cast<uint32_t>(NT * p.n * p.ldb * 4);
    const buf_rsrc ra = make_rsrc(p.a, a_bytes);
    const buf_rsrc rbs = make_rsrc(reinterpret_cast<const float*>(p.b) + static_cast<int64_t>(g) * p.b_group_stride, b_bytes);
    // DMA instruction i: rows 8 i + lane / 8 of the A block (i < 4) or of B's
    uint32_t off[kLoads];
    const int slot = lane & 7;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int local = 8 * i + (lane >> 3);
        const int chunk = slot ^ ((local >> 1) & 7);
        if (i < 4) {
            const int64_t r = row0 + local;
            int64_t src = r < re ? r : row0;
            if (p.a_rows) src = p.a_rows[src];
            off[i] = (src < 0 || src >= p.a_rows_limit) ? a_bytes : static_cast<uint32_t>(src * p.lda * 4 + chunk * 16);
        } else {
            const int64_t col = ncol0 + ((local - 32) & 31);
            const int64_t brow = col < p.n ? (local >= 64 ? p.n + col : col) : 0;
            off[i] = static_cast<uint32_t>(brow * p.ldb * 4 + chunk * 16);
        }
    }
    auto issue = [&](float* st, int64_t idx) __attribute__((always_inline)) {
        const int64_t sl = min(wave + 4 * min(idx, mine - 1), all_slabs - 1);
        const int64_t at = max(sl, int64_t(0));
        const bool cut = tail != 0 && at == all_slabs - 1;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int local = 8 * i + (lane >> 3);
            const uint32_t past = i < 4 ? a_bytes : b_bytes;
            const uint32_t o = cut && (slot ^ ((local >> 1) & 7)) >= tail ? past : off[i];
            lds_dma16_buf(i < 4 ? ra : rbs, o, static_cast<uint32_t>(at * 128),
                          reinterpret_cast<uint16_t*>(st + wave * kWaveStage + i * 256));
        }
    };
    floatx16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
    const int sw = (l32 >> 1) & 7;
    // The newest NS - 2 slabs may still be in flight when slab idx is read.
    auto slab = [&](const float* cur, float* free, int64_t idx) __attribute__((always_inline)) {
        wait_vmem<(NS - 2) * kLoads>();
        asm volatile("" ::: "memory");
        const float* st = cur + wave * kWaveStage;
        float4 fa[4], fb[4][NT];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            fa[j] = *reinterpret_cast<const float4*>(st + l32 * 32 + ((2 * j + half) ^ sw) * 4);
#pragma unroll
            for (int n = 0; n < NT; ++n)
                fb[j][n] = *reinterpret_cast<const float4*>(st + (32 + 32 * n + l32) * 32 + ((2 * j + half) ^ sw) * 4);
        }
        issue(free, idx + NS - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[j].x, fb[j][n].x, acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[j].y, fb[j][n].y, acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[j].z, fb[j][n].z, acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[j].w, fb[j][n].w, acc[n], 0, 0, 0);
            }
        // this slab's reads are done before the next one's DMA may reuse it
        wait_lds();
    };
    issue(s0, 0);
    issue(s1, 1);
    if constexpr (NS > 3) issue(s2, 2);
    int64_t i = 0;
    if constexpr (NS == 4) {
        for (; i + 4 <= mine; i += 4) {
            slab(s0, s3, i);
            slab(s1, s0, i + 1);
            slab(s2, s1, i + 2);
            slab(s3, s2, i + 3);
        }
        if (i < mine) slab(s0, s3, i);
        if (i + 1 < mine) slab(s1, s0, i + 1);
        if (i + 2 < mine) slab(s2, s1, i + 2);
    } else {
        for (; i + 3 <= mine; i += 3) {
            slab(s0, s2, i);
            slab(s1, s0, i + 1);
            slab(s2, s1, i + 2);
        }
        if (i < mine) slab(s0, s2, i);
        if (i + 1 < mine) slab(s1, s0, i + 1);
    }
    wait_vmem<0>();
    // partial sums into this wave's own ring, then wave w adds up registers
    // 4 w .. 4 w + 3 (rows 8 w + 4 half + 0 .. 3) of all four
    float* const part = s0 + wave * kWaveStage;
    static_assert(kWaveStage >= NT * 16 * 64, "a wave's stage holds its partial");
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[(n * 16 + r) * 64 + lane] = acc[n][r];
    __syncthreads();
    const int64_t col = ncol0 + l32;
    const int64_t at = min(col, p.n - 1);
    float sum[NT][4], res[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t row = min(row0 + 8 * wave + 4 * half + e, re - 1);
        res[e] = EPI == SFG_EPI_RESIDUAL ? p.residual[row * p.ldr + at] : 0.f;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            sum[n][e] = s0[(n * 16 + 4 * wave + e) * 64 + lane];
#pragma unroll
            for (int w = 1; w < 4; ++w) sum[n][e] += s0[w * kWaveStage + (n * 16 + 4 * wave + e) * 64 + lane];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t row = row0 + 8 * wave + 4 * half + e;
        if (row >= re || col >= p.n) continue;
        float v;
        if constexpr (kGlu) v = glu_combine(EPI, sum[0][e], sum[1][e]);
        else v = sum[0][e] + res[e];
        store_out(p.c, p.c_dtype, row * p.ldc + col, v);
    }
}

namespace {

template <int BDT, int BM, int BN, int NW, int NS>
int launch_ring_tile(const TiledArgs& a, dim3 grid, int tm, int tn, int epi, float* part, hipStream_t s) {
    constexpr bool kPairs = (BN / 64) % 2 == 0;  // GLU tiles pair gate and up blocks
    const dim3 block(NW * 64);
    if constexpr (BDT != SFG_F32) if (part) {
        if (epi == SFG_EPI_SWIGLU || epi == SFG_EPI_GLU_SILU_UP) {
            if constexpr (kPairs) gemm_ring_kernel<BDT, BM, BN, NW, NS, SFG_EPI_SWIGLU, true><<<grid, block, 0, s>>>(a, tm, tn, part);
            else return SFG_ERR_UNSUPPORTED;
        } else {
            gemm_ring_kernel<BDT, BM, BN, NW, NS, SFG_EPI_NONE, true><<<grid, block, 0, s>>>(a, tm, tn, part);
        }
        return SFG_OK;
    }
    switch (epi) {
        case SFG_EPI_NONE: gemm_ring_kernel<BDT, BM, BN, NW, NS, SFG_EPI_NONE, false><<<grid, block, 0, s>>>(a, tm, tn, nullptr); break;
        case SFG_EPI_RESIDUAL: gemm_ring_kernel<BDT, BM, BN, NW, NS, SFG_EPI_RESIDUAL, false><<<grid, block, 0, s>>>(a, tm, tn, nullptr); break;
        case kEpiQkvRope:
            if constexpr (BDT != SFG_F32 && BM * BN < 256 * 256) {
                gemm_ring_kernel<BDT, BM, BN, NW, NS, kEpiQkvRope, false><<<grid, block, 0, s>>>(a, tm, tn, nullptr);
                break;
            } else {
                return SFG_ERR_UNSUPPORTED;
            }
        default:
            if constexpr (kPairs) {
                if (epi == SFG_EPI_SWIGLU) gemm_ring_kernel<BDT, BM, BN, NW, NS, SFG_EPI_SWIGLU, false><<<grid, block, 0, s>>>(a, tm, tn, nullptr);
                else gemm_ring_kernel<BDT, BM, BN, NW, NS, SFG_EPI_GLU_SILU_UP, false><<<grid, block, 0, s>>>(a, tm, tn, nullptr);
                break;
            } else {
                return SFG_ERR_UNSUPPORTED;
            }
    }
    return SFG_OK;
}

template <int BDT>
int launch_ring_b(const TiledArgs& a, const RingPlan& plan, dim3 grid, int tm, int tn, int epi, float* part,
                  hipStream_t s) {
    switch (plan.tile) {
        case kRingTileV:  // bf16: gemm_dma_kernel's
            if constexpr (BDT == SFG_I8) return part ? SFG_ERR_UNSUPPORTED : launch_ring_tile<BDT, 256, 256, 4, 3>(a, grid, tm, tn, epi, nullptr, s);
            else return SFG_ERR_UNSUPPORTED;
        case kRingTile256x128: return launch_ring_tile<BDT, 256, 128, 8, 3>(a, grid, tm, tn, epi, part, s);
        case kRingTile128x128:  // (eight waves 5 - 10% faster; int8 converts per wave, and four convert less)
            return launch_ring_tile<BDT, 128, 128, BDT == SFG_I8 ? 4 : 8, 4>(a, grid, tm, tn, epi, part, s);
        case kRingTile64x128: return launch_ring_tile<BDT, 64, 128, 4, 6>(a, grid, tm, tn, epi, part, s);
        case kRingTile128x64: return launch_ring_tile<BDT, 128, 64, 4, 6>(a, grid, tm, tn, epi, part, s);
        default: return launch_ring_tile<BDT, 64, 64, 4, 5>(a, grid, tm, tn, epi, part, s);
    }
}

}  // namespace

int launch_ring(const TiledArgs& a, const RingPlan& plan, int b_dtype, int epi, float* part, hipStream_t s) {
    const bool glu = epi == SFG_EPI_SWIGLU || epi == SFG_EPI_GLU_SILU_UP;
    const bool small = plan.tile == kRingTileSmall;
    const int64_t cols = glu && !small ? plan.bn / 2 : plan.bn;
    const int64_t tn = (a.n + cols - 1) / cols, tm = (a.m + plan.bm - 1) / plan.bm;
    const dim3 grid = a.offsets ? dim3(static_cast<unsigned>(tn), static_cast<unsigned>(tm + a.groups))
                                : dim3(static_cast<unsigned>(tm * tn), static_cast<unsigned>(plan.splits));
    const int itm = a.offsets ? 0 : static_cast<int>(tm);
    if (small) {
        const int itn = static_cast<int>(tn);
        switch (epi) {
            case SFG_EPI_NONE: gemm_f32_small_kernel<SFG_EPI_NONE><<<grid, 256, 0, s>>>(a, itm, itn); return SFG_OK;
            case SFG_EPI_RESIDUAL: gemm_f32_small_kernel<SFG_EPI_RESIDUAL><<<grid, 256, 0, s>>>(a, itm, itn); return SFG_OK;
            case SFG_EPI_SWIGLU: gemm_f32_small_kernel<SFG_EPI_SWIGLU><<<grid, 256, 0, s>>>(a, itm, itn); return SFG_OK;
            case SFG_EPI_GLU_SILU_UP: gemm_f32_small_kernel<SFG_EPI_GLU_SILU_UP><<<grid, 256, 0, s>>>(a, itm, itn); return SFG_OK;
            default: return SFG_ERR_UNSUPPORTED;
        }
    }
    if (b_dtype == SFG_F32) return launch_ring_b<SFG_F32>(a, plan, grid, itm, static_cast<int>(tn), epi, part, s);
    if (b_dtype == SFG_I8) return launch_ring_b<SFG_I8>(a, plan, grid, itm, static_cast<int>(tn), epi, part, s);
    return launch_ring_b<SFG_BF16>(a, plan, grid, itm, static_cast<int>(tn), epi, part, s);
}

}  // namespace sfg
