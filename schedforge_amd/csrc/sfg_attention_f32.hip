// sfg_attention_f32.hip -- fp32 flash prefill (attention_compiler.cpp:286-377)
// on the fp32 matrix instructions, head_dim 64 and 128.
#include "sfg_kernels.hpp"

namespace sfg {

// ===========================================================================
// fp32 flash prefill.  A workgroup of four waves owns 32 QW query rows of one
// (batch, head); wave (qw, kw) takes query block qw and every KW-th 32-key
// tile, so a long row's key chain is cut KW ways, and the KW partial softmaxes
// merge through LDS at the end.  Everything is fp32: v_mfma_f32_32x32x2_f32 for
// K Q^T and V^T P^T, online softmax with expf.
//
// Scores are formed transposed: lane l owns query l % 32 and, in accumulator
// register r, key 8 (r / 4) + 4 (l / 32) + r % 4 of the tile, which is exactly
// the P^T operand of the value product for the key pair of register r.  The
// k order of an MFMA is free, so the operands are read as vectors: a K read of
// 16 bytes feeds four MFMAs, and the value product's row i of block n stands for
// dim NB i + n (NB = D / 32), so one V read of NB floats feeds NB MFMAs.
// K rows keep 16-byte chunk c in slot c ^ (row & 15): the 16 rows of one LDS
// pass touch all 64 banks.
//
// What bounds it: the matrix pipe (64 clocks per MFMA, 256 FLOP/clk/CU) against
// the imbalance of the causal triangle; heaviest blocks first, two workgroups
// per CU at D = 64.  S 2048, 16 heads of 64 (8.6 GFLOP, 65 us at the fp32
// peak): 134 us, against 4037 us for one wave per query row on the VALU.
// ===========================================================================
namespace {

constexpr int kF32Keys = 32;  // keys per wave and step

template <int kD, int KW>
constexpr int kF32TileFloats = KW * kF32Keys * kD;  // K (or V) floats per stage

template <int kD, int QW, int KW, typename OutT>
__global__ __launch_bounds__(256) void attn_prefill_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    OutT* __restrict__ out, int q_heads, int kv_heads, int seq_q, int seq_kv, int heads_batch, int q_blocks,
    int causal, float scale) {
    static_assert(QW * KW == 4 && (kD == 64 || kD == 128), "four waves");
    constexpr int NB = kD / 32;
    constexpr int kTile = kF32TileFloats<kD, KW>;
    constexpr int kChunks = kD / 4;               // 16-byte chunks per row
    constexpr int kRowsPer = 64 / kChunks;        // rows per DMA instruction
    constexpr int kInstr = KW * kF32Keys / kRowsPer / 4;  // per wave, for K and again for V
    __shared__ __attribute__((aligned(1024))) float sk0[kTile];
    __shared__ __attribute__((aligned(1024))) float sk1[kTile];
    __shared__ __attribute__((aligned(1024))) float sv0[kTile];
    __shared__ __attribute__((aligned(1024))) float sv1[kTile];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qw = wave / KW, kw = wave % KW;
    const int l32 = lane & 31, half = lane >> 5;
    const int hb = blockIdx.x % heads_batch;
    const int qb = q_blocks - 1 - static_cast<int>(blockIdx.x) / heads_batch;  // heaviest first
    const int h = hb % q_heads, b = hb / q_heads;
    const int kvh = h * kv_heads / q_heads;
    const int q0 = qb * (32 * QW);
    const int offset = seq_kv - seq_q;
    const int block_last = min(q0 + 32 * QW, seq_q) - 1;
    const int keys = causal ? min(offset + block_last + 1, seq_kv) : seq_kv;  // keys the workgroup reads
    const int steps = (keys + KW * kF32Keys - 1) / (KW * kF32Keys);

    const int64_t kv_off = (static_cast<int64_t>(b) * kv_heads + kvh) * seq_kv * kD;
    const uint32_t kv_bytes = static_cast<uint32_t>(seq_kv) * kD * 4;  // rows past the end load zeros
    const buf_rsrc rk = make_rsrc(k + kv_off, kv_bytes), rv = make_rsrc(v + kv_off, kv_bytes);
    // DMA instruction i: rows kRowsPer (4 i + wave) + lane / kChunks of the stage
    uint32_t k_off[kInstr], v_off[kInstr];
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
        const int row = kRowsPer * (4 * i + wave) + lane / kChunks, slot = lane % kChunks;
        k_off[i] = static_cast<uint32_t>(row * kD + (slot ^ (row & 15)) * 4) * 4;
        v_off[i] = static_cast<uint32_t>(row * kD + slot * 4) * 4;
    }
    auto issue = [&](float* dk, float* dv, int step) __attribute__((always_inline)) {
        const uint32_t so = static_cast<uint32_t>(step) * (kTile * 4);
#pragma unroll
        for (int i = 0; i < kInstr; ++i) {
            lds_dma16_buf(rk, k_off[i], so, reinterpret_cast<uint16_t*>(dk + (4 * i + wave) * 256));
            lds_dma16_buf(rv, v_off[i], so, reinterpret_cast<uint16_t*>(dv + (4 * i + wave) * 256));
        }
    };

    const int qi = q0 + qw * 32 + l32;
    const int limit = causal ? offset + qi : seq_kv - 1;  // last key this lane's query sees
    const int first_limit = causal ? offset + q0 + qw * 32 : seq_kv - 1;
    const int wave_last = causal ? offset + min(q0 + qw * 32 + 31, seq_q - 1) : seq_kv - 1;
    const bool wave_live = q0 + qw * 32 < seq_q;
    float4 qf[kD / 8];
    {
        const float* qr = q + ((static_cast<int64_t>(b) * q_heads + h) * seq_q + min(qi, seq_q - 1)) * kD;
#pragma unroll
        for (int j = 0; j < kD / 8; ++j) qf[j] = *reinterpret_cast<const float4*>(qr + (2 * j + half) * 4);
    }
    floatx16 o[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[n][r] = 0.f;
    float m = -INFINITY, l = 0.f;

    auto tile = [&](const float* tk, const float* tv, int step) __attribute__((always_inline)) {
        const int kt = (step * KW + kw) * kF32Keys;  // first key of this wave's tile
        if (!wave_live || kt > wave_last || kt >= seq_kv) return;
        tk += kw * kF32Keys * kD;
        tv += kw * kF32Keys * kD;
        floatx16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int j = 0; j < kD / 8; ++j) {
            const float4 kf = *reinterpret_cast<const float4*>(tk + l32 * kD + (((2 * j + half) ^ (l32 & 15)) * 4));
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.x, qf[j].x, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.y, qf[j].y, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.z, qf[j].z, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.w, qf[j].w, s, 0, 0, 0);
        }
        const bool masked = kt + kF32Keys - 1 > min(first_limit, seq_kv - 1);  // wave-uniform
        float p[16];
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            p[r] = s[r] * scale;
            if (masked) {
                const int key = kt + 8 * (r >> 2) + 4 * half + (r & 3);
                if (key > limit || key >= seq_kv) p[r] = -INFINITY;
            }
            mx = fmaxf(mx, p[r]);
        }
        const float m_new = fmaxf(m, xor32_max(mx));
        const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            p[r] = p[r] == -INFINITY ? 0.f : expf(p[r] - m_new);
            sum += p[r];
        }
        l = l * alpha + xor32_sum(sum);
        if (__any(m_new != m)) {
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[n][r] *= alpha;
        }
        m = m_new;
        auto vrow = [&](int key, float (&vf)[NB]) __attribute__((always_inline)) {
            const float* src = tv + key * kD + NB * l32;
            if constexpr (NB == 4) {
                const float4 t = *reinterpret_cast<const float4*>(src);
                vf[0] = t.x; vf[1] = t.y; vf[2] = t.z; vf[3] = t.w;
            } else {
                const float2 t = *reinterpret_cast<const float2*>(src);
                vf[0] = t.x; vf[1] = t.y;
            }
        };
        if (masked) {
            // 0 * inf: a key hidden from some of the queries may hold
            // non-finite values, which must not reach their sums
            float bad = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float vf[NB];
                vrow(8 * (r >> 2) + 4 * half + (r & 3), vf);
#pragma unroll
                for (int n = 0; n < NB; ++n) bad = fmaf(vf[n], 0.f, bad);
            }
            if (__any(bad != 0.f)) {  // NaN
#pragma unroll 1
                for (int r = 0; r < 16; ++r)
#pragma unroll 1
                    for (int hh = 0; hh < 2; ++hh) {
                        const int key = 8 * (r >> 2) + 4 * hh + (r & 3);
                        float mine = 0.f;
#pragma unroll
                        for (int e = 0; e < 16; ++e) mine = e == r ? p[e] : mine;
                        const float pv = __shfl(mine, l32 + 32 * hh, 64);
                        if (kt + key > limit || kt + key >= seq_kv) continue;
#pragma unroll
                        for (int n = 0; n < NB; ++n)
#pragma unroll
                            for (int e = 0; e < 16; ++e)
                                o[n][e] = fmaf(pv, tv[key * kD + NB * (8 * (e >> 2) + 4 * half + (e & 3)) + n], o[n][e]);
                    }
                return;
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float vf[NB];
            vrow(8 * (r >> 2) + 4 * half + (r & 3), vf);
#pragma unroll
            for (int n = 0; n < NB; ++n) o[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[n], p[r], o[n], 0, 0, 0);
        }
    };

    // Two stages: at each barrier every wave's loads of this step have landed
    // and every wave is done with the other stage, which the next loads fill.
    issue(sk0, sv0, 0);
    for (int step = 0; step < steps; step += 2) {
        wait_vmem<0>();
        wait_lds();
        barrier_no_fence();
        if (step + 1 < steps) issue(sk1, sv1, step + 1);
        tile(sk0, sv0, step);
        if (step + 1 >= steps) break;
        wait_vmem<0>();
        wait_lds();
        barrier_no_fence();
        if (step + 2 < steps) issue(sk0, sv0, step + 2);
        tile(sk1, sv1, step + 1);
    }

    if constexpr (KW > 1) {
        // merge the key splits of each query block in order
        wait_lds();
        barrier_no_fence();
        constexpr int kPart = NB * 16 * 64;  // floats of one wave's accumulators
        static_assert(kTile >= kPart + 128, "a stage array holds one wave's partial");
        
        float* dst = wave == 0 ? sk0 : wave == 1 ? sv0 : wave == 2 ? sk1 : sv1;
        if (kw > 0) {
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) dst[(n * 16 + r) * 64 + lane] = o[n][r];
            dst[kPart + lane] = m;
            dst[kPart + 64 + lane] = l;
        }
        wait_lds();
        barrier_no_fence();
        if (kw > 0) return;
#pragma unroll
        for (int w = 1; w < KW; ++w) {
            const int from = wave + w;
            const float* src = from == 1 ? sv0 : from == 2 ? sk1 : sv1;
            const float mw = src[kPart + lane], lw = src[kPart + 64 + lane];
            const float m_new = fmaxf(m, mw);
            const float a0 = m == -INFINITY ? 0.f : expf(m - m_new);
            const float a1 = mw == -INFINITY ? 0.f : expf(mw - m_new);
            l = l * a0 + lw * a1;
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    // a split that saw no key holds zeros, which stay out of the sum
                    const float other = mw == -INFINITY ? 0.f : src[(n * 16 + r) * 64 + lane] * a1;
                    o[n][r] = o[n][r] * a0 + other;
                }
            m = m_new;
        }
    }
    if (qi >= seq_q) return;
    OutT* dst = out + (static_cast<int64_t>(b) * seq_q + qi) * (static_cast<int64_t>(q_heads) * kD) + h * kD;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        // dims NB (8 g + 4 half) .. + 4 NB of this query
        float t[4 * NB];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int n = 0; n < NB; ++n) t[e * NB + n] = o[n][4 * g + e] / l;
        OutT* d = dst + NB * (8 * g + 4 * half);
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            if constexpr (sizeof(OutT) == 4)
                *reinterpret_cast<float4*>(d + 4 * e) = make_float4(t[4 * e], t[4 * e + 1], t[4 * e + 2], t[4 * e + 3]);
            else
                *reinterpret_cast<uint2*>(d + 4 * e) = make_uint2(pack_bf16x2(t[4 * e], t[4 * e + 1]), pack_bf16x2(t[4 * e + 2], t[4 * e + 3]));
        }
    }
}

template <int kD, int QW, int KW>
void launch_f32_flash(const float* q, const float* k, const float* v, void* out, int out_dtype, int64_t batch,
                      int64_t q_heads, int64_t kv_heads, int64_t seq_q, int64_t seq_kv, int causal, float scale,
                      hipStream_t stream) {
    const int blocks = static_cast<int>((seq_q + 32 * QW - 1) / (32 * QW));
    const int hb = static_cast<int>(q_heads * batch);
    const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(blocks) * hb));
    if (out_dtype == SFG_F32)
        attn_prefill_f32_kernel<kD, QW, KW, float><<<grid, 256, 0, stream>>>(
            q, k, v, static_cast<float*>(out), static_cast<int>(q_heads), static_cast<int>(kv_heads),
            static_cast<int>(seq_q), static_cast<int>(seq_kv), hb, blocks, causal, scale);
    else
        attn_prefill_f32_kernel<kD, QW, KW, uint16_t><<<grid, 256, 0, stream>>>(
            q, k, v, static_cast<uint16_t*>(out), static_cast<int>(q_heads), static_cast<int>(kv_heads),
            static_cast<int>(seq_q), static_cast<int>(seq_kv), hb, blocks, causal, scale);
}

}  // namespace

// head_dim 64 / 128, 16-byte aligned tensors, K and V of one head within 32-bit
// byte offsets, a grid within 32 bits of work items.
bool attn_prefill_f32_mfma_supported(const float* q, const float* k, const float* v, const void* out,
                                     int64_t batch, int64_t q_heads, int64_t seq_q, int64_t seq_kv, int64_t head_dim) {
    const uintptr_t low = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                          reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(out);
    return (head_dim == 64 || head_dim == 128) && (low & 15) == 0 && seq_kv <= (int64_t(1) << 22) &&
           seq_q <= (int64_t(1) << 22) && batch * q_heads * ((seq_q + 31) / 32) < (int64_t(1) << 24);
}

void launch_attn_prefill_f32_mfma(const float* q, const float* k, const float* v, void* out, int out_dtype,
                                  int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q, int64_t seq_kv,
                                  int64_t head_dim, int causal, float scale, hipStream_t stream) {
    if (head_dim == 128) {
        launch_f32_flash<128, 2, 2>(q, k, v, out, out_dtype, batch, q_heads, kv_heads, seq_q, seq_kv, causal, scale, stream);
        return;
    }
    // Four key splits of one 32-row block while 64-row blocks leave CUs idle.
    if (batch * q_heads * ((seq_q + 63) / 64) < 256)
        launch_f32_flash<64, 1, 4>(q, k, v, out, out_dtype, batch, q_heads, kv_heads, seq_q, seq_kv, causal, scale, stream);
    else
        launch_f32_flash<64, 2, 2>(q, k, v, out, out_dtype, batch, q_heads, kv_heads, seq_q, seq_kv, causal, scale, stream);
}

}  // namespace sfg
