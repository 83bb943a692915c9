// Many-token prefill on the matrix cores, gfx950 (q4, q8 and f16 weights).
//
// Replaces the reference's multi-token path (Shaders.swift:676-1216: k_rmsnorm_rows_h,
// llm_gemm_tile, k_g3_*, k_qk_norm_rope, k_prefill_attn) for prompts longer than one GEMV pass;
// math per tools/reference/qwen3vl_ref.py:243-292 (fp32 activations, fp16 KV cache).
//
// Projections.  q4: y[t][r] = sum_g (s_rg sum_{k in g} q_rk x_tk + b_rg sum_{k in g} x_tk) over
// 64-groups; q8: y[t][r] = sum_g s_rg sum_{k in g} q_rk x_tk over 32-groups; f16: y = W x.  A prep
// kernel scales every activation row by a power of two that puts its largest |x| in
// [2^14, 2^15) and splits it into fp16 hi + lo parts (x'' = hi + lo to ~22 bits; the scaling
// keeps every part that matters far above the fp16 subnormal range).  The GEMM runs
// v_mfma_f32_16x16x32_f16 on (hi, lo) x the weights as fp16 B operands: the q4 and q8 integer
// codes are exact in fp16, so each group's sum C_g = sum_k q_k x''_k comes out of one
// accumulator chain; the group epilogue is acc += s C_g (q4 and q8: the q4 bias term
// sum_g b_g X_g, X_g = sum_k x''_k, runs on the matrix cores once per tile before the loop),
// f16 weights accumulate directly, and the row scale 2^(E_t - 14) is applied once at the end.
// With fp16 operands alone (ICUA_FLAG_PREFILL_FP16, the reference engine's precision) there is
// no lo part, and the B operands are the weights dequantised to fp16 (q4 fp16(s q + b), q8
// fp16(s q)), so the products accumulate straight into the outputs with no group epilogue.
//
// Attention.  Causal GQA flash attention on v_mfma_f32_16x16x32_f16: scores are computed
// transposed (S^T = K Q^T) so that the probabilities come out of the accumulator already in
// the B-operand layout of the P.V product (O^T = V^T P^T); V is transposed through LDS.  The
// fp32 queries and probabilities are split into fp16 hi + lo parts (two products each), which
// keeps them at ~22 bits against the fp16 cache (one part with fp16 operands alone).  Each wave
// holds 32 queries, so every K and V operand it reads from LDS feeds two products.
#include <algorithm>

#include "icua_device.h"
#include "icua_kernels.h"

namespace icua {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float swiglu(float y, float up) {
    return y * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-y * 1.4426950408889634f)) * up;
}

// ------------------------------------------------------------------------------------------
// Activation operands.  XA: [Mpad / 16][K / 32][parts (hi, lo)][64 lanes][8 halves], lane l
// holding token 16 tb + l % 16.  q8 / f16: K = 32 ks + 8 (l / 16) + 0..7 of k-step ks, in order.
// q4 takes the K order in which its nibbles unpack without cross-lane moves: k-step 2 g + h of
// 64-group g holds K = 64 g + 16 (l / 16) + 8 h + {0, 2, 4, 6, 1, 3, 5, 7}.  XB (q4, hi + lo):
// the 64-group sums of hi + lo times 2^-8 (into fp16 range), as fp16 hi and lo A operands over
// groups, [Mpad / 16][ceil(K / 2048)][2][64 lanes][8].  TS: [Mpad] row scales 2^(E_t - 14).  One
// workgroup per token row (rows >= M are zero).  A row writes 16-byte pieces of lines that the 16
// rows of its token block share, so rows are dealt to the 8 XCDs (workgroup i runs on XCD i % 8)
// in contiguous ranges: the lines are completed in one L2 rather than written back in parts.
//
// The source row is what the previous kernel left, so that no pass over memory only moves data:
// a residual row, to which the O / down GEMM's K-split partial sums (and DeepStack rows) are
// added and written back; attention rows, or their key-split partials, merged; SwiGLU rows, or
// the gate|up GEMM's K-split partials.
//
// What bounds it at a few hundred rows is the chain of memory round trips, so partials are requested
// several at a time, whatever their count: through a buffer resource that ends with the last one
// (past it: zeros, no traffic).
struct Parts {
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ Parts(const float* p, size_t floats)
        : rs(__builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)(floats * 4), 0x00020000)) {}
    __device__ __forceinline__ float4 load4(int at) const {  // floats at .. at + 3
        return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, at * 4, 0, 0));
    }
    __device__ __forceinline__ float load(int at) const { return as_f32(__builtin_amdgcn_raw_buffer_load_b32(rs, at * 4, 0, 0)); }
};
__device__ __forceinline__ void add8(float (&d)[8], const float4& a0, const float4& a1) {
    d[0] += a0.x; d[1] += a0.y; d[2] += a0.z; d[3] += a0.w;
    d[4] += a1.x; d[5] += a1.y; d[6] += a1.z; d[7] += a1.w;
}
// PARTS: the source has partials.
template <int K, int SRC, int HL, bool Q4, bool PARTS>
__global__ __launch_bounds__(256) void pf_prep_kernel(PfPrepArgs a) {
    constexpr int NU = K / 8 / 256;  // units of 8 activations per thread
    constexpr int NKS = K / 32, NXB = (K / 64 + 31) / 32;
    const int t = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);  // gridDim.x % 8 == 0
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    __shared__ float red[8];
    float v[NU][8];
#pragma unroll
    for (int j = 0; j < NU; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[j][i] = 0.f;
    float4 w0, w1;  // requested with the row, not after its sum of squares
    if constexpr (SRC == PF_SRC_RESID) {
        static_assert(SRC != PF_SRC_RESID || NU == 1, "one unit per thread");
        w0 = ((const float4*)(a.norm_w + tid * 8))[0];
        w1 = ((const float4*)(a.norm_w + tid * 8))[1];
    }
    if (t < a.M) {
        if constexpr (SRC == PF_SRC_ATTN && PARTS) {
            // Merge of the attention's key splits (at most 32): head tid / 16, dims 8 (tid % 16) .. + 7.
            // The head's 16 lanes load a pair of splits' (max, denominator) each and share the weights.
            const int head = tid >> 4, l16 = lane & 15;
            const Parts op(a.part, (size_t)a.nsplit * a.M * H);
            const float2* ml = (const float2*)a.part_ml + (size_t)t * NH + head;
            float2 x[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                x[i] = l16 + 16 * i < a.nsplit ? ml[(size_t)(l16 + 16 * i) * a.M * NH] : make_float2(-__builtin_inff(), 0.f);
            float m = fmaxf(x[0].x, x[1].x);  // finite over the splits: each row sees its own key
            m = fmaxf(m, dpp<DPP_XOR1>(m));
            m = fmaxf(m, dpp<DPP_XOR2>(m));
            m = fmaxf(m, dpp<DPP_HALF_MIRROR>(m));
            m = fmaxf(m, dpp<DPP_MIRROR>(m));
            const float f0 = __builtin_amdgcn_exp2f(x[0].x - m), f1 = __builtin_amdgcn_exp2f(x[1].x - m);
            const float l = sum16(fmaf(x[0].y, f0, x[1].y * f1));
            for (int s0 = 0; s0 < a.nsplit; s0 += 8) {
                float4 o[8][2];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int at = ((s0 + i) * a.M + t) * H + 8 * tid;
                    o[i][0] = op.load4(at);
                    o[i][1] = op.load4(at + 4);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float f = __shfl(s0 & 16 ? f1 : f0, (lane & 48) + (s0 & 15) + i);
                    v[0][0] = fmaf(o[i][0].x, f, v[0][0]); v[0][1] = fmaf(o[i][0].y, f, v[0][1]);
                    v[0][2] = fmaf(o[i][0].z, f, v[0][2]); v[0][3] = fmaf(o[i][0].w, f, v[0][3]);
                    v[0][4] = fmaf(o[i][1].x, f, v[0][4]); v[0][5] = fmaf(o[i][1].y, f, v[0][5]);
                    v[0][6] = fmaf(o[i][1].z, f, v[0][6]); v[0][7] = fmaf(o[i][1].w, f, v[0][7]);
                }
            }
            const float inv = 1.0f / l;
#pragma unroll
            for (int i = 0; i < 8; ++i) v[0][i] *= inv;
        } else if constexpr (SRC == PF_SRC_SWIGLU && PARTS) {
            // Units 8 u .. + 7 are row block u of the gate|up GEMM: 8 gate rows, then 8 up rows.
            const Parts gu(a.part, (size_t)a.nsplit * a.M * GU);
            float up[NU][8];
#pragma unroll
            for (int j = 0; j < NU; ++j)
#pragma unroll
                for (int i = 0; i < 8; ++i) up[j][i] = 0.f;
            for (int s0 = 0; s0 < a.nsplit; s0 += 2) {
                float4 o[2][NU][4];
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NU; ++j)
#pragma unroll
                        for (int c = 0; c < 4; ++c) o[i][j][c] = gu.load4(((s0 + i) * a.M + t) * GU + (tid + 256 * j) * 16 + 4 * c);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NU; ++j) {
                        add8(v[j], o[i][j][0], o[i][j][1]);
                        add8(up[j], o[i][j][2], o[i][j][3]);
                    }
            }
#pragma unroll
            for (int j = 0; j < NU; ++j)
#pragma unroll
                for (int i = 0; i < 8; ++i) v[j][i] = swiglu(v[j][i], up[j][i]);
        } else {
            float4 x[NU][2];
#pragma unroll
            for (int j = 0; j < NU; ++j) {
                const float4* p = (const float4*)(a.src + (size_t)t * K + (tid + 256 * j) * 8);
                x[j][0] = p[0];
                x[j][1] = p[1];
            }
            if constexpr (SRC == PF_SRC_RESID && PARTS) {
                const Parts rp(a.part, (size_t)a.nsplit * a.M * H);
                // DeepStack residual of a visual row (Shaders.swift:696-707)
                const int vrow = a.row0 + t - a.vis_offset;
                const bool vis = a.ds && a.vis_offset >= 0 && vrow >= 0 && vrow < a.n_vis;
                float4 d0, d1;
                if (vis) {
                    d0 = ((const float4*)(a.ds + (size_t)vrow * H + tid * 8))[0];
                    d1 = ((const float4*)(a.ds + (size_t)vrow * H + tid * 8))[1];
                }
                for (int s0 = 0; s0 < a.nsplit; s0 += 8) {
                    float4 o[8][2];
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int at = ((s0 + i) * a.M + t) * H + tid * 8;
                        o[i][0] = rp.load4(at);
                        o[i][1] = rp.load4(at + 4);
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i) add8(v[0], o[i][0], o[i][1]);
                }
                add8(v[0], x[0][0], x[0][1]);
                if (vis) add8(v[0], d0, d1);
                float4* xo = (float4*)(a.dst + (size_t)t * K + tid * 8);
                xo[0] = make_float4(v[0][0], v[0][1], v[0][2], v[0][3]);
                xo[1] = make_float4(v[0][4], v[0][5], v[0][6], v[0][7]);
            } else {
#pragma unroll
                for (int j = 0; j < NU; ++j) add8(v[j], x[j][0], x[j][1]);
            }
        }
    }
    if constexpr (SRC == PF_SRC_RESID) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < NU; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += v[j][i] * v[j][i];
        ss = wave_sum(ss);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        const float tot = (red[0] + red[1]) + (red[2] + red[3]);
        const float scale = 1.0f / sqrtf(tot / (float)K + EPS);
        const float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) v[0][i] = v[0][i] * scale * w[i];
    }
    // Row exponent: largest |x| in [2^E, 2^(E+1)).
    float amax = 0.f;
#pragma unroll
    for (int j = 0; j < NU; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[j][i]));
    amax = wave_max(amax);
    if (lane == 0) red[4 + wave] = amax;
    __syncthreads();
    const float rmax = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
    const int E = (rmax > 0.f) ? ((int)((as_u32(rmax) >> 23) & 0xFF) - 127) : 0;
    const int sh = 14 - E;
    const int tb = t >> 4, tr = t & 15;
#pragma unroll
    for (int j = 0; j < NU; ++j) {
        const int k0 = (tid + 256 * j) * 8;
        uint32_t hw[4], lw[4];
        float gs = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // Word i holds K 2 i, 2 i + 1, or in q4 order (0, 2) (4, 6) (1, 3) (5, 7).
            const int i0 = Q4 ? 4 * (i & 1) + (i >> 1) : 2 * i, i1 = Q4 ? i0 + 2 : i0 + 1;
            const float x0 = ldexpf(v[j][i0], sh), x1 = ldexpf(v[j][i1], sh);
            const f16 h0 = (f16)x0, h1 = (f16)x1;
            const f16 l0 = (f16)(x0 - (float)h0), l1 = (f16)(x1 - (float)h1);
            gs += ((float)h0 + (float)l0) + ((float)h1 + (float)l1);
            hw[i] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
            lw[i] = (uint32_t)__builtin_bit_cast(uint16_t, l0) | ((uint32_t)__builtin_bit_cast(uint16_t, l1) << 16);
        }
        const int ks = Q4 ? 2 * (k0 / 64) + (k0 % 16) / 8 : k0 / 32, qq = Q4 ? (k0 % 64) / 16 : (k0 % 32) / 8;
        uint16_t* base = a.xa + ((size_t)(tb * NKS + ks) * HL) * 512 + (tr + 16 * qq) * 8;
        *(uint4*)base = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        if constexpr (HL == 2) *(uint4*)(base + 512) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        if constexpr (Q4 && HL == 2) {
            // Group sums over the 8 adjacent lanes holding the group's 64 values.
            gs += dpp<DPP_XOR1>(gs);
            gs += dpp<DPP_XOR2>(gs);
            gs += dpp<DPP_HALF_MIRROR>(gs);
            if (k0 % 64 == 0) {
                const int g = k0 / 64;
                const float x = gs * 0.00390625f;  // 2^-8: a group sum of 64 values below 2^15
                const f16 hx = (f16)x;
                uint16_t* xb = a.xb + ((size_t)(tb * NXB + g / 32) * 2 * 64 + tr + 16 * ((g % 32) / 8)) * 8 + g % 8;
                xb[0] = __builtin_bit_cast(uint16_t, hx);
                xb[512] = f2h(x - (float)hx);
            }
        }
    }
    if (tid == 0) a.ts[t] = ldexpf(1.0f, -sh);
}

// The residual row t0 after a GEMM that left K-split partials: dst = src + partials (+ DeepStack).
__global__ __launch_bounds__(256) void pf_last_row_kernel(PfPrepArgs a, int t) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    float y = 0.f;
    for (int s = 0; s < a.nsplit; ++s) y += a.part[((size_t)s * a.M + t) * H + i];
    float v = a.src[(size_t)t * H + i] + y;
    const int vrow = a.row0 + t - a.vis_offset;
    if (a.ds && a.vis_offset >= 0 && vrow >= 0 && vrow < a.n_vis) v += a.ds[(size_t)vrow * H + i];
    a.dst[i] = v;
}

// ------------------------------------------------------------------------------------------
// Weight codes as fp16 B operands, exactly.

// Eight q4 codes of a dword (byte j: K j low, K 4 + j high): a nibble or'ed into 0x6400 is the
// fp16 value 1024 + q (or 1024 + 16 q in place of the high nibble), and one packed operation
// leaves q.  Halves in K order 0, 2, 4, 6, 1, 3, 5, 7.
__device__ __forceinline__ uint32_t and_or(uint32_t d, uint32_t mask, uint32_t bits) {
    uint32_t r;  // one instruction (from two literals the compiler makes two)
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(d), "s"(mask), "v"(bits));
    return r;
}
__device__ __forceinline__ void unpack_q4(uint32_t d, f16x2 (&o)[4]) {
    const f16x2 k1024 = {(f16)1024.f, (f16)1024.f}, k16 = {(f16)0.0625f, (f16)0.0625f}, k64 = {(f16)-64.f, (f16)-64.f};
    const uint32_t e = d >> 8;
    o[0] = as_h2(and_or(d, 0x000F000Fu, 0x64006400u)) - k1024;
    o[1] = __builtin_elementwise_fma(as_h2(and_or(d, 0x00F000F0u, 0x64006400u)), k16, k64);
    o[2] = as_h2(and_or(e, 0x000F000Fu, 0x64006400u)) - k1024;
    o[3] = __builtin_elementwise_fma(as_h2(and_or(e, 0x00F000F0u, 0x64006400u)), k16, k64);
}
// Eight q8 codes of two dwords in order: a signed byte with its top bit flipped, put under the
// exponent of 1024 by a byte permute, is the fp16 value 1152 + b.
__device__ __forceinline__ void unpack_q8(uint32_t d0, uint32_t d1, f16x2 (&o)[4]) {
    const f16x2 k1152 = {(f16)1152.f, (f16)1152.f};
    const uint32_t u0 = d0 ^ 0x80808080u, u1 = d1 ^ 0x80808080u;
    o[0] = as_h2(__builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u)) - k1152;
    o[1] = as_h2(__builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u)) - k1152;
    o[2] = as_h2(__builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u)) - k1152;
    o[3] = as_h2(__builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)) - k1152;
}
// The same halves by way of zero-extended bytes (b ^ 0x80 or'ed into 0x6400).  Two instructions more a
// dword, but in the hi + lo tiles of pf_gemm_kernel, which unpack between products, the compiler then
// needs up to 40 registers fewer: 3000 rows, 4 layers and the head 4.14 ms, with unpack_q8 4.33.
__device__ __forceinline__ void unpack_q8_bytes(uint32_t d0, uint32_t d1, f16x2 (&o)[4]) {
    const f16x2 k1152 = {(f16)1152.f, (f16)1152.f};
    const uint32_t d[2] = {d0, d1};
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const uint32_t s0 = __builtin_amdgcn_perm(d[w], d[w], 0x0C010C00u);  // b0, b1
        const uint32_t s1 = __builtin_amdgcn_perm(d[w], d[w], 0x0C030C02u);  // b2, b3
        o[2 * w] = as_h2((s0 ^ 0x00800080u) | 0x64006400u) - k1152;
        o[2 * w + 1] = as_h2((s1 ^ 0x00800080u) | 0x64006400u) - k1152;
    }
}
__device__ __forceinline__ uint4 pack4(const f16x2 (&o)[4]) {
    return make_uint4(h2_bits(o[0]), h2_bits(o[1]), h2_bits(o[2]), h2_bits(o[3]));
}

// One output of a GEMM tile: token t of weight row `row` (y with the row scale applied).
template <int EPI>
__device__ __forceinline__ void pf_store(const PfGemmArgs& a, int t, int row, float y) {
    if constexpr (EPI == EPI_STORE) {
        if (t < a.M) a.y[(size_t)t * a.N + row] = y;
    } else if constexpr (EPI == EPI_RESID) {
        if (t < a.M) {
            float* xo = a.y + (size_t)t * a.N + row;
            float v = *xo + y;
            if (a.ds) {  // DeepStack residual of a visual row (Shaders.swift:696-707)
                const int vrow = a.row0 + t - a.vis_offset;
                if (a.vis_offset >= 0 && vrow >= 0 && vrow < a.n_vis) v = v + a.ds[(size_t)vrow * H + row];
            }
            *xo = v;
        }
    } else {  // EPI_SWIGLU: a row block holds 8 gate units, then their up rows (lanes r16, r16 ^ 8)
        const float up = dpp<0x128>(y);  // lane r16 ^ 8 of the row of 16 (a rotation by 8)
        if (t < a.M && (row & 15) < 8) a.h[(size_t)t * FF + (row >> 4) * 8 + (row & 15)] = swiglu(y, up);
    }
}

// ------------------------------------------------------------------------------------------
// GEMM: a workgroup of 8 waves computes 64 TB tokens x 16 RB weight rows (TB = 1 or 2 token
// blocks per wave, RB = 8 or 16 row blocks); wave w owns token blocks 4 TB tm + TB (w % 4) ..
// against row blocks RB / 2 (w / 4) onwards (RB / 2 row blocks), two waves per SIMD, and takes
// its row blocks in halves of four per group.  Each 128-K step, the weight chunks of the RB row
// blocks (q4 one 1 KiB chunk, q8 two, f16 four) become fp16 B operands in LDS once
// (double-buffered, 64 or 128 KiB) and are shared by the waves; the waves' activation operands
// stream from global memory straight into registers two 64-K groups ahead.  The launch takes
// the largest tile (most products per operand byte) whose count still fills the CUs evenly.
template <int FMT, int K, int EPI, int PG_RB, int TB, int HL>
__global__ __launch_bounds__(512) void pf_gemm_kernel(PfGemmArgs a) {
    static_assert((PG_RB == 8 || PG_RB == 16) && (TB == 1 || TB == 2), "tile shape");
    static_assert(FMT == FMT_Q8 || HL == 2, "q4 and f16 with fp16 operands alone take the K-split GEMM");
    constexpr int NHF = PG_RB / 8;         // halves of four row blocks per wave
    constexpr int TR = 16 * PG_RB;         // rows of a tile
    constexpr int NG = K / 64, NKS = K / 32, NC = K / 128;
    constexpr int CPS = FMT == FMT_Q4 ? 1 : FMT == FMT_Q8 ? 2 : 4;  // 1 KiB chunks per 128-K step
    constexpr int NCH = NC * CPS;                                      // chunks per row block
    // DQ: the B operands are the dequantised q8 weights s q in fp16 (the reference engine's prefill
    // precision, taken with fp16 operands alone) or the f16 weights themselves, so the products
    // accumulate straight into the outputs; otherwise codes are exact fp16 integers and each group's
    // sums take their scale in an epilogue.
    constexpr bool DQ = HL == 1 || FMT == FMT_F16;
    const int TN = a.N / (16 * PG_RB), TM = a.Mpad / (64 * TB), T = TM * TN;
    const int per = (T + 7) / 8;
    const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= T) return;
    const int tm = tile / TN, tn = tile % TN;

    __shared__ uint4 Bs[2][PG_RB][4][64];  // fp16 codes: [buffer][row block][k-step][lane]
    // Per-step words: [buffer][i] fp16 (scale, bias) of group 2 c + i / TR, row i % TR.
    __shared__ __attribute__((aligned(16))) uint32_t Vs[2][512];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, r16 = lane & 15;
    const int tb0 = tm * 4 * TB + TB * (wave & 3), rb0 = (PG_RB / 2) * (wave >> 2);
    const uint16_t* xa = a.xa + (size_t)tb0 * NKS * 512 * HL + lane * 8;   // token block tb0 (+ NKS * 512 HL for tb0 + 1)
    // Staging: thread t unpacks nibble lane t % 64 of row block t / 64 (and t / 64 + 8).
    const int srb = tid >> 6;
    const uint8_t* wsrc = a.w + (size_t)(tn * PG_RB + srb) * NCH * 1024 + lane * 16;
    constexpr size_t WSRC2 = (size_t)8 * NCH * 1024;  // row block srb + 8
    // Thread t < 2 TR loads one scale word per step (stride 2 words): row t % TR of the tile, q4
    // the (scale, bias) half2 of 64-group 2 c + t / TR; q8 the scales of 32-groups
    // 4 c + 2 (t / TR), + 1 (the same word offsets: a q8 row holds K / 64 words of scale pairs).
    const uint32_t* vsrc = (const uint32_t*)a.sb + (size_t)(tn * TR + (tid % TR)) * NG + (tid / TR);
    constexpr int vstride = 2;
    const bool vload = !DQ && (2 * TR >= 512 || tid < 2 * TR);
    // DQ q8: the unpacking thread's own scale words, row (tn RB + srb + 8 hb) 16 + lane % 16, words 2 c
    // and 2 c + 1 of step c (the scales of 32-groups 4 c .. 4 c + 3).
    const uint32_t* dsrc = (const uint32_t*)a.sb + (size_t)((tn * PG_RB + srb) * 16 + (lane & 15)) * NG;
    constexpr size_t DSRC2 = (size_t)8 * 16 * NG;  // row block srb + 8

    f32x4 acc[TB][4 * NHF];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int r = 0; r < 4 * NHF; ++r) acc[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Activation operands of one 64-group (two k-steps), prefetched one group ahead.
    uint4 Ae[TB][2][HL], Ao[TB][2][HL];  // [token block][k-step of the group][hi, lo]
    uint4 Wn[NHF][CPS];
    uint32_t Vn = 0;
    uint32_t Dn[NHF][2];
    auto aload = [&](int g, uint4(&A)[TB][2][HL]) {
#pragma unroll
        for (int i = 0; i < TB; ++i) {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int hl = 0; hl < HL; ++hl)
                    A[i][kk][hl] = *(const uint4*)(xa + (size_t)i * NKS * 512 * HL + ((size_t)(2 * g + kk) * HL + hl) * 512);
        }
    };
    auto wload = [&](int c) {
#pragma unroll
        for (int hb = 0; hb < NHF; ++hb)
#pragma unroll
            for (int j = 0; j < CPS; ++j) Wn[hb][j] = *(const uint4*)(wsrc + hb * WSRC2 + (size_t)(c * CPS + j) * 1024);
        if (vload) Vn = vsrc[(size_t)c * vstride];
        if constexpr (DQ && FMT != FMT_F16) {  // f16 weights have no scales
#pragma unroll
            for (int hb = 0; hb < NHF; ++hb)
#pragma unroll
                for (int j = 0; j < 2; ++j) Dn[hb][j] = dsrc[hb * DSRC2 + 2 * c + j];
        }
    };
    // A chunk's lane is the B-operand lane of every format (XA follows the q4 K order).
    auto lstore = [&](int b) {
#pragma unroll
        for (int hb = 0; hb < NHF; ++hb) {
            const int sr = srb + 8 * hb;
            if constexpr (FMT == FMT_F16) {  // chunk j is k-step j
#pragma unroll
                for (int j = 0; j < 4; ++j) Bs[b][sr][j][lane] = Wn[hb][j];
            } else if constexpr (FMT == FMT_Q8) {
                // Bytes 0-7 of a lane of chunk j are k-step 2 j, bytes 8-15 k-step 2 j + 1.
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t dd[4] = {Wn[hb][j].x, Wn[hb][j].y, Wn[hb][j].z, Wn[hb][j].w};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        f16x2 o[4];
                        if constexpr (!DQ) unpack_q8_bytes(dd[2 * h], dd[2 * h + 1], o);
                        if constexpr (DQ) {  // 32-group 4 c + 2 j + h: the scale in half h of word 2 c + j
                            unpack_q8(dd[2 * h], dd[2 * h + 1], o);
                            const f16 sc = h ? as_h2(Dn[hb][j]).y : as_h2(Dn[hb][j]).x;
                            const f16x2 sc2 = {sc, sc};
#pragma unroll
                            for (int i = 0; i < 4; ++i) o[i] = o[i] * sc2;
                        }
                        Bs[b][sr][2 * j + h][lane] = pack4(o);
                    }
                }
            } else {
                // Dword 2 gg + h of a lane is k-step 2 gg + h.
                const uint32_t dd[4] = {Wn[hb][0].x, Wn[hb][0].y, Wn[hb][0].z, Wn[hb][0].w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    f16x2 o[4];
                    unpack_q4(dd[j], o);
                    Bs[b][sr][j][lane] = pack4(o);
                }
            }
        }
        if constexpr (!DQ) Vs[b][tid] = Vn;
    };
    // One activation operand (token block tb0 + i, k-step kk of group g, hi / lo part hl).
    auto aload1 = [&](int g, int i, int kk, int hl) {
        return *(const uint4*)(xa + (size_t)i * NKS * 512 * HL + ((size_t)(2 * g + kk) * HL + hl) * 512);
    };
    // One 64-group, in halves of four row blocks: a half's 8 B fragments first, then 4 x 2
    // accumulator chains of 4 MFMAs, then its scale epilogue.  In the last half, each activation
    // register is requested again for group gn (two groups on) as soon as its last product is
    // issued, so the loads have two groups' work to land in.
    auto group = [&](int b, int gg, uint4(&Ac)[TB][2][HL], int gn) {
#pragma unroll
      for (int hf = 0; hf < NHF; ++hf) {
        v8h Bf[4][2];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) Bf[r][kk] = __builtin_bit_cast(v8h, Bs[b][rb0 + 4 * hf + r][2 * gg + kk][lane]);
        if constexpr (DQ) {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int hl = 0; hl < HL; ++hl) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int i = 0; i < TB; ++i)
                            acc[i][4 * hf + r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                __builtin_bit_cast(v8h, Ac[i][kk][hl]), Bf[r][kk], acc[i][4 * hf + r], 0, 0, 0);
                    if (hf == NHF - 1) {
#pragma unroll
                        for (int i = 0; i < TB; ++i) Ac[i][kk][hl] = aload1(gn, i, kk, hl);
                    }
                }
            continue;
        }
        float2 sb[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f16x2 sb2 = as_h2(Vs[b][gg * TR + (rb0 + 4 * hf + r) * 16 + r16]);
            sb[r] = make_float2((float)sb2.x, (float)sb2.y);  // q4 (scale, bias); q8 the two 32-groups' scales
        }
        if constexpr (FMT == FMT_Q8) {
            // Two 32-groups, one k-step each.
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                f32x4 C[4][TB];
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < TB; ++i) C[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int hl = 0; hl < HL; ++hl) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int i = 0; i < TB; ++i)
                            C[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, Ac[i][kk][hl]),
                                                                             Bf[r][kk], C[r][i], 0, 0, 0);
                    if (hf == NHF - 1) {
#pragma unroll
                        for (int i = 0; i < TB; ++i) Ac[i][kk][hl] = aload1(gn, i, kk, hl);
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < TB; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[i][4 * hf + r][e] = fmaf(kk ? sb[r].y : sb[r].x, C[r][i][e], acc[i][4 * hf + r][e]);
            }
            continue;
        }
        f32x4 C[4][TB];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < TB; ++i) C[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int hl = 0; hl < HL; ++hl) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < TB; ++i)
                        C[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, Ac[i][kk][hl]), Bf[r][kk],
                                                                         C[r][i], 0, 0, 0);
                if (hf == NHF - 1) {
#pragma unroll
                    for (int i = 0; i < TB; ++i) Ac[i][kk][hl] = aload1(gn, i, kk, hl);
                }
            }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < TB; ++i) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // q4: the bias term sum_g b_g X_g went in before the loop
                    acc[i][4 * hf + r][e] = fmaf(sb[r].x, C[r][i][e], acc[i][4 * hf + r][e]);
                }
            }
      }
    };

    // Even groups use Ae, odd groups Ao: each register is reloaded (for two groups on) as its
    // group's last product using it issues, so no register copy waits on an outstanding load.
    aload(0, Ae);
    aload(1, Ao);
    wload(0);
    if constexpr (FMT == FMT_Q4) {
        // The q4 bias term sum_g b_g X_g of every output, on the matrix cores before the loop:
        // per 32 groups, A = the token block's group sums X (scaled by 2^-8 into fp16 range,
        // hi + lo parts) and B = the rows' fp16 biases, exact.  The loop's group epilogue is then
        // one fma per output (acc += s C_g).
#pragma unroll 1
        for (int cg = 0; cg < NG / 32; ++cg) {
            v8h Xh[TB], Xl[TB], Bb[4];
#pragma unroll
            for (int i = 0; i < TB; ++i) {
                const uint16_t* xp = a.xb + ((size_t)((tb0 + i) * (NG / 32) + cg) * 2 * 64 + lane) * 8;
                Xh[i] = *(const v8h*)xp;
                Xl[i] = *(const v8h*)(xp + 512);
            }
#pragma unroll
            for (int hf = 0; hf < NHF; ++hf) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint4* bp = (const uint4*)((const uint32_t*)a.sb +
                                                     (size_t)(tn * TR + (rb0 + 4 * hf + r) * 16 + r16) * NG + 32 * cg + 8 * q);
                    const uint4 w0 = bp[0], w1 = bp[1];
                    const uint32_t wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
                    for (int j = 0; j < 8; ++j) Bb[r][j] = as_h2(wv[j]).y;
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < TB; ++i) {
                        f32x4 B = f32x4{0.f, 0.f, 0.f, 0.f};
                        B = __builtin_amdgcn_mfma_f32_16x16x32_f16(Xh[i], Bb[r], B, 0, 0, 0);
                        B = __builtin_amdgcn_mfma_f32_16x16x32_f16(Xl[i], Bb[r], B, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][4 * hf + r][e] = fmaf(256.f, B[e], acc[i][4 * hf + r][e]);
                    }
            }
        }
    }
    lstore(0);
    __syncthreads();
    for (int c = 0; c < NC; ++c) {
        const int b = c & 1;
        // The next step's codes (the last step reloads step 0 into the idle buffer: no branch).
        wload(c + 1 < NC ? c + 1 : 0);
        group(b, 0, Ae, 2 * c + 2 < NG ? 2 * c + 2 : 0);
        group(b, 1, Ao, 2 * c + 3 < NG ? 2 * c + 3 : 1);
        lstore(b ^ 1);
        __syncthreads();
    }

    // Epilogue: lane holds tokens 16 tb + 4 q + e of weight row TR tn + 16 rb + r16.
#pragma unroll
    for (int i = 0; i < TB; ++i) {
        const int tq = (tb0 + i) * 16 + 4 * q;
        const float4 tsv = *(const float4*)(a.ts + tq);
        const float tsc[4] = {tsv.x, tsv.y, tsv.z, tsv.w};
#pragma unroll
        for (int r = 0; r < 4 * NHF; ++r) {
            const int rb = rb0 + r;
            const int row = tn * TR + rb * 16 + r16;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pf_store<EPI>(a, tq + e, row, acc[i][r][e] * tsc[e]);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// GEMM of prompts whose 128-token tiles leave the chip idle: K split over workgroups.
//
// A workgroup of 8 waves computes 16 TB tokens x 64 WN weight rows over a range of K: wave w owns
// row blocks 4 (w / WK) .. + 3 and every WK-th K unit of KU values (WK = 8 / WN), all tokens.  So
// a wave's weights are its own: they go from HBM to its registers (one unit ahead) and become B
// operands there, with no LDS round trip and no sharing.  The activation operands, which the WN
// row groups share, go to LDS by direct global-to-LDS loads, one iteration (WK units) ahead, in
// operand order (1 KiB per fragment, no bank conflicts).  One barrier an iteration.  At the end
// the WK waves of a row group add their sums through LDS (a fixed order).
//
// With a.splits > 1 the workgroup stores its sums as partials [split][M][N] and the kernel that
// consumes the result adds them (prep, q/k norm): no atomics, the same sums on every run.
//
// Workgroups run row tile by row tile on one XCD (token tiles innermost), so that the weights
// cross HBM once.
//
// Measured against the 128-token tiles, whose 96-192 workgroups each walked the whole K: q4, 307
// rows, hi + lo: gate|up 60 -> 40 us, down 65 -> 26, QKV 26 -> 20, O 25 -> 17; q8, 41 rows (padded
// to 128 there): 65 -> 16, 85 -> 13, 37 -> 10, 32 -> 9.  The loop runs at the rate of its products
// (33 of gate|up's 40 us with the products alone, at the clock that they leave); the rest is the
// first stage's arrival, ~3 us, the exchange and the stores, ~2-3 us.
template <int FMT, int K, int EPI, int TB, int HL, int WN>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void pf_split_kernel(PfGemmArgs a) {
    constexpr int WK = 8 / WN, NG = K / 64, NKS = K / 32, NXB = (NG + 31) / 32;
    // k-steps of a unit (KU = 32 KSU): a q4 chunk's 128 K, or 64 where that would not leave LDS for two stages.
    constexpr int KSU = FMT == FMT_Q4 && WN == 4 ? 4 : 2;
    constexpr int CPU = FMT == FMT_F16 ? 2 : 1;                     // 1 KiB weight chunks of a unit
    constexpr bool HALFCH = FMT == FMT_Q4 && KSU == 2;              // a unit is half a chunk (8 bytes a lane)
    constexpr int IKS = WK * KSU, NIT = NKS / IKS;                  // k-steps of an iteration, iterations of K
    constexpr int ACH = IKS * HL * TB, AW = ACH / 8;                // 1 KiB operand chunks of a stage, per wave
    constexpr int UN = TB * 4, UW = UN / WK;                        // 16 x 16 blocks of a wave's tile, finished per wave
    constexpr int REDCH = WN * UN * (WK - 1);                       // KiB of the final exchange
    constexpr int LDSB = (2 * ACH > REDCH ? 2 * ACH : REDCH) * 1024;
    constexpr bool DQ = HL == 1 || FMT == FMT_F16;
    static_assert(NKS % IKS == 0 && ACH % 8 == 0 && UN % WK == 0 && (UW == 2 || UW % 4 == 0) && LDSB <= 160 * 1024, "shape");
    __shared__ __align__(1024) uint8_t lds[LDSB];

    const int TN = a.N / (64 * WN), TM = (a.M + 16 * TB - 1) / (16 * TB), T = TM * TN * a.splits;
    const int per = (T + 7) / 8;
    const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= T) return;
    const int tm = tile % TM, sk = (tile / TM) % a.splits, tn = tile / TM / a.splits;
    const int it0 = sk * NIT / a.splits, it1 = (sk + 1) * NIT / a.splits;

    // The wave's index in a scalar register: its base addresses are scalar, its lanes add 32-bit offsets.
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), q = lane >> 4, r16 = lane & 15;
    const int wn = wave / WK, part = wave % WK;
    const int tb0 = tm * TB, rb0 = (tn * WN + wn) * 4;

    // A stage: chunk ((ks HL) + hl) TB + tb of the iteration's k-steps.
    // Buffer resources: a request is a scalar offset plus the lane's (no 64-bit lane addresses).
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.xa + (size_t)tb0 * NKS * HL * 512), (short)0, TB * NKS * HL * 1024, 0x00020000);
    auto aload = [&](int st, int it) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < AW; ++u) {
            const int ch = wave + 8 * u, tb = ch % TB, kh = ch / TB;  // kh = ks HL + hl
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (__attribute__((address_space(3))) void*)(lds + (st * ACH + ch) * 1024),
                                                     16, lane * 16, (tb * NKS * HL + it * IKS * HL + kh) * 1024, 0, 0);
        }
    };
    // Weights of one unit: row blocks rb0 .. + 3, and their scale words (q4 (scale, bias) of the
    // unit's two 64-groups; q8 the scales of its two 32-groups).
    struct Unit {
        uint4 w[4][CPU];
        uint2 s[4];
    };
    constexpr int RBW = FMT == FMT_Q4 ? K * 8 : FMT == FMT_Q8 ? K * 16 : K * 32;  // bytes of a row block's codes
    const uint8_t* sp = a.sb + (size_t)rb0 * 16 * NG * 4;  // (unused for f16)
    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + (size_t)rb0 * RBW), (short)0, 4 * RBW, 0x00020000);
    const __amdgpu_buffer_rsrc_t srs = __builtin_amdgcn_make_buffer_rsrc((void*)sp, (short)0, 64 * NG * 4, 0x00020000);
    const int wlane = lane * 16, slane = r16 * NG * 4;
    auto wload = [&](int it, Unit& u) __attribute__((always_inline)) {
        const int un = it * WK + part;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (HALFCH) {
                const uint2 h = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(wrs, wlane, r * RBW + (un >> 1) * 1024 + (un & 1) * 8, 0));
                u.w[r][0].x = h.x;
                u.w[r][0].y = h.y;
                u.s[r].x = __builtin_amdgcn_raw_buffer_load_b32(srs, slane, r * 16 * NG * 4 + un * 4, 0);
                continue;
            }
#pragma unroll
            for (int c = 0; c < CPU; ++c)
                u.w[r][c] = __builtin_bit_cast(
                    uint4, __builtin_amdgcn_raw_buffer_load_b128(wrs, wlane, r * RBW + (un * CPU + c) * 1024, 0));
            if constexpr (FMT == FMT_Q4)
                u.s[r] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(srs, slane, r * 16 * NG * 4 + un * 8, 0));
            if constexpr (FMT == FMT_Q8)
                u.s[r].x = __builtin_amdgcn_raw_buffer_load_b32(srs, slane, r * 16 * NG * 4 + un * 4, 0);
        }
    };

    f32x4 acc[TB][4];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};

    Unit un;
    aload(0, it0);
    wload(it0, un);
    if constexpr (FMT == FMT_Q4 && !DQ) {
        // The q4 bias term sum_g b_g X_g over the range's groups, on the matrix cores: 32 groups are
        // one k-step, A = the group sums (times 2^-8, hi + lo), B = the rows' fp16 biases, exact.  The
        // sums stay 2^-8 of their value until the end (the loop's scales are taken down with them).
        // Biases outside the range are requested past the buffer's end, which gives zeros (ranges
        // are whole fours of groups).
        const int g0 = it0 * IKS / 2, g1 = it1 * IKS / 2;
#pragma unroll 1
        for (int cg = g0 / 32; cg < (g1 + 31) / 32; ++cg) {
            if (cg % WK != part) continue;
            v8h Xh[TB], Xl[TB];
            uint4 w0[4], w1[4];
#pragma unroll
            for (int i = 0; i < TB; ++i) {
                const uint16_t* xp = a.xb + (size_t)((tb0 + i) * NXB + cg) * 2 * 64 * 8;
                Xh[i] = *(const v8h*)(xp + lane * 8);
                Xl[i] = *(const v8h*)(xp + 512 + lane * 8);
            }
            const int g = 32 * cg + 8 * q;
            const int o0 = g >= g0 && g < g1 ? slane + g * 4 : (int)0x80000000, o1 = g + 4 >= g0 && g + 4 < g1 ? slane + g * 4 + 16 : (int)0x80000000;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                w0[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(srs, o0 + r * 16 * NG * 4, 0, 0));
                w1[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(srs, o1 + r * 16 * NG * 4, 0, 0));
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint4 b = make_uint4(__builtin_amdgcn_perm(w0[r].y, w0[r].x, 0x07060302u), __builtin_amdgcn_perm(w0[r].w, w0[r].z, 0x07060302u),
                                           __builtin_amdgcn_perm(w1[r].y, w1[r].x, 0x07060302u), __builtin_amdgcn_perm(w1[r].w, w1[r].z, 0x07060302u));
#pragma unroll
                for (int i = 0; i < TB; ++i) {
                    acc[i][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Xh[i], __builtin_bit_cast(v8h, b), acc[i][r], 0, 0, 0);
                    acc[i][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Xl[i], __builtin_bit_cast(v8h, b), acc[i][r], 0, 0, 0);
                }
            }
        }
    }

    // One unit against the operands of stage st.
    auto mac = [&](int st, Unit u) __attribute__((always_inline)) {
        const uint8_t* A0 = lds + (size_t)(st * ACH + part * KSU * HL * TB) * 1024 + lane * 16;
#pragma unroll 1
        for (int g = 0; g < KSU / 2; ++g, A0 += 2 * HL * TB * 1024) {  // 64 K
            v8h A[2][HL][TB];
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int hl = 0; hl < HL; ++hl)
#pragma unroll
                    for (int i = 0; i < TB; ++i)
                        A[kk][hl][i] = *(const v8h*)(A0 + (size_t)((kk * HL + hl) * TB + i) * 1024);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v8h B[2];
                float s0 = 1.f, s1 = 1.f;
                if constexpr (FMT == FMT_F16) {
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) B[kk] = __builtin_bit_cast(v8h, u.w[r][kk]);
                } else {
                    const uint32_t dd[4] = {u.w[r][0].x, u.w[r][0].y, u.w[r][0].z, u.w[r][0].w};
                    const f16x2 sw = as_h2(u.s[r].x);
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) {
                        f16x2 o[4];
                        if constexpr (FMT == FMT_Q4)
                            unpack_q4(dd[kk], o);
                        else
                            unpack_q8(dd[2 * kk], dd[2 * kk + 1], o);
                        if constexpr (DQ) {  // one rounding each, as the 128-token tiles
                            const f16x2 sc2 = FMT == FMT_Q8 && kk ? f16x2{sw.y, sw.y} : f16x2{sw.x, sw.x};
                            const f16x2 bi2 = {sw.y, sw.y};
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                o[i] = FMT == FMT_Q4 ? __builtin_elementwise_fma(o[i], sc2, bi2) : o[i] * sc2;
                        }
                        B[kk] = __builtin_bit_cast(v8h, pack4(o));
                    }
                    s0 = FMT == FMT_Q4 ? (float)sw.x * 0.00390625f : (float)sw.x;
                    s1 = (float)sw.y;
                }
                if constexpr (DQ) {
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                        for (int hl = 0; hl < HL; ++hl)
#pragma unroll
                            for (int i = 0; i < TB; ++i)
                                acc[i][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[kk][hl][i], B[kk], acc[i][r], 0, 0, 0);
                } else {
                    f32x4 C[TB];
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) {
                        if (FMT == FMT_Q8 || kk == 0) {
#pragma unroll
                            for (int i = 0; i < TB; ++i) C[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                        }
#pragma unroll
                        for (int hl = 0; hl < HL; ++hl)
#pragma unroll
                            for (int i = 0; i < TB; ++i)
                                C[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[kk][hl][i], B[kk], C[i], 0, 0, 0);
                        if (FMT == FMT_Q8 || kk == 1) {
                            const float s = FMT == FMT_Q8 && kk ? s1 : s0;
#pragma unroll
                            for (int i = 0; i < TB; ++i)
#pragma unroll
                                for (int e = 0; e < 4; ++e) acc[i][r][e] = fmaf(s, C[i][e], acc[i][r][e]);
                        }
                    }
                }
                if constexpr (FMT == FMT_Q4) {  // the unit's second 64-group moves down
                    u.w[r][0].x = u.w[r][0].z;
                    u.w[r][0].y = u.w[r][0].w;
                    u.s[r].x = u.s[r].y;
                }
            }
        }
    };
    // Every load of the iteration was issued an iteration ago: wait for this wave's, then for every
    // wave's; the barrier also frees the stage read in the iteration before.
    auto arrive = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    for (int it = it0; it < it1; ++it) {
        arrive();
        const Unit u = un;  // landed: the copy waits for nothing, and its registers take the next unit
        const int st = (it - it0) & 1;
        if (it + 1 < it1) {
            aload(st ^ 1, it + 1);
            wload(it + 1, un);
        }
        mac(st, u);
    }

    // The row group's WK sums: block u (token block u / 4, row block u % 4) is finished by part u / UW.
    // (The code of a launch that lasts microseconds is fetched once per CU, so its length counts.)
    f32x4 sum[UW];
    {
        f32x4* red = (f32x4*)lds + (size_t)wn * UN * (WK - 1) * 64 + lane;
        __syncthreads();  // every operand read is done (no load is in flight)
#pragma unroll
        for (int p = 0; p < WK; ++p) {
            if (part != p) continue;  // one straight run of writes per part
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int own = u / UW;
                if (own == p)
                    sum[u % UW] = acc[u / 4][u % 4];
                else
                    red[(u * (WK - 1) + (p < own ? p : p - 1)) * 64] = acc[u / 4][u % 4];
            }
        }
        __syncthreads();
        red += (size_t)part * UW * (WK - 1) * 64;
#pragma unroll
        for (int i = 0; i < UW; ++i)
#pragma unroll
            for (int p = 0; p < WK - 1; ++p) {
                const f32x4 o = red[(i * (WK - 1) + p) * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[i][e] += o[e];
            }
    }
    // Lane: tokens 16 tb + 4 q + e of weight row 16 rb + r16.  Rows of tokens past M are past the
    // end of the destination's buffer resource and are dropped (the whole offset is the lane's: a
    // scalar offset past the end would wrap the bounds check).
    constexpr float UNBIAS = FMT == FMT_Q4 && !DQ ? 256.f : 1.f;
    const int tb1 = tb0 + part * UW / 4, r1 = part * UW % 4;  // UW is 2 or a multiple of 4
    float* dst = a.splits > 1 ? a.part + (size_t)sk * a.M * a.N : a.y;
    const __amdgpu_buffer_rsrc_t drs =
        __builtin_amdgcn_make_buffer_rsrc((void*)dst, (short)0, (int)((size_t)a.M * a.N * 4), 0x00020000);
#pragma unroll
    for (int i = 0; i < UW; ++i) {
        const int tq = (tb1 + i / 4) * 16, rb = rb0 + (UW < 4 ? r1 + i : i % 4);
        const float4 tsv = *(const float4*)(a.ts + tq + 4 * q);
        const float tsc[4] = {tsv.x, tsv.y, tsv.z, tsv.w};
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = sum[i][e] * (tsc[e] * UNBIAS);
        if (EPI == EPI_STORE || a.splits > 1) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                __builtin_amdgcn_raw_buffer_store_b32(as_u32(y[e]), drs, ((tq + 4 * q + e) * a.N + rb * 16 + r16) * 4, 0, 0);
        } else if constexpr (EPI == EPI_SWIGLU) {
            // Lanes r16 < 8 hold gate rows, r16 ^ 8 their up rows: the first take tokens 4 q, 4 q + 1, the
            // second 4 q + 2, 4 q + 3, so that every lane has two units.
            const bool lo = r16 < 8;
            const float o0 = dpp<0x128>(lo ? y[2] : y[0]), o1 = dpp<0x128>(lo ? y[3] : y[1]);
            const float h0 = lo ? swiglu(y[0], o0) : swiglu(o0, y[2]), h1 = lo ? swiglu(y[1], o1) : swiglu(o1, y[3]);
            const int t = tq + 4 * q + (lo ? 0 : 2);
            float* h = a.h + (size_t)t * FF + rb * 8 + (r16 & 7);
            if (t < a.M) h[0] = h0;
            if (t + 1 < a.M) h[FF] = h1;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) pf_store<EPI>(a, tq + 4 * q + e, rb * 16 + r16, y[e]);
        }
    }
}

// ------------------------------------------------------------------------------------------
// Per-head q/k RMSNorm + M-RoPE of every prompt row, K/V written to the fp16 cache, queries
// pre-scaled by log2(e) / sqrt(128) and split into fp16 hi + lo.  Grid (M, 8): wave 4 y + w handles
// vector 4 y + w of row x (q heads 0-15, k groups 16-23, v groups 24-31).

__global__ __launch_bounds__(256) void pf_qk_kernel(PfQkArgs a) {
    const int t = blockIdx.x, lane = threadIdx.x % 64, vec = blockIdx.y * 4 + threadIdx.x / 64;
    if (t >= a.M) return;
    const int slot = a.p0 + t;
    // The vector's two elements of this lane (vectors are q heads, k groups, v groups in row order),
    // the sum of the QKV GEMM's K-split partials.
    float x0, x1;
    if (a.nsplit == 1) {
        const float* row = a.qkv + (size_t)t * QKV + vec * HD + lane;
        x0 = row[0];
        x1 = row[64];
    } else {
        const Parts qp(a.qkv, (size_t)a.nsplit * a.M * QKV);
        x0 = x1 = 0.f;
        for (int s0 = 0; s0 < a.nsplit; s0 += 8) {
            float y[8][2];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int at = ((s0 + i) * a.M + t) * QKV + vec * HD + lane;
                y[i][0] = qp.load(at);
                y[i][1] = qp.load(at + 64);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                x0 += y[i][0];
                x1 += y[i][1];
            }
        }
    }
    const float* cs = a.rope + (size_t)slot * 128;
    if (vec < NH) {
        norm_rope_pair(x0, x1, a.q_norm, cs, lane);
        // 1/sqrt(128) and log2(e): the scores come out in base-2 units, so every softmax
        // exponential of the attention is one v_exp_f32.
        const float qscale = (1.0f / sqrtf((float)HD)) * 1.4426950408889634f;
        x0 *= qscale;
        x1 *= qscale;
        const size_t o = ((size_t)t * NH + vec) * HD + lane;
        const f16 h0 = (f16)x0, h1 = (f16)x1;
        a.qh[o] = __builtin_bit_cast(uint16_t, h0);
        a.qh[o + 64] = __builtin_bit_cast(uint16_t, h1);
        if (a.ql) {
            a.ql[o] = f2h(x0 - (float)h0);
            a.ql[o + 64] = f2h(x1 - (float)h1);
        }
    } else if (vec < NH + NKV) {
        const int g = vec - NH;
        norm_rope_pair(x0, x1, a.k_norm, cs, lane);
        uint16_t* kd = a.kc + ((size_t)g * a.maxctx + slot) * HD;
        kd[lane] = f2h(x0);
        kd[lane + 64] = f2h(x1);
    } else {
        const int g = vec - NH - NKV;
        uint16_t* vd = a.vc + ((size_t)g * a.maxctx + slot) * HD;
        vd[lane] = f2h(x0);
        vd[lane + 64] = f2h(x1);
    }
}

// ------------------------------------------------------------------------------------------
// Causal GQA flash attention.  Workgroup = (KV group g, 64-token query block), 8 waves.  Wave w
// handles head 2 g + ((w >> 1) & 1) for tokens 32 (w & 1) .. + 31 of the block as two 16-row
// query tiles, so every K and V operand it reads from LDS feeds two products.  Each iteration
// stages 128 key slots in LDS as two 64-slot halves (K row-major, V transposed; double-buffered)
// and wave w takes half w >> 2: the two key-parity waves of a (head, tokens) pair keep separate
// running softmax states, merged through LDS after the last iteration.  Slots at or beyond the
// block's last query are masked for all of its queries; causal masking uses cache slots.  The
// softmax denominators come from the matrix cores too: a ones operand against the probabilities.
//
// With a.nsplit > 1 (few query blocks) a block's key iterations are dealt to nsplit workgroups,
// each storing its unnormalised rows and their (maximum, denominator); the operand prep of the O
// projection merges them.

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int PA_KB = 64;     // keys per half
constexpr int PA_KROW = 136;  // halves per K row in LDS (128 + 8 pad)
constexpr int PA_VROW = 68;   // halves per V^T row in LDS (64 keys + 4 pad)
constexpr int PA_BUF = PA_KB * PA_KROW + HD * PA_VROW;  // halves per 64-slot half
constexpr size_t PA_LDS = 4 * PA_BUF * 2;                // two stages of two halves: 139,264 B

template <int HL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void pf_attn_kernel(PfAttnArgs a) {
    extern __shared__ __align__(16) uint16_t pa_lds[];
    const int QB = (a.M + 63) / 64;
    const int g = (int)(blockIdx.x % NKV), qs = (int)(blockIdx.x / NKV), qb = QB - 1 - qs / a.nsplit, sp = qs % a.nsplit;
    if (qb < 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, r16 = lane & 15;
    const int par = wave >> 2, wi = wave & 3;
    const int head = 2 * g + (wi >> 1);
    const int t0 = qb * 64 + 32 * (wi & 1);
    const int kv_lim = a.p0 + min(a.M, qb * 64 + 64);  // past the block's last query slot
    const int nkb = (kv_lim - 1) / PA_KB + 1;          // 64-slot key halves with unmasked keys
    const int nit = (nkb + 1) / 2;
    const int it0 = sp * nit / a.nsplit, it1 = (sp + 1) * nit / a.nsplit;  // may be empty
    const bool active = t0 < a.M;
    const int w_first = a.p0 + t0;
    const int w_last = a.p0 + min(a.M - 1, t0 + 31);

    v8h Qh[2][4], Ql[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const size_t qo = ((size_t)(t0 + 16 * u + r16) * NH + head) * HD + 8 * q;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            Qh[u][ks] = *(const v8h*)(a.qh + qo + 32 * ks);
            if constexpr (HL == 2) Ql[u][ks] = *(const v8h*)(a.ql + qo + 32 * ks);
        }
    }
    const uint16_t* kg = a.kc + (size_t)g * a.maxctx * HD;
    const uint16_t* vg = a.vc + (size_t)g * a.maxctx * HD;

    // Staging through buffer resources bounded at kv_lim: slots at or past it (masked for every
    // query of the block) read as zeros, with no branch.  Half hb of iteration it: K key tid / 8,
    // dims 16 (tid % 8) .. + 15; V keys 4 (tid / 32) .. + 3, dims 4 (tid % 32) .. + 3 (transposed
    // in registers, 8-byte LDS writes).
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)kg, (short)0, kv_lim * HD * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)vg, (short)0, kv_lim * HD * 2, 0x00020000);
    struct Half {
        u32x4 k0, k1;
        u32x2 v0, v1, v2, v3;
    };
    Half h0, h1;
    const int koff = ((tid >> 3) * HD + 16 * (tid & 7)) * 2, voff = (4 * (tid >> 5) * HD + 4 * (tid & 31)) * 2;
    auto gload_half = [&](int base, Half& h) {
        const int o = base * HD * 2;
        h.k0 = __builtin_amdgcn_raw_buffer_load_b128(krs, o + koff, 0, 0);
        h.k1 = __builtin_amdgcn_raw_buffer_load_b128(krs, o + koff + 16, 0, 0);
        h.v0 = __builtin_amdgcn_raw_buffer_load_b64(vrs, o + voff, 0, 0);
        h.v1 = __builtin_amdgcn_raw_buffer_load_b64(vrs, o + voff + HD * 2, 0, 0);
        h.v2 = __builtin_amdgcn_raw_buffer_load_b64(vrs, o + voff + HD * 4, 0, 0);
        h.v3 = __builtin_amdgcn_raw_buffer_load_b64(vrs, o + voff + HD * 6, 0, 0);
    };
    auto gload = [&](int it) {
        gload_half(2 * it * PA_KB, h0);
        gload_half((2 * it + 1) * PA_KB, h1);
    };
    auto lstore_half = [&](uint16_t* Ks, const Half& h) {
        uint16_t* Vt = Ks + PA_KB * PA_KROW;
        u32x4* kd = (u32x4*)(Ks + (tid >> 3) * PA_KROW + 16 * (tid & 7));
        kd[0] = h.k0;
        kd[1] = h.k1;
        const int d0 = 4 * (tid & 31), k0 = 4 * (tid >> 5);
        // Output row d0 + j holds dim d0 + j of keys k0 .. k0 + 3: byte selects from the four rows.
        const u32x2 vr[4] = {h.v0, h.v1, h.v2, h.v3};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int w = j >> 1;
            const unsigned sel = (j & 1) ? 0x07060302u : 0x05040100u;  // high or low halves of two words
            *(u32x2*)(Vt + (d0 + j) * PA_VROW + k0) =
                u32x2{__builtin_amdgcn_perm(vr[1][w], vr[0][w], sel), __builtin_amdgcn_perm(vr[3][w], vr[2][w], sel)};
        }
    };
    auto lstore = [&](int stage) {
        lstore_half(pa_lds + (2 * stage) * PA_BUF, h0);
        lstore_half(pa_lds + (2 * stage + 1) * PA_BUF, h1);
    };

    f32x4 O[2][8], Lr[2];  // Lr: the running denominator of query r16 in every element
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        Lr[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) O[u][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float m_run[2] = {-__builtin_inff(), -__builtin_inff()};
    const f16 one = (f16)1.0f;
    const v8h ones = {one, one, one, one, one, one, one, one};

    gload(it0);
    lstore(0);
    __syncthreads();
    for (int it = it0; it < it1; ++it) {
        const int st = (it - it0) & 1;
        if (it + 1 < it1) gload(it + 1);
        const int kb = 2 * it + par;
        if (active && kb * PA_KB <= w_last) {
            const uint16_t* Ks = pa_lds + (2 * st + par) * PA_BUF;
            const uint16_t* Vt = Ks + PA_KB * PA_KROW;
            // S^T tiles: keys 16 kt + (4 q + i) of this lane, query r16 of tile u.
            f32x4 S[2][4];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                S[0][kt] = S[1][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const v8h kf = *(const v8h*)(Ks + (kt * 16 + r16) * PA_KROW + 32 * ks + 8 * q);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        S[u][kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, Qh[u][ks], S[u][kt], 0, 0, 0);
                        if constexpr (HL == 2)
                            S[u][kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, Ql[u][ks], S[u][kt], 0, 0, 0);
                    }
                }
            }
            // Schedule: the K operands of key tile kt + 1 are read while tile kt's products issue.
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                __builtin_amdgcn_sched_group_barrier(0x008, 8 * HL, 0);
                if (kt < 2) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            }
            // Masking only where some key of the half lies past some query of the wave (a
            // wave-uniform branch: the halves below the diagonal skip it).
            if (kb * PA_KB + PA_KB - 1 > w_first) {
                asm volatile("");  // keeps the branch: the selects below are not speculated
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int qslot = w_first + 16 * u + r16;
#pragma unroll
                    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (kb * PA_KB + kt * 16 + 4 * q + i > qslot) S[u][kt][i] = -__builtin_inff();
                }
            }
            v8h Ph[2][2], Pl[2][2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float mb = -__builtin_inff();
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) mb = fmaxf(mb, S[u][kt][i]);
                mb = max_x4(mb);
                const float m_new = fmaxf(m_run[u], mb);
                const float corr = m_new == m_run[u] ? 1.f
                                 : m_run[u] == -__builtin_inff() ? 0.f
                                 : __builtin_amdgcn_exp2f(m_run[u] - m_new);
                // A query whose keys so far are all masked keeps m = -inf: subtract 0 there, so
                // that every masked score gives exp2(-inf) = 0 without a per-element test.
                const float m_use = m_new == -__builtin_inff() ? 0.f : m_new;
                float p[4][4];
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) p[kt][i] = __builtin_amdgcn_exp2f(S[u][kt][i] - m_use);
                m_run[u] = m_new;
                // The running maximum settles after the first blocks: rescale only when it moved.
                if (__builtin_amdgcn_ballot_w64(corr != 1.f)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) Lr[u][i] *= corr;
#pragma unroll
                    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) O[u][dt][i] *= corr;
                }
                // P^T of key tiles 2c, 2c + 1 is the B operand over keys {32 c + 4 q + i, 32 c + 16 + 4 q + i}.
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f16 h0 = (f16)p[2 * c][i], h1 = (f16)p[2 * c + 1][i];
                        Ph[u][c][i] = h0;
                        Ph[u][c][4 + i] = h1;
                        if constexpr (HL == 2) {
                            Pl[u][c][i] = (f16)(p[2 * c][i] - (float)h0);
                            Pl[u][c][4 + i] = (f16)(p[2 * c + 1][i] - (float)h1);
                        }
                    }
            }
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    Lr[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, Ph[u][c], Lr[u], 0, 0, 0);
                    if constexpr (HL == 2) Lr[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, Pl[u][c], Lr[u], 0, 0, 0);
                }
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) {
                    const uint16_t* vp = Vt + (dt * 16 + r16) * PA_VROW + 32 * c + 4 * q;
                    const v4h va = *(const v4h*)vp, vb = *(const v4h*)(vp + 16);
                    const v8h vf = {va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        O[u][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, Ph[u][c], O[u][dt], 0, 0, 0);
                        if constexpr (HL == 2)
                            O[u][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, Pl[u][c], O[u][dt], 0, 0, 0);
                    }
                }
            // Schedule (fp16 operands alone; the hi + lo instance measured faster without it):
            // each group of four V operands is read two groups ahead of its products.
            if constexpr (HL == 1) {
                __builtin_amdgcn_sched_group_barrier(0x100, 4, 1);
                __builtin_amdgcn_sched_group_barrier(0x100, 4, 1);
                __builtin_amdgcn_sched_group_barrier(0x002 | 0x400, 200, 1);
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 8, 1);
                    if (k < 2) __builtin_amdgcn_sched_group_barrier(0x100, 4, 1);
                }
            }
        }
        if (it + 1 < it1) lstore(st ^ 1);
        __syncthreads();
    }

    // Key-parity merge: waves 4..7 hand (O, m, l) to waves 0..3 through LDS (free after the loop's
    // last barrier).  Unsplit, waves 0..3 always have a finite maximum: half 0 holds key slot 0.  A
    // split may see no key of a query: its maximum stays -inf, its sums 0.
    float* mo = (float*)pa_lds;               // [4 waves][2 tiles][8 dim tiles][64 lanes] x 4
    float* mml = mo + 4 * 2 * 8 * 64 * 4;     // [4 waves][2 tiles][64 lanes] x (m, l)
    if (par == 1) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) *(f32x4*)(mo + (((wi * 2 + u) * 8 + dt) * 64 + lane) * 4) = O[u][dt];
            *(float2*)(mml + ((wi * 2 + u) * 64 + lane) * 2) = make_float2(m_run[u], Lr[u][0]);
        }
    }
    __syncthreads();
    if (par == 0 && active) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int t = t0 + 16 * u + r16;
            const float2 ml1 = *(const float2*)(mml + ((wi * 2 + u) * 64 + lane) * 2);
            const float m = fmaxf(m_run[u], ml1.x);
            const float f0 = m == m_run[u] ? 1.f : __builtin_amdgcn_exp2f(m_run[u] - m);
            const float f1 = ml1.x == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(ml1.x - m);
            const float l = Lr[u][0] * f0 + ml1.y * f1;
            const float inv = a.nsplit > 1 ? 1.0f : 1.0f / l;
            float* out = a.nsplit > 1 ? a.part + (size_t)sp * a.M * H : a.out;
            if (t < a.M) {
                if (a.nsplit > 1 && q == 0) ((float2*)a.part_ml)[((size_t)sp * a.M + t) * NH + head] = make_float2(m, l);
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) {
                    const f32x4 o1 = *(const f32x4*)(mo + (((wi * 2 + u) * 8 + dt) * 64 + lane) * 4);
                    const float4 o = make_float4((O[u][dt][0] * f0 + o1[0] * f1) * inv, (O[u][dt][1] * f0 + o1[1] * f1) * inv,
                                                 (O[u][dt][2] * f0 + o1[2] * f1) * inv, (O[u][dt][3] * f0 + o1[3] * f1) * inv);
                    *(float4*)(out + (size_t)t * H + head * HD + dt * 16 + 4 * q) = o;
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------

template <int K, int SRC, bool PARTS>
static hipError_t pf_prep_src(int fmt, const PfPrepArgs& a, hipStream_t s) {
    const dim3 grid(a.Mpad), block(256);
    if (a.parts == 2 && fmt == FMT_Q4)
        hipLaunchKernelGGL((pf_prep_kernel<K, SRC, 2, true, PARTS>), grid, block, 0, s, a);
    else if (a.parts == 2)
        hipLaunchKernelGGL((pf_prep_kernel<K, SRC, 2, false, PARTS>), grid, block, 0, s, a);
    else if (fmt == FMT_Q4)
        hipLaunchKernelGGL((pf_prep_kernel<K, SRC, 1, true, PARTS>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((pf_prep_kernel<K, SRC, 1, false, PARTS>), grid, block, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pf_prep(int fmt, int src, const PfPrepArgs& a, hipStream_t s) {
    if (a.M < 1 || a.Mpad < a.M || a.Mpad % 8 || (a.parts != 1 && a.parts != 2) || a.nsplit < 0 ||
        (a.nsplit > 0 && !a.part))
        return hipErrorInvalidValue;
    switch (src) {
        case PF_SRC_RESID:
            return a.nsplit > 0 ? pf_prep_src<H, PF_SRC_RESID, true>(fmt, a, s) : pf_prep_src<H, PF_SRC_RESID, false>(fmt, a, s);
        case PF_SRC_ATTN:
            if (a.nsplit > 32) return hipErrorInvalidValue;
            return a.nsplit > 1 ? pf_prep_src<H, PF_SRC_ATTN, true>(fmt, a, s) : pf_prep_src<H, PF_SRC_ATTN, false>(fmt, a, s);
        case PF_SRC_SWIGLU:
            return a.nsplit > 1 ? pf_prep_src<FF, PF_SRC_SWIGLU, true>(fmt, a, s) : pf_prep_src<FF, PF_SRC_SWIGLU, false>(fmt, a, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_pf_last_row(const PfPrepArgs& a, int t, hipStream_t s) {
    if (t < 0 || t >= a.M || a.nsplit < 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pf_last_row_kernel, dim3(H / 256), dim3(256), 0, s, a, t);
    return hipGetLastError();
}

template <int FMT, int RB, int TB, int HL>
static hipError_t pf_gemm_shape(int K, int epi, const PfGemmArgs& a, hipStream_t s) {
    const int T = (a.Mpad / (64 * TB)) * (a.N / (16 * RB));
    const dim3 grid(8 * ((T + 7) / 8));
    if (K == H && epi == EPI_STORE)
        hipLaunchKernelGGL((pf_gemm_kernel<FMT, H, EPI_STORE, RB, TB, HL>), grid, dim3(512), 0, s, a);
    else if (K == H && epi == EPI_RESID)
        hipLaunchKernelGGL((pf_gemm_kernel<FMT, H, EPI_RESID, RB, TB, HL>), grid, dim3(512), 0, s, a);
    else if (K == H && epi == EPI_SWIGLU)
        hipLaunchKernelGGL((pf_gemm_kernel<FMT, H, EPI_SWIGLU, RB, TB, HL>), grid, dim3(512), 0, s, a);
    else if (K == FF && epi == EPI_RESID)
        hipLaunchKernelGGL((pf_gemm_kernel<FMT, FF, EPI_RESID, RB, TB, HL>), grid, dim3(512), 0, s, a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// Tiles that fill the 256 CUs evenly: at least one each, and a whole number each or at least four.
static bool even_fill(int tiles) { return tiles >= 256 && (tiles % 256 == 0 || tiles >= 1024); }

// The largest tile whose count fills the CUs evenly: 128 tokens x 256 rows, 128 x 128, else
// 64 x 128.  f16 weights keep 128-row tiles (their four chunks a step would not fit the registers of
// the larger one).  fp16 operands alone keep 128-row tiles: their 128-row tile needs ~110 registers and 64 KiB of LDS, so two
// workgroups share a CU (measured 21.55 -> 20.97 ms per 4096-row prefill against 256-row tiles).
template <int FMT, int HL>
static hipError_t pf_gemm_fmt(int K, int epi, const PfGemmArgs& a, hipStream_t s) {
    const int tm128 = a.Mpad / 128;
    if constexpr (HL == 2 && FMT != FMT_F16)
        if (even_fill(tm128 * (a.N / 256))) return pf_gemm_shape<FMT, 16, 2, HL>(K, epi, a, s);
    if (even_fill(tm128 * (a.N / 128))) return pf_gemm_shape<FMT, 8, 2, HL>(K, epi, a, s);
    return pf_gemm_shape<FMT, 8, 1, HL>(K, epi, a, s);
}

template <int FMT, int TB, int HL, int WN>
static hipError_t pf_split_shape(int K, int epi, const PfGemmArgs& a, hipStream_t s) {
    const int T = ((a.M + 16 * TB - 1) / (16 * TB)) * (a.N / (64 * WN)) * a.splits;
    const dim3 grid(8 * ((T + 7) / 8)), block(512);
    if (K == H && epi == EPI_STORE)
        hipLaunchKernelGGL((pf_split_kernel<FMT, H, EPI_STORE, TB, HL, WN>), grid, block, 0, s, a);
    else if (K == H && epi == EPI_RESID)
        hipLaunchKernelGGL((pf_split_kernel<FMT, H, EPI_RESID, TB, HL, WN>), grid, block, 0, s, a);
    else if (K == H && epi == EPI_SWIGLU)
        hipLaunchKernelGGL((pf_split_kernel<FMT, H, EPI_SWIGLU, TB, HL, WN>), grid, block, 0, s, a);
    else if (K == FF && epi == EPI_RESID)
        hipLaunchKernelGGL((pf_split_kernel<FMT, FF, EPI_RESID, TB, HL, WN>), grid, block, 0, s, a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// Tiles of the K-split GEMM: 32 tokens (two token blocks) up to 32 rows, else 64; 128 weight rows
// while there is one token tile, and for O and down (N = 2048) up to four, where the partials of
// twice the splits would cost more than the operands of twice the tiles (q4 at 128 rows 0.461 /
// 0.483 ms, 4 layers and the head; 0.590 / 0.616 at 256, 0.657 / 0.654 at 307), else 256 (a tile's
// operands are then shared by four row groups).
// With fp16 operands alone there are half the products per unpacked weight, and the unpacking bounds
// a 64-token tile: 128 tokens from the size on where that pays (4 layers and the head, 128 / 64
// tokens, ms): q8 0.57 / 0.59 at 256 rows, 1.04 / 1.21 at 1000; f16 0.69 / 0.74 at 384, 0.62 / 0.60 at
// 256; q4 1.08 / 1.28 at 1280, 0.93 / 0.89 at 1000.
struct PfSplitShape {
    int tb, wn, nit;  // token blocks, row groups, iterations of K
};
static int pf_wide_rows(int fmt) { return fmt == FMT_Q8 ? 192 : fmt == FMT_F16 ? 320 : 1152; }
static PfSplitShape pf_split_tile(int fmt, int parts, int K, int N, int M) {
    const int tb = M <= 32 ? 2 : parts == 1 && M >= pf_wide_rows(fmt) ? 8 : 4;
    const int wn = M <= 64 || (M <= 256 && N == H && tb == 4) ? 2 : 4;
    const int unit = fmt == FMT_Q4 && wn == 4 ? 128 : 64;
    return {tb, wn, K / (8 / wn * unit)};
}

template <int FMT>
static hipError_t pf_split_fmt(int K, int epi, const PfGemmArgs& a, hipStream_t s) {
    const PfSplitShape t = pf_split_tile(FMT, a.parts, K, a.N, a.M);
    if (a.parts == 1)
        return t.tb == 2   ? pf_split_shape<FMT, 2, 1, 2>(K, epi, a, s)
               : t.tb == 8 ? pf_split_shape<FMT, 8, 1, 4>(K, epi, a, s)
               : t.wn == 2 ? pf_split_shape<FMT, 4, 1, 2>(K, epi, a, s)
                           : pf_split_shape<FMT, 4, 1, 4>(K, epi, a, s);
    return t.tb == 2   ? pf_split_shape<FMT, 2, 2, 2>(K, epi, a, s)
           : t.wn == 2 ? pf_split_shape<FMT, 4, 2, 2>(K, epi, a, s)
                       : pf_split_shape<FMT, 4, 2, 4>(K, epi, a, s);
}

int pf_gemm_splits(int fmt, int parts, int K, int N, int M) {
    if (!pf_use_split(fmt, parts, M)) return 1;
    const PfSplitShape t = pf_split_tile(fmt, parts, K, N, M);
    const int tiles = ((M + 16 * t.tb - 1) / (16 * t.tb)) * (N / (64 * t.wn));
    const int most = std::max(1, std::min(t.nit, 256 / tiles));
    const int its = (t.nit + most - 1) / most;
    return (t.nit + its - 1) / its;
}

hipError_t launch_pf_gemm(int fmt, int K, int epi, const PfGemmArgs& a, hipStream_t s) {
    if (a.M < 1 || a.N % 256 || (a.parts != 1 && a.parts != 2) || a.splits < 1 || (a.splits > 1 && !a.part))
        return hipErrorInvalidValue;
    if (pf_use_split(fmt, a.parts, a.M)) {
        // The tiles of 128 tokens (fp16 operands alone) need rows up to a multiple of 128.
        const int pad = a.parts == 1 && a.M > 64 ? 128 : 64;
        if (a.splits != pf_gemm_splits(fmt, a.parts, K, a.N, a.M) || a.Mpad < (a.M + pad - 1) / pad * pad)
            return hipErrorInvalidValue;
        switch (fmt) {
            case FMT_Q4: return pf_split_fmt<FMT_Q4>(K, epi, a, s);
            case FMT_Q8: return pf_split_fmt<FMT_Q8>(K, epi, a, s);
            case FMT_F16: return pf_split_fmt<FMT_F16>(K, epi, a, s);
        }
        return hipErrorInvalidValue;
    }
    if (a.Mpad < a.M || a.Mpad % 128 || a.splits != 1) return hipErrorInvalidValue;
    if (fmt == FMT_Q8) return a.parts == 2 ? pf_gemm_fmt<FMT_Q8, 2>(K, epi, a, s) : pf_gemm_fmt<FMT_Q8, 1>(K, epi, a, s);
    if (fmt == FMT_Q4 && a.parts == 2) return pf_gemm_fmt<FMT_Q4, 2>(K, epi, a, s);
    if (fmt == FMT_F16 && a.parts == 2) return pf_gemm_fmt<FMT_F16, 2>(K, epi, a, s);
    return hipErrorInvalidValue;  // pf_use_split sends every other chunk the other way
}

hipError_t launch_pf_qk(const PfQkArgs& a, hipStream_t s) {
    if (a.M < 1 || a.p0 < 0 || a.p0 + a.M > a.maxctx || a.nsplit < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pf_qk_kernel, dim3(a.M, (NH + 2 * NKV) / 4), dim3(256), 0, s, a);
    return hipGetLastError();
}

int pf_attn_splits(int M, int p0) {
    const int QB = (M + 63) / 64, nit = (p0 + M + 2 * PA_KB - 1) / (2 * PA_KB);  // iterations of the last block
    return std::max(1, std::min(nit, 256 / (QB * NKV)));
}

hipError_t launch_pf_attn(const PfAttnArgs& a, hipStream_t s) {
    if (a.M < 1 || a.p0 < 0 || a.p0 + a.M > a.maxctx || a.nsplit < 1 || (a.nsplit > 1 && (!a.part || !a.part_ml)))
        return hipErrorInvalidValue;
    static bool attr_set = false;
    if (!attr_set) {
        for (const void* k : {(const void*)pf_attn_kernel<1>, (const void*)pf_attn_kernel<2>}) {
            hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)PA_LDS);
            if (e != hipSuccess) return e;
        }
        attr_set = true;
    }
    const dim3 grid((a.M + 63) / 64 * NKV * a.nsplit);
    if (a.ql)
        hipLaunchKernelGGL(pf_attn_kernel<2>, grid, dim3(512), PA_LDS, s, a);
    else
        hipLaunchKernelGGL(pf_attn_kernel<1>, grid, dim3(512), PA_LDS, s, a);
    return hipGetLastError();
}

}  // namespace icua
