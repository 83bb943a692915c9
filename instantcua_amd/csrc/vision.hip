// Qwen3-VL vision tower on gfx950: patchify, patch embedding with the interpolated position
// table, 24 pre-norm blocks (2D RoPE, bidirectional attention, GELU-tanh MLP), three DeepStack
// mergers after blocks 5, 11 and 17, and the final merger (Sources/Engine/Engine.swift:317-473;
// Shaders.swift:59-454).  Weights are fp16 [out][in] matrices with float32 biases and norms.
//
// Every projection is one matrix-core GEMM (v_mfma_f32_16x16x32_f16) with its elementwise
// work in the epilogue: bias, position table, residual add, GELU (tanh or erf) with the fp16
// rounding of the next GEMM's operand, and for QKV the 2D RoPE of q and k with a head-major
// fp16 split and V stored transposed for the attention.  Attention is one flash-style kernel
// per (head, 64 queries) on the matrix cores with an online softmax.  fp16 rounding points are
// those of the reference engine: LayerNorm outputs, q / k / v, probabilities, attention output
// and fc1 activations; the residual stream is float32.
#include "icua_device.h"
#include "icua_kernels.h"

namespace icua {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// RGB8 [16 gh][16 gw][3] -> fp16 patches in 2 x 2 merge-block order: patch p = 4 block + 2 ir +
// ic, element c * 256 + dy * 16 + dx, value u8 * (2 / 255) - 1 (k_vit_patchify_rgb,
// Shaders.swift:84-111).
__global__ __launch_bounds__(256) void vit_patchify_kernel(const uint8_t* __restrict__ rgb, uint16_t* __restrict__ patches,
                                                           int gh, int gw) {
#pragma clang fp contract(off)
    const int p = blockIdx.x;
    const int mw = gw / 2, blk = p / 4, in = p % 4;
    const int pr = (blk / mw) * 2 + in / 2, pc = (blk % mw) * 2 + in % 2;
    const int img_w = gw * 16;
    for (int i = threadIdx.x; i < VPATCH; i += 256) {
        const int c = i / 256, dy = (i % 256) / 16, dx = i % 16;
        const uint8_t v = rgb[((size_t)(pr * 16 + dy) * img_w + pc * 16 + dx) * 3 + c];
        const float a = (float)v * (2.0f / 255.0f);
        patches[(size_t)p * VPATCH + i] = f2h(a - 1.0f);
    }
}

// LayerNorm (eps 1e-6) over N columns, one wave per row, fp16 out (k_vit_ln1024 / k_vit_ln4096,
// Shaders.swift:116-199): ((x - mean) * rstd) * w + b.
template <int N>
__global__ __launch_bounds__(256) void vit_layernorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ b, uint16_t* __restrict__ out,
                                                            int rows) {
#pragma clang fp contract(off)
    constexpr int NV = N / 256;
    const int r = blockIdx.x * 4 + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (r >= rows) return;
    const float4* xr = (const float4*)(x + (size_t)r * N);
    float4 v[NV];
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        v[k] = xr[lane + WAVE * k];
        s += (v[k].x + v[k].y) + (v[k].z + v[k].w);
    }
    const float mean = wave_sum(s) / (float)N;
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        v[k].x -= mean;
        v[k].y -= mean;
        v[k].z -= mean;
        v[k].w -= mean;
        ss += (v[k].x * v[k].x + v[k].y * v[k].y) + (v[k].z * v[k].z + v[k].w * v[k].w);
    }
    const float rstd = 1.0f / sqrtf(wave_sum(ss) / (float)N + 1e-6f);
    uint2* o = (uint2*)(out + (size_t)r * N);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int i = lane + WAVE * k;
        const float4 wv = ((const float4*)w)[i], bv = ((const float4*)b)[i];
        const uint32_t h0 = f2h(v[k].x * rstd * wv.x + bv.x), h1 = f2h(v[k].y * rstd * wv.y + bv.y);
        const uint32_t h2 = f2h(v[k].z * rstd * wv.z + bv.z), h3 = f2h(v[k].w * rstd * wv.w + bv.w);
        o[i] = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
    }
}

// Barrier for LDS filled by global-to-LDS loads: this wave waits until at most `pending` of its
// vector-memory loads are outstanding (expcnt and lgkmcnt at their maximum), then all waves meet.
// __syncthreads() would also drain every load in flight, which empties the load pipeline; the
// empty asm statements keep the compiler from moving memory accesses across the barrier.
template <int pending>
__device__ __forceinline__ void dma_barrier() {
    static_assert(pending >= 0 && pending <= 63, "vmcnt");
    __builtin_amdgcn_s_waitcnt((pending & 15) | (7 << 4) | (15 << 8) | ((pending >> 4) << 14));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 0.5 x (1 + tanh(u)) = x / (1 + exp(-2 u)), u = sqrt(2 / pi) (x + 0.044715 x^3): one v_exp and one
// v_rcp (tanhf made the epilogue of fc1 half as long as its loop).
__device__ __forceinline__ float gelu_tanh(float x) {
    const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.0f * 1.4426950408889634f * u));
}
__device__ __forceinline__ float gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.7071067811865475f)); }

// Four consecutive outputs n .. n + 3 of token m: bias and the mode's elementwise work.
template <int MODE>
__device__ __forceinline__ void vit_store(const VitGemmArgs& g, int m, int n, const f32x4& acc) {
#pragma clang fp contract(off)
    const float4 bv = *(const float4*)(g.bias + n);
    float4 v = make_float4(acc[0] + bv.x, acc[1] + bv.y, acc[2] + bv.z, acc[3] + bv.w);
    const size_t o = (size_t)m * g.N + n;
    if constexpr (MODE == VG_F32) {
        *(float4*)(g.outf + o) = v;
    } else if constexpr (MODE == VG_F32_ADD) {
        float4 r = *(const float4*)(g.outf + o);
        r.x += v.x;
        r.y += v.y;
        r.z += v.z;
        r.w += v.w;
        *(float4*)(g.outf + o) = r;
    } else if constexpr (MODE == VG_F32_POS) {
        const float4 p = *(const float4*)(g.pos + o);
        *(float4*)(g.outf + o) = make_float4(v.x + p.x, v.y + p.y, v.z + p.z, v.w + p.w);
    } else {
        float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = MODE == VG_GELU_TANH ? gelu_tanh(e[i]) : gelu_erf(e[i]);
        const uint32_t h0 = f2h(e[0]), h1 = f2h(e[1]), h2 = f2h(e[2]), h3 = f2h(e[3]);
        *(uint2*)(g.outh + o) = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
    }
}

// C[m][n] = sum_k X[m][k] W[n][k] over fp16 X [M][K] and W [N][K].  Workgroup tile BN x BM
// (outputs x tokens), 4 waves in a WN x WM grid; each wave holds TN x TM 16 x 16 accumulators.
// W rows are the A operand and X rows the B operand of v_mfma_f32_16x16x32_f16, so lane l
// ends with C[m = l % 16][n = 4 (l / 16) + i], four consecutive outputs of one token.
//
// K runs in steps of 64 through a ring of S LDS stages filled by direct global-to-LDS loads
// (global_load_lds_dwordx4, 16 bytes a lane), S - 1 steps ahead of the products.  A stage
// holds 128-byte rows; the 16-byte chunk c of row r sits at chunk c ^ (r % 8), so the 16 rows
// of a fragment read spread over the banks.  Token rows past M read row M - 1 and are not
// stored.
//
// (The launch bound is twice the 256 threads that run: a wave then has at most 256 registers, all of
// them VGPRs.  With more, the compiler keeps the accumulators in AGPRs and moves them to and fro
// around every few products.)
template <int BN, int BM, int WN, int WM, int MODE, int S>
__global__ __launch_bounds__(512) void vit_gemm_kernel(VitGemmArgs g) {
#pragma clang fp contract(off)
    constexpr int TN = BN / WN / 16, TM = BM / WM / 16, BK = 64;
    constexpr int WLOADS = (BN + BM) / 8;  // 1 KiB wave loads per stage (8 rows each)
    constexpr int L = WLOADS / 4;          // per wave
    static_assert(WN * WM == 4 && TN >= 1 && TM >= 1 && WLOADS % 4 == 0 && S >= 2 && (S - 2) * L <= 63, "tile");
    static_assert(MODE != VG_QKV || (BN == 64 && WN == 1), "the RoPE pairs (d, d + 32) of a head stay in one lane");
    __shared__ __align__(1024) uint8_t ring[S][(BN + BM) * 128];
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, r16 = lane & 15, q4 = lane >> 4;
    const int wn = wave / WM, wm = wave % WM;
    const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM;
    const int K = g.K, nk = K / BK;
    // Lane l of wave load j (rows 8 j .. 8 j + 7 of the stage: W rows first, then X rows) lands at
    // row 8 j + l / 8, chunk l % 8, and reads source chunk (l % 8) ^ (l / 8).
    const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
    auto issue = [&](int kt) __attribute__((always_inline)) {
        uint8_t* st = ring[kt % S];
        const int k0 = kt * BK + 8 * lchunk;
#pragma unroll
        for (int u = 0; u < L; ++u) {
            const int j = wave + 4 * u, row = 8 * j + lrow;
            const uint16_t* src = row < BN ? g.W + (size_t)(n0 + row) * K + k0
                                           : g.X + (size_t)min(m0 + row - BN, g.M - 1) * K + k0;
            __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)(st + 1024 * j), 16, 0, 0);
        }
    };
    auto frag = [&](const uint8_t* st, int row, int chunk) __attribute__((always_inline)) {
        return *(const v8h*)(st + row * 128 + ((chunk ^ (row & 7)) << 4));
    };

    f32x4 acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < S - 1; ++p) issue(min(p, nk - 1));
    for (int kt = 0; kt < nk; ++kt) {
        // This wave's loads of step kt have landed once at most (S - 2) * L newer ones are
        // outstanding; after the barrier every wave's have, and the stage read in step kt - 1
        // is free (its reads completed before each wave's products of that step).
        dma_barrier<(S - 2) * L>();
        issue(min(kt + S - 1, nk - 1));  // past the end: a repeat into a stage no one reads again
        const uint8_t* st = ring[kt % S];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            v8h af[TN], bf[TM];
#pragma unroll
            for (int a = 0; a < TN; ++a) af[a] = frag(st, (wn * TN + a) * 16 + r16, 4 * ks + q4);
#pragma unroll
            for (int b = 0; b < TM; ++b) bf[b] = frag(st, BN + (wm * TM + b) * 16 + r16, 4 * ks + q4);
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[a], bf[b], acc[a][b], 0, 0, 0);
        }
    }
    __builtin_amdgcn_s_waitcnt(0);  // no load is in flight when the workgroup ends

#pragma unroll
    for (int b = 0; b < TM; ++b) {
        const int m = m0 + (wm * TM + b) * 16 + r16;
        if (m >= g.M) continue;
        if constexpr (MODE == VG_QKV) {
            // Head n0 / 64 of the fused rows: q heads 0-15, k heads 16-31, v heads 32-47.  Lane
            // holds dims d = 16 a + 4 q4 + i; pairs (d, d + 32) are accumulators a and a + 2.
            const int hh = blockIdx.x;
            float v[4][4];
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const float4 bv = *(const float4*)(g.bias + n0 + 16 * a + 4 * q4);
                v[a][0] = acc[a][b][0] + bv.x;
                v[a][1] = acc[a][b][1] + bv.y;
                v[a][2] = acc[a][b][2] + bv.z;
                v[a][3] = acc[a][b][3] + bv.w;
            }
            if (hh < 2 * VNH) {
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int d = 16 * a + 4 * q4 + i;
                        const float2 cs = *(const float2*)(g.rope + ((size_t)m * 32 + d) * 2);
                        const float x0 = v[a][i], x1 = v[a + 2][i];
                        v[a][i] = x0 * cs.x - x1 * cs.y;
                        v[a + 2][i] = x1 * cs.x + x0 * cs.y;
                    }
                uint16_t* dst = (hh < VNH ? g.q + (size_t)hh * g.ld * VHD : g.k + (size_t)(hh - VNH) * g.ld * VHD) +
                                (size_t)m * VHD;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const uint32_t h0 = f2h(v[a][0]), h1 = f2h(v[a][1]), h2 = f2h(v[a][2]), h3 = f2h(v[a][3]);
                    *(uint2*)(dst + 16 * a + 4 * q4) = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
                }
            } else {
                uint16_t* dst = g.vt + (size_t)(hh - 2 * VNH) * VHD * g.ld + m;
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int i = 0; i < 4; ++i) dst[(size_t)(16 * a + 4 * q4 + i) * g.ld] = f2h(v[a][i]);
            }
        } else {
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                const int n = n0 + (wn * TN + a) * 16 + 4 * q4;
                vit_store<MODE>(g, m, n, acc[a][b]);
            }
        }
    }
}

// The same product where K is long and there are more 32 x 64 tiles than CUs (fc2 and the mergers'
// first product; gemm_long): 64 outputs x 64 tokens per workgroup, 4 waves, each computing the whole
// tile over its own steps of K (step w, w + 4, ...) through an LDS ring of its own, so no wave waits
// for another before the end, where their sums meet in LDS.  LDS traffic bounds these products (with
// four waves sharing a stage as 32 x 32 quarters, 48 KiB a step at 128 bytes a clock): a wave's 64 x
// 64 tile reads each operand once, 32 KiB a step.  (The launch bound as above.)  At 960 patches fc2
// takes 19.0 us and a merger's first product 20.8 (with 32 x 64 tiles over shared stages 21.2 and
// 26.7).  Small tiles with shared stages stay better where K is short (proj 8.7 against 9.7, the patch
// embedding 9.4 against 9.9) or 64 x 64 tiles fill half of the chip (a merger's second product, 17.8
// against 18.5).
template <int MODE>
__global__ __launch_bounds__(512) void vit_deep_kernel(VitGemmArgs g) {
#pragma clang fp contract(off)
    static_assert(MODE != VG_QKV, "the rotation pairs of a head are not in one lane here");
    constexpr int KW = 4;
    __shared__ __align__(1024) uint8_t rings[KW][2][128 * 128];  // [wave][stage][64 W rows, 64 X rows][64 K]
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), r16 = lane & 15, q4 = lane >> 4;
    const int n0 = blockIdx.x * 64, m0 = blockIdx.y * 64, K = g.K, nk = K / 64;
    // As in vit_gemm_kernel: load j brings rows 8 j .. + 7, 16-byte chunk c of row r lands at c ^ (r % 8).
    const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
    auto issue = [&](int st, int kt) __attribute__((always_inline)) {
        const int k0 = kt * 64 + 8 * lchunk;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint16_t* src = j < 8 ? g.W + (size_t)(n0 + 8 * j + lrow) * K + k0
                                        : g.X + (size_t)min(m0 + 8 * (j - 8) + lrow, g.M - 1) * K + k0;
            __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)(rings[wave][st] + 1024 * j), 16, 0, 0);
        }
    };
    f32x4 acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // A step's two k-steps alternate between two register sets: while one is multiplied, the other's
    // operands are read.  Behind the first, the next step's stage has to have landed; behind the
    // second, the present stage is free for the step after that.
    struct Ops {
        v8h w[4], x[4];
    };
    auto read = [&](int st, int ks) __attribute__((always_inline)) {
        const uint8_t* s = rings[wave][st];
        Ops o;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int row = 16 * t + r16, at = row * 128 + (((4 * ks + q4) ^ (row & 7)) << 4);
            o.w[t] = *(const v8h*)(s + at);
            o.x[t] = *(const v8h*)(s + 64 * 128 + at);
        }
        return o;
    };
    auto mac = [&](const Ops& o) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.w[a], o.x[b], acc[a][b], 0, 0, 0);
    };
    constexpr int VM0 = (7 << 4) | (15 << 8), VM16 = VM0 | ((16 >> 4) << 14), LGKM0 = 15 | (7 << 4) | (3 << 14);
    if (wave < nk) {
        issue(0, wave);
        if (wave + KW < nk) {
            issue(1, wave + KW);
            __builtin_amdgcn_s_waitcnt(VM16);
        } else {
            __builtin_amdgcn_s_waitcnt(VM0);
        }
        asm volatile("" ::: "memory");
        Ops p0 = read(0, 0);
        for (int kt = wave, st = 0; kt < nk; kt += KW, st ^= 1) {
            const Ops p1 = read(st, 1);
            __builtin_amdgcn_sched_barrier(0);
            mac(p0);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(LGKM0);  // the stage has been read
            asm volatile("" ::: "memory");
            if (kt + 2 * KW < nk) {
                issue(st, kt + 2 * KW);
                __builtin_amdgcn_s_waitcnt(VM16);
            } else {
                __builtin_amdgcn_s_waitcnt(VM0);
            }
            asm volatile("" ::: "memory");
            p0 = read(st ^ 1, 0);  // (after the last step: a stage that is not used)
            __builtin_amdgcn_sched_barrier(0);
            mac(p1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // Wave w finishes output rows 16 w .. + 15 of the tile (blocks (w, 0 .. 3)), the sums in wave order.
    __syncthreads();
    f32x4* sums = (f32x4*)&rings[0][0][0];  // [wave][block][lane], 64 KiB
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) sums[(wave * 16 + 4 * a + b) * WAVE + lane] = acc[a][b];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        f32x4 y = sums[(4 * wave + b) * WAVE + lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) {
            const f32x4 o = sums[(w * 16 + 4 * wave + b) * WAVE + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] += o[e];
        }
        const int m = m0 + 16 * b + r16;
        if (m < g.M) vit_store<MODE>(g, m, n0 + 16 * wave + 4 * q4, y);
    }
}

// Bidirectional attention of one head over all patches (k_vit_attn, Shaders.swift:294-395),
// grid (ceil(np / 64), 16 heads), 4 PARTS waves.  Waves w, w + 4, .. own the same 16 queries,
// 64 x + 16 (w % 4) .. + 15 (lane l: query l % 16), and split the key blocks in PARTS parts, so
// the serial chain of block loads and softmax updates, which bounds the kernel (the products of
// 960 patches take ~3 us of it), is shorter by that factor.  Per block of 64 keys: S^T = K . Q^T on
// v_mfma_f32_16x16x32_f16 (lane: keys 16 j + 4 (l / 16) + i of sub-block j), in log2 units
// (log2(e) / 8, so that every exponential is one v_exp_f32); an online softmax per query column
// whose denominators stay per lane until the end; O^T += V^T . P^T on v_mfma_f32_16x16x16_f16 with
// the fp16 probabilities straight from the score registers and V^T read from LDS, rescaled only
// when some column's maximum moved.  The parts' (max, sum, O) are combined through LDS.  Keys past np are
// masked (their rows hold finite values; only the last block has any).  Two parts up to ten key blocks,
// where more waves cost more to start and to combine than they shorten (us, two / four parts: 4.7 /
// 6.0 for 64 patches, 5.4 / 5.9 for 256, 7.9 / 8.5 for 480, 9.2 / 10.2 for 640); four above (10.5 /
// 10.1 for 644, 10.7 / 10.2 for 768, 12.8 / 12.7 for 960).
constexpr int VA_ROW = 72, VA_TILE = 64 * VA_ROW;
constexpr size_t va_lds_bytes(int parts) { return (size_t)parts * 2 * 2 * VA_TILE * 2; }  // [part][K, V^T][buffer]
template <int VA_PARTS>
__global__ __launch_bounds__(256 * VA_PARTS) void vit_attention_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                             const uint16_t* __restrict__ vt, uint16_t* __restrict__ out,
                                                             int np, int ld) {
    // V^T rows with (row / 8) odd hold their 4-key chunks pairwise swapped (chunk c at c ^ 1): the
    // P.V reads of 16 rows x one chunk then cover all 32 banks.
    extern __shared__ __align__(16) uint16_t va_lds[];
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, r16 = lane & 15, q4 = lane >> 4;
    const int grp = wave >> 2, gt = tid & 255;
    uint16_t* kt = va_lds + (size_t)grp * 4 * VA_TILE;  // K of buffer 0, 1, then V^T of buffer 0, 1
    uint16_t* vtl = kt + 2 * VA_TILE;
    const int h = blockIdx.y;
    const int qt = blockIdx.x * 64 + (wave & 3) * 16 + r16;
    const uint16_t* qh = q + (size_t)h * ld * VHD;
    const uint16_t* kh = k + (size_t)h * ld * VHD;
    const uint16_t* vh = vt + (size_t)h * VHD * ld;
    const int qc = min(qt, np - 1);
    v8h qf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) qf[ks] = *(const v8h*)(qh + (size_t)qc * VHD + 32 * ks + 8 * q4);

    // Register-staged block loads by the 256 threads of a part: rows gt / 8 and 32 + gt / 8, columns
    // 8 (gt % 8) .. + 7.
    struct Block {
        uint4 k0, k1, v0, v1;
    };
    const int row = gt >> 3, col = (gt & 7) * 8;
    auto gload = [&](int blk) __attribute__((always_inline)) {
        const uint16_t* kp = kh + (size_t)(64 * blk + row) * VHD + col;
        const uint16_t* vp = vh + (size_t)row * ld + 64 * blk + col;
        return Block{*(const uint4*)kp, *(const uint4*)(kp + 32 * VHD), *(const uint4*)vp, *(const uint4*)(vp + (size_t)32 * ld)};
    };
    auto lstore = [&](int buf, const Block& x) __attribute__((always_inline)) {
        uint16_t* kd = kt + buf * VA_TILE + row * VA_ROW + col;
        uint16_t* vd = vtl + buf * VA_TILE + row * VA_ROW + col;
        const bool odd = (row >> 3) & 1;
        *(uint4*)kd = x.k0;
        *(uint4*)(kd + 32 * VA_ROW) = x.k1;
        *(uint4*)vd = odd ? make_uint4(x.v0.z, x.v0.w, x.v0.x, x.v0.y) : x.v0;
        *(uint4*)(vd + 32 * VA_ROW) = odd ? make_uint4(x.v1.z, x.v1.w, x.v1.x, x.v1.y) : x.v1;
    };

    const int nblk = (np + 63) / 64, nh = (nblk + VA_PARTS - 1) / VA_PARTS;
    const int b0 = min(nblk, grp * nh), bend = min(nblk, b0 + nh);  // this part's blocks [b0, bend), maybe none
    float m_run = -__builtin_inff(), l_run = 0.f;  // maximum of query r16; this lane's share of its denominator
    f32x4 O[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    lstore(0, gload(min(b0, nblk - 1)));
    __syncthreads();
    for (int it = 0; it < nh; ++it) {
        const int blk = b0 + it, buf = it & 1;
        const Block next = gload(min(blk + 1, nblk - 1));  // a valid block either way
        {  // (no branch around it: a step past the part's blocks masks every key)
            const int lim = blk < bend ? np : 0;
            const uint16_t* Ks = kt + buf * VA_TILE;
            const uint16_t* Vs = vtl + buf * VA_TILE;
            f32x4 S[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    const v8h kf = *(const v8h*)&Ks[(16 * j + r16) * VA_ROW + 32 * ks + 8 * q4];
                    S[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[ks], S[j], 0, 0, 0);
                }
            }
            // The V operands, read behind the softmax.
            v4h vf[4][4];
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int j = 0; j < 4; ++j) vf[dt][j] = *(const v4h*)&Vs[(16 * dt + r16) * VA_ROW + 4 * ((4 * j + q4) ^ (r16 >> 3))];
            if (64 * blk + 64 > lim) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (64 * blk + 16 * j + 4 * q4 + i >= lim) S[j][i] = -__builtin_inff();
            }
            float mb = -__builtin_inff();
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) mb = fmaxf(mb, S[j][i]);
            constexpr float SC = 0.125f * 1.4426950408889634f;
            const float m_new = fmaxf(m_run, max_x4(mb) * SC);
            const float m_use = m_new == -__builtin_inff() ? 0.f : m_new;  // a part without a block yet
            const float corr = __builtin_amdgcn_exp2f(m_run - m_use);
            float ls = 0.f;
            v4h P[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = __builtin_amdgcn_exp2f(S[j][i] * SC - m_use);
                    ls += p;
                    P[j][i] = (_Float16)p;
                }
            if (__builtin_amdgcn_ballot_w64(m_new != m_run)) {
                l_run *= corr;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) O[dt][i] *= corr;
            }
            l_run += ls;
            m_run = m_new;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) O[dt] = __builtin_amdgcn_mfma_f32_16x16x16f16(vf[dt][j], P[j], O[dt], 0, 0, 0);
        }
        lstore(buf ^ 1, next);  // the last fills an idle buffer
        __syncthreads();
    }
    l_run = sum_x4(l_run);
    // Combine the parts: the states of parts 1 .. 3 go through LDS (every tile read is done) as
    // [part - 1][O tile, then (max, sum)][256 lanes], and part 0 finishes.
    f32x4* xo = (f32x4*)va_lds;
    float2* xm = (float2*)(xo + (size_t)(VA_PARTS - 1) * 4 * 256);
    if (grp > 0) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) xo[((grp - 1) * 4 + dt) * 256 + gt] = O[dt];
        xm[(grp - 1) * 256 + gt] = make_float2(m_run, l_run);
    }
    __syncthreads();
    if (grp == 0 && qt < np) {
        float2 ml[VA_PARTS - 1];
        float m = m_run;  // finite: the first part is never empty
#pragma unroll
        for (int p = 0; p < VA_PARTS - 1; ++p) {
            ml[p] = xm[p * 256 + gt];
            m = fmaxf(m, ml[p].x);
        }
        const float f0 = __builtin_amdgcn_exp2f(m_run - m);
        float l = l_run * f0;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) O[dt][i] *= f0;
#pragma unroll
        for (int p = 0; p < VA_PARTS - 1; ++p) {
            const float f = __builtin_amdgcn_exp2f(ml[p].x - m);  // 0 for a part without blocks
            l = fmaf(ml[p].y, f, l);
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const f32x4 o = xo[(p * 4 + dt) * 256 + gt];
#pragma unroll
                for (int i = 0; i < 4; ++i) O[dt][i] = fmaf(o[i], f, O[dt][i]);
            }
        }
        const float inv = 1.0f / l;
        uint16_t* dst = out + (size_t)qt * VH + h * VHD;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            const uint32_t h0 = f2h(O[dt][0] * inv), h1 = f2h(O[dt][1] * inv), h2 = f2h(O[dt][2] * inv), h3 = f2h(O[dt][3] * inv);
            *(uint2*)(dst + 16 * dt + 4 * q4) = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
        }
    }
}

int attention_parts(int np) { return np <= 640 ? 2 : 4; }

hipError_t attention_setup(int np) {
    const int parts = attention_parts(np);
    return hipFuncSetAttribute(parts == 2 ? (const void*)vit_attention_kernel<2> : (const void*)vit_attention_kernel<4>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)va_lds_bytes(parts));
}

hipError_t attention(const VitBuffers& b, int np, hipStream_t s) {
    const int parts = attention_parts(np);
    hipLaunchKernelGGL(parts == 2 ? vit_attention_kernel<2> : vit_attention_kernel<4>, dim3((np + 63) / 64, VNH),
                       dim3(256 * parts), va_lds_bytes(parts), s, b.q, b.k, b.vt, b.attn, np, NPATCH_MAX);
    return hipGetLastError();
}

template <int BN, int BM, int WN, int WM, int MODE, int S>
hipError_t gemm(const VitGemmArgs& g, hipStream_t s) {
    if (g.N % BN || g.K % 64 || g.M < 1) return hipErrorInvalidValue;
    const dim3 grid(g.N / BN, (g.M + BM - 1) / BM);
    hipLaunchKernelGGL((vit_gemm_kernel<BN, BM, WN, WM, MODE, S>), grid, dim3(256), 0, s, g);
    return hipGetLastError();
}

template <int MODE>
hipError_t gemm_deep(const VitGemmArgs& g, hipStream_t s) {
    if (g.N % 64 || g.K % 64 || g.M < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(vit_deep_kernel<MODE>, dim3(g.N / 64, (g.M + 63) / 64), dim3(256), 0, s, g);
    return hipGetLastError();
}

// A product over a long K: 32 x 64 tiles over shared stages while every tile has a CU to itself, more
// tiles as 64 x 64 ones with private rings.  (us, 32 x 64 / 64 x 64: fc2 17.4 / 21.5 for 64 patches,
// 17.4 / 18.9 for 256, 17.7 / 18.5 for 512, 18.1 / 17.4 for 516, 20.0 / 18.4 for 640; a merger's first
// product 19.2 / 23.2 for 256 patches, 19.3 / 22.7 for 512, 19.5 / 18.9 for 516, 20.7 / 20.2 for 640.)
template <int MODE>
hipError_t gemm_long(const VitGemmArgs& g, hipStream_t s) {
    return g.N / 32 * ((g.M + 63) / 64) <= 256 ? gemm<32, 64, 2, 2, MODE, 4>(g, s) : gemm_deep<MODE>(g, s);
}

template <int N>
hipError_t layernorm(const float* x, const float* w, const float* b, uint16_t* out, int rows, hipStream_t s) {
    hipLaunchKernelGGL((vit_layernorm_kernel<N>), dim3((rows + 3) / 4), dim3(256), 0, s, x, w, b, out, rows);
    return hipGetLastError();
}

#define VCK(x)                            \
    do {                                  \
        const hipError_t e_ = (x);        \
        if (e_ != hipSuccess) return e_;  \
    } while (0)

hipError_t merger(const VitMerger& mg, const uint16_t* xn, int nvis, uint16_t* hbuf, float* out, hipStream_t s) {
    VitGemmArgs g{};
    g.X = xn;
    g.W = mg.fc1w;
    g.bias = mg.fc1b;
    g.outh = hbuf;
    g.M = nvis;
    g.N = MH;
    g.K = MH;
    VCK((gemm_long<VG_GELU_ERF>(g, s)));
    g = VitGemmArgs{};
    g.X = hbuf;
    g.W = mg.fc2w;
    g.bias = mg.fc2b;
    g.outf = out;
    g.M = nvis;
    g.N = H;
    g.K = MH;
    return gemm<32, 32, 2, 2, VG_F32, 4>(g, s);
}

}  // namespace

hipError_t launch_vision(const VitWeights& w, const VitBuffers& b, int gh, int gw, hipStream_t s) {
    const int np = gh * gw, nvis = np / 4;
    if (gh < 2 || gw < 2 || gh % 2 || gw % 2 || np > NPATCH_MAX) return hipErrorInvalidValue;
    VCK(attention_setup(np));
    hipLaunchKernelGGL(vit_patchify_kernel, dim3(np), dim3(256), 0, s, b.rgb, b.patches, gh, gw);
    VCK(hipGetLastError());
    VitGemmArgs g{};
    g.X = b.patches;
    g.W = w.patch_w;
    g.bias = w.patch_b;
    g.outf = b.x;
    g.pos = b.pos;
    g.M = np;
    g.N = VH;
    g.K = VPATCH;
    VCK((gemm<32, 64, 2, 2, VG_F32_POS, 4>(g, s)));
    int ds = 0;
    for (int l = 0; l < VLAYERS; ++l) {
        const VitBlock& L = w.blk[l];
        VCK(layernorm<VH>(b.x, L.n1w, L.n1b, b.xn, np, s));
        g = VitGemmArgs{};
        g.X = b.xn;
        g.W = L.qkvw;
        g.bias = L.qkvb;
        g.rope = b.rope;
        g.q = b.q;
        g.k = b.k;
        g.vt = b.vt;
        g.ld = NPATCH_MAX;
        g.M = np;
        g.N = VQKV;
        g.K = VH;
        // A head's 64 outputs x 64 tokens while these tiles all run at once, two a CU (640 patches), x
        // 128 above (us, x 64 / x 128: 8.7 / 12.0 for 256 patches, 11.3 / 12.2 for 480, 11.7 / 12.2 for
        // 640, 15.6 / 13.0 for 644, 17.0 / 14.8 for 960; x 192 as x 128 there, x 256 a fifth slower).
        if (VQKV / 64 * ((np + 63) / 64) <= 512)
            VCK((gemm<64, 64, 1, 4, VG_QKV, 4>(g, s)));
        else
            VCK((gemm<64, 128, 1, 4, VG_QKV, 3>(g, s)));
        VCK(attention(b, np, s));
        g = VitGemmArgs{};
        g.X = b.attn;
        g.W = L.projw;
        g.bias = L.projb;
        g.outf = b.x;
        g.M = np;
        g.N = VH;
        g.K = VH;
        VCK((gemm<32, 64, 2, 2, VG_F32_ADD, 4>(g, s)));
        VCK(layernorm<VH>(b.x, L.n2w, L.n2b, b.xn, np, s));
        g = VitGemmArgs{};
        g.X = b.xn;
        g.W = L.fc1w;
        g.bias = L.fc1b;
        g.outh = b.h;
        g.M = np;
        g.N = VFF;
        g.K = VH;
        // (16.2 us; 19.8 with the accumulators in AGPRs; 128 x 128 tiles, one a CU, 18.9)
        VCK((gemm<128, 64, 2, 2, VG_GELU_TANH, 3>(g, s)));
        g = VitGemmArgs{};
        g.X = b.h;
        g.W = L.fc2w;
        g.bias = L.fc2b;
        g.outf = b.x;
        g.M = np;
        g.N = VH;
        g.K = VFF;
        VCK((gemm_long<VG_F32_ADD>(g, s)));
        if (l == 5 || l == 11 || l == 17) {
            // DeepStack merger: LayerNorm over each 2 x 2 block's 4096 values (Engine.swift:420-447).
            VCK(layernorm<MH>(b.x, w.mg[ds].nw, w.mg[ds].nb, b.xn, nvis, s));
            VCK(merger(w.mg[ds], b.xn, nvis, b.h, b.ds[ds], s));
            ++ds;
        }
    }
    // Final merger: LayerNorm per patch, then 2 x 2 blocks as rows of 4096 (Engine.swift:450-472).
    VCK(layernorm<VH>(b.x, w.mg[3].nw, w.mg[3].nb, b.xn, np, s));
    return merger(w.mg[3], b.xn, nvis, b.h, b.pooler, s);
}

}  // namespace icua
