// Gated Delta Net (Qwen 3.5 / 3.6 / 3.8 linear-attention layers) -- decode step and sequential prefill.
//
// One kernel per layer does everything between the input projection GEMV/GEMM and the output
// projection (reference: ops/gdn/layer.rs:122-182 = ~12 candle launches for the conv alone,
// ops/gdn/conv.rs:63-73):
//   causal depthwise conv1d (k = 4) + SiLU with rolling state        ops/gdn/conv.rs:23-101
//   split q|k|v, key-head -> value-head expansion (HF "Interleaved")  ops/gdn/layer.rs:184-238
//   L2-norm(q), L2-norm(k) (eps 1e-6), q * 1/sqrt(K)                   ops/gdn/backend.rs:26-56,100-108
//   beta = sigmoid(b), g = -exp(A_log) * softplus(a + dt_bias)         ops/gdn/backend.rs:197-211
//   S *= exp(g); kv = S^T k; delta = (v - kv) beta; S += k (x) delta; y = S^T q   backend.rs:90-156,
//                                                                      kernels/cuda/gdn.cu:83-124
//   RmsNormGated: rms_norm(y, w) * silu(z)  (plain weight)             ops/gdn/norm.rs:39-45
// State is f32 (ops/gdn/cache.rs:12-13).  HBM-bound at decode: 2 * K * V * 4 B per value head per
// token (read + write of the state), 0.5 flop/byte.
//
// Layout: one block per value head, one thread per state COLUMN v (V = 128 threads); the column's
// K = 128 state values live in registers across the two passes (kv needs all of k before the
// update); S[k][v] is stored [K][V] so a wave reads/writes 256 contiguous bytes per k.
// Conv state is double-buffered by position parity so that the blocks of one key-head group (which
// share q/k channels) never read a window another block is rolling.
#include <cstdlib>

#include "dev_common.h"
#include "kernels.h"

namespace cm {

// a gated, normalised value of a prompt row: f32, or the two bfloat16 terms that the projection behind multiplies (a launch that split the f32 rows was 6.7 us
// a layer of 2048 tokens and 2048 values; the stores of the terms in their place cost 1.2)
__device__ __forceinline__ void gdn_put(const GdnArgs& a, size_t at, float v) {
    if (a.out_hi == nullptr) { a.out[at] = v; return; }
    const uint16_t h = f32_to_bf16(v);
    a.out_hi[at] = h;
    if (a.out_lo != nullptr) a.out_lo[at] = f32_to_bf16(v - bf16_to_f32(h));
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }

// grid = NV value heads, block = 128 threads.  Processes S tokens sequentially (S = 1 at decode).
__global__ __launch_bounds__(128) void gdn_kernel(GdnArgs a) {
    constexpr int K = 128, V = 128, KER = 4;
    __shared__ float qs[K], ks[K];
    __shared__ float red[8];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bq = blockIdx.y;                                 // sequence of a batched decode step (0 otherwise)
    const int nk = a.NV / a.vpg;
    const int kh = a.chunked ? h % nk : h / a.vpg;             // Interleaved (HF): h / vpg; Chunked (GGUF): h % NK
    const int cq = kh * K + tid, ck = a.key_dim + kh * K + tid, cv = 2 * a.key_dim + h * V + tid;
    const int conv_dim = 2 * a.key_dim + a.NV * V;
    const int proj_stride = a.proj_stride;
    const bool writer = a.chunked ? (h < nk) : (h % a.vpg) == 0;   // one block per key head rolls the q/k windows

    // conv weights of my three channels, state column in registers
    float wq[KER], wk[KER], wv[KER];
#pragma unroll
    for (int j = 0; j < KER; ++j) { wq[j] = a.conv_w[cq * KER + j]; wk[j] = a.conv_w[ck * KER + j]; wv[j] = a.conv_w[cv * KER + j]; }
    const int start_pos = a.st ? a.st[bq].pos : a.start_pos;
    const int slot = a.st ? a.st[bq].slot : a.slot;
    float* conv_state = a.conv_pool + ((size_t)slot * a.gdn_layers + a.layer_idx) * 2 * conv_dim * (KER - 1);
    const int par_in = start_pos & 1;
    const float* cs_in = conv_state + (size_t)par_in * conv_dim * (KER - 1);
    float hq[KER - 1], hk[KER - 1], hv[KER - 1];
#pragma unroll
    for (int j = 0; j < KER - 1; ++j) {
        hq[j] = cs_in[cq * (KER - 1) + j]; hk[j] = cs_in[ck * (KER - 1) + j]; hv[j] = cs_in[cv * (KER - 1) + j];
    }
    float* Sg = a.state_pool + (((size_t)slot * a.gdn_layers + a.layer_idx) * a.NV + h) * K * V;
    float S[K];
#pragma unroll
    for (int k = 0; k < K; ++k) S[k] = Sg[k * V + tid];
    const float neg_exp_a = -expf(a.A_log[h]);
    const float dtb = a.dt_bias[h];
    const float gw = a.gnorm_w[tid];
    const float qscale = 0.08838834764831845f;                 // 1/sqrt(128)

    for (int t = 0; t < a.S; ++t) {
        const float* pr = a.proj + (size_t)bq * a.batch_proj_stride + (size_t)t * proj_stride;
        // ---- conv + SiLU; roll the windows ----
        const float xq = pr[cq], xk = pr[ck], xv = pr[cv];
        float q = hq[0] * wq[0] + hq[1] * wq[1] + hq[2] * wq[2] + xq * wq[3];
        float k = hk[0] * wk[0] + hk[1] * wk[1] + hk[2] * wk[2] + xk * wk[3];
        float v = hv[0] * wv[0] + hv[1] * wv[1] + hv[2] * wv[2] + xv * wv[3];
        hq[0] = hq[1]; hq[1] = hq[2]; hq[2] = xq;
        hk[0] = hk[1]; hk[1] = hk[2]; hk[2] = xk;
        hv[0] = hv[1]; hv[1] = hv[2]; hv[2] = xv;
        q = silu_f(q); k = silu_f(k); v = silu_f(v);
        // ---- L2 norms over the key head (128 threads = 2 waves) ----
        float sq = wave_sum(q * q), sk = wave_sum(k * k);
        __syncthreads();                                        // previous iteration done with qs/ks/red
        if (lane == 0) { red[wave] = sq; red[2 + wave] = sk; }
        __syncthreads();
        q = q / sqrtf(red[0] + red[1] + 1e-6f) * qscale;
        k = k / sqrtf(red[2] + red[3] + 1e-6f);
        qs[tid] = q; ks[tid] = k;
        // ---- gates ----
        const float beta = 1.0f / (1.0f + expf(-pr[conv_dim + a.NV * V + h]));
        const float av = pr[conv_dim + a.NV * V + a.NV + h] + dtb;
        const float g = neg_exp_a * logf(1.0f + expf(av));
        const float decay = expf(g);
        __syncthreads();
        // ---- recurrence on my column ----
        float kv4[4] = {0.f, 0.f, 0.f, 0.f};                     // 4 independent chains instead of one 128-deep dependent one
#pragma unroll
        for (int kk = 0; kk < K; ++kk) { S[kk] *= decay; kv4[kk & 3] += S[kk] * ks[kk]; }
        const float kv = (kv4[0] + kv4[1]) + (kv4[2] + kv4[3]);
        const float delta = (v - kv) * beta;
        float y4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < K; ++kk) { S[kk] += ks[kk] * delta; y4[kk & 3] += S[kk] * qs[kk]; }
        const float y = (y4[0] + y4[1]) + (y4[2] + y4[3]);
        // ---- gated RMSNorm over the value head ----
        const float sy = wave_sum(y * y);
        if (lane == 0) red[4 + wave] = sy;
        __syncthreads();
        const float rms = 1.0f / sqrtf((red[4] + red[5]) / (float)V + a.eps);
        const float z = pr[conv_dim + h * V + tid];
        gdn_put(a, (size_t)bq * a.batch_out_stride + (size_t)t * a.out_stride + h * V + tid, y * rms * gw * silu_f(z));
    }
    // ---- write back state and conv windows (other parity buffer) ----
#pragma unroll
    for (int k = 0; k < K; ++k) Sg[k * V + tid] = S[k];
    float* cs_out = conv_state + (size_t)((start_pos + a.S) & 1) * conv_dim * (KER - 1);
#pragma unroll
    for (int j = 0; j < KER - 1; ++j) {
        if (writer) { cs_out[cq * (KER - 1) + j] = hq[j]; cs_out[ck * (KER - 1) + j] = hk[j]; }
        cs_out[cv * (KER - 1) + j] = hv[j];
    }
}

// ---------------------------------------------------------------------------------------------------------
// Decode step on NV x 4 workgroups.  The fused kernel above reads and writes a value head's 64 KiB state from ONE
// workgroup: 16 (Qwen3.5-0.8B) ... 48 (Qwen3.8-27B) of 256 CUs stream the only HBM-bound bytes of the layer (measured
// 8.7 us per layer on the 0.8B model = 0.24 TB/s).  Here a value head is four workgroups of 32 state columns each
// (one column = 256 threads / 32: 8 k-slices of 16 state values per thread; a wave reads 2 x 128 contiguous bytes per k).
// Everything per token is recomputed by each of them (conv + SiLU + L2 norm of the key head's q / k: 256 channels), the
// recurrence runs on the workgroup's own columns, and the gated RMSNorm -- which needs the head's 128 y values -- is done
// by the LAST of the four workgroups to arrive: raw y and the partial sums of squares go out as write-through (sc1)
// stores, every wave drains them, one lane takes a ticket; the workgroup that draws 3 reads them back with sc1 loads
// (no fences, no polling: MI355X_MICROARCH.md "handoff-flag", Guideline 16 R1).  Same arithmetic as gdn_kernel except
// for the association of the two 128-term sums over k (8 partial sums of 16 terms).
// ---------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gdn_decode_kernel(GdnArgs a) {
    constexpr int K = 128, V = 128, KER = 4, CB = 32, KS = 8, KP = K / KS;
    __shared__ float qs[K], ks_[K], vs[CB];
    __shared__ float red[8];
    __shared__ float part[KS][CB];
    __shared__ float bd[2];
    __shared__ int last_flag;
    const int h = blockIdx.x, cb = blockIdx.y, bq = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = tid & (CB - 1), ksl = tid / CB;              // column inside the block, k-slice
    const int v = cb * CB + c;
    const int nk = a.NV / a.vpg;
    const int kh = a.chunked ? h % nk : h / a.vpg;
    const int conv_dim = 2 * a.key_dim + a.NV * V;
    const bool qk_writer = cb == 0 && (a.chunked ? (h < nk) : (h % a.vpg) == 0);
    const int start_pos = a.st[bq].pos, slot = a.st[bq].slot;
    float* conv_state = a.conv_pool + ((size_t)slot * a.gdn_layers + a.layer_idx) * 2 * conv_dim * (KER - 1);
    const float* cs_in = conv_state + (size_t)(start_pos & 1) * conv_dim * (KER - 1);
    float* cs_out = conv_state + (size_t)((start_pos + 1) & 1) * conv_dim * (KER - 1);
    const float* pr = a.proj + (size_t)bq * a.batch_proj_stride;
    // state slice: requested first (the only HBM-bound bytes)
    float* Sg = a.state_pool + (((size_t)slot * a.gdn_layers + a.layer_idx) * a.NV + h) * K * V;
    float S[KP];
#pragma unroll
    for (int k = 0; k < KP; ++k) S[k] = __builtin_nontemporal_load(&Sg[(ksl * KP + k) * V + v]);
    const float A_log = a.A_log[h], dt_bias = a.dt_bias[h];
    float own;                                                 // this thread's q or k channel
    // conv + SiLU: threads 0..127 the q channel, 128..255 the k channel of the key head; threads < 32 also this block's v columns
    {
        const int ch = (tid < K ? kh * K + tid : a.key_dim + kh * K + (tid - K));
        const float w0 = a.conv_w[ch * KER], w1 = a.conv_w[ch * KER + 1], w2 = a.conv_w[ch * KER + 2], w3 = a.conv_w[ch * KER + 3];
        const float h0 = cs_in[ch * (KER - 1)], h1 = cs_in[ch * (KER - 1) + 1], h2 = cs_in[ch * (KER - 1) + 2];
        const float x = pr[ch];
        const float y = silu_f(h0 * w0 + h1 * w1 + h2 * w2 + x * w3);
        if (qk_writer) { cs_out[ch * (KER - 1)] = h1; cs_out[ch * (KER - 1) + 1] = h2; cs_out[ch * (KER - 1) + 2] = x; }
        const float ss = wave_sum(y * y);                      // waves 0,1 = q; 2,3 = k
        if (lane == 0) red[wave] = ss;
        own = y;
        if (tid < CB) {
            const int cv = 2 * a.key_dim + h * V + v;          // v == cb * CB + tid here
            const float u0 = a.conv_w[cv * KER], u1 = a.conv_w[cv * KER + 1], u2 = a.conv_w[cv * KER + 2], u3 = a.conv_w[cv * KER + 3];
            const float g0 = cs_in[cv * (KER - 1)], g1 = cs_in[cv * (KER - 1) + 1], g2 = cs_in[cv * (KER - 1) + 2];
            const float xv = pr[cv];
            vs[tid] = silu_f(g0 * u0 + g1 * u1 + g2 * u2 + xv * u3);
            cs_out[cv * (KER - 1)] = g1; cs_out[cv * (KER - 1) + 1] = g2; cs_out[cv * (KER - 1) + 2] = xv;
        }
        if (a.ba_w == nullptr && tid == 192) {                 // (not the wave with the v columns)
            const float beta = 1.0f / (1.0f + expf(-pr[conv_dim + a.NV * V + h]));
            const float av = pr[conv_dim + a.NV * V + a.NV + h] + dt_bias;
            bd[0] = beta;
            bd[1] = expf(-expf(A_log) * logf(1.0f + expf(av)));
        }
    }
    if (a.ba_w != nullptr) {
        // the head's b and a: two dot products of RMSNorm(x) * w with bf16 rows (the whole workgroup; the norm's scale is factored out)
        const float* xr = a.ba_x + (size_t)bq * a.ba_H;
        const uint16_t* wb = a.ba_w + (size_t)h * a.ba_H;
        const uint16_t* wa = a.ba_w + (size_t)(a.NV + h) * a.ba_H;
        float s2 = 0.f, sb = 0.f, sa = 0.f;
        for (int i0 = tid * 4; i0 < a.ba_H; i0 += 4096) {          // (four chunks' loads together: the sums keep their order)
            f32x4 xv4[4], nv4[4]; u32x2 pb4[4], pa4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = i0 + 1024 * j < a.ba_H ? i0 + 1024 * j : i0;
                xv4[j] = *(const f32x4*)(xr + i); nv4[j] = *(const f32x4*)(a.ba_nw + i);
                pb4[j] = *(const u32x2*)(wb + i); pa4[j] = *(const u32x2*)(wa + i);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (i0 + 1024 * j >= a.ba_H) break;
                const f32x4 xv = xv4[j], nv = nv4[j];
                const u32x2 pb = pb4[j], pa = pa4[j];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float xn = xv[e] * nv[e];
                    const float fb = bf16_to_f32((uint16_t)((pb[e >> 1] >> (16 * (e & 1))) & 0xFFFFu));
                    const float fa = bf16_to_f32((uint16_t)((pa[e >> 1] >> (16 * (e & 1))) & 0xFFFFu));
                    s2 = fmaf(xv[e], xv[e], s2); sb = fmaf(xn, fb, sb); sa = fmaf(xn, fa, sa);
                }
            }
        }
        __shared__ float bared[3][4];
        const float t2 = wave_sum(s2), tb = wave_sum(sb), ta = wave_sum(sa);
        __syncthreads();                                           // (red[] of the q / k norms is written above: separate array, but order the phases)
        if (lane == 0) { bared[0][wave] = t2; bared[1][wave] = tb; bared[2][wave] = ta; }
        __syncthreads();
        if (tid == 0) {
            const float rr = 1.0f / sqrtf(((bared[0][0] + bared[0][1]) + (bared[0][2] + bared[0][3])) / (float)a.ba_H + a.eps);
            const float bv = rr * ((bared[1][0] + bared[1][1]) + (bared[1][2] + bared[1][3]));
            const float av = rr * ((bared[2][0] + bared[2][1]) + (bared[2][2] + bared[2][3])) + dt_bias;
            bd[0] = 1.0f / (1.0f + expf(-bv));
            bd[1] = expf(-expf(A_log) * logf(1.0f + expf(av)));
        }
    }
    __syncthreads();
    // every channel is divided by its norm once, not by each of the 32 columns that read it (32 divisions a thread, and
    // the gates' logarithm in the wave that has the value columns too: 16 heads, 6.1 -> 4.7 us; what is left is three round trips to memory)
    if (tid < K) qs[tid] = own / sqrtf(red[0] + red[1] + 1e-6f) * 0.08838834764831845f;       // 1/sqrt(128)
    else ks_[tid - K] = own / sqrtf(red[2] + red[3] + 1e-6f);
    __syncthreads();
    const float beta = bd[0], decay = bd[1];
    float kf[KP], qf[KP];
#pragma unroll
    for (int k = 0; k < KP; ++k) { kf[k] = ks_[ksl * KP + k]; qf[k] = qs[ksl * KP + k]; }
    // ---- recurrence on this thread's 16 state values of column v ----
    float kv2[2] = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KP; ++k) { S[k] *= decay; kv2[k & 1] += S[k] * kf[k]; }
    part[ksl][c] = kv2[0] + kv2[1];
    __syncthreads();
    float kv = 0.f;
#pragma unroll
    for (int j = 0; j < KS; ++j) kv += part[j][c];
    const float delta = (vs[c] - kv) * beta;
    float y2[2] = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KP; ++k) { S[k] += kf[k] * delta; y2[k & 1] += S[k] * qf[k]; }
#pragma unroll
    for (int k = 0; k < KP; ++k) __builtin_nontemporal_store(S[k], &Sg[(ksl * KP + k) * V + v]);
    __syncthreads();                                           // everyone has read part[][] (kv)
    part[ksl][c] = y2[0] + y2[1];
    __syncthreads();
    if (a.defer_norm) {          // single-sequence decode: the out_proj GEMV normalises while it stages x (PRO_GDNNORM)
        if (tid < CB) {
            float y = 0.f;
#pragma unroll
            for (int j = 0; j < KS; ++j) y += part[j][tid];
            a.out[(size_t)bq * a.batch_out_stride + h * V + cb * CB + tid] = y;
        }
        return;
    }
    // ---- raw y of the block's 32 columns + partial sum of squares -> write-through; ticket; last arriver normalises ----
    float* yraw = a.gdn_scratch + ((size_t)bq * a.NV + h) * (V + 4);
    int* ticket = a.gdn_ticket + (size_t)bq * a.NV + h;
    if (tid < CB) {
        float y = 0.f;
#pragma unroll
        for (int j = 0; j < KS; ++j) y += part[j][tid];
        __hip_atomic_store(&yraw[cb * CB + tid], y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const float sy = group_sum(fmaf(y, y, lane_xor<16>(y * y)), 16);      // (written out: the first sum takes its own square unrounded)
        if (tid == 0) __hip_atomic_store(&yraw[V + cb], sy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // every storing wave drains its write-through stores
    __syncthreads();
    if (tid == 0) last_flag = (atomicAdd(ticket, 1) == (int)gridDim.y - 1) ? 1 : 0;
    __syncthreads();
    if (!last_flag) return;
    if (tid < V) {
        const float y = __hip_atomic_load(&yraw[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        float tot = 0.f;
        for (int j = 0; j < (int)gridDim.y; ++j) tot += __hip_atomic_load(&yraw[V + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const float rms = 1.0f / sqrtf(tot / (float)V + a.eps);
        const float z = pr[conv_dim + h * V + tid];
        a.out[(size_t)bq * a.batch_out_stride + h * V + tid] = y * rms * a.gnorm_w[tid] * silu_f(z);
    }
    if (tid == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);     // next launch starts from 0
}

// ---------------------------------------------------------------------------------------------------------
// Prefill in three passes.  The fused kernel above walks a prompt with 4 barriers, two block reductions and a handful
// of transcendental functions per token on ONE block per value head (~5 us per token and layer).  Everything except
// the state recurrence is independent across tokens, so:
//   gdn_pre_kernel  (a wave per head and 4 or 8 tokens): conv + SiLU, L2 norms, q scale, beta, exp(g)  -> q^ k^ v beta decay per token
//   gdn_scan_kernel (grid NV x 4): the recurrence only; 16 lanes share a state column (8 of the 128 k each, partial
//                   sums folded with one DPP row reduction), q^ / k^ of 8 tokens staged per barrier
//   gdn_post_kernel (grid S x NV): gated RMSNorm of the raw y rows in place
// Same per-token arithmetic as the fused kernel except for the association of the two 128-term sums over k.
// ---------------------------------------------------------------------------------------------------------
// A wave takes one head (q, k or v; lane l its channels 2 l, 2 l + 1) over PT tokens: the convolution's window rolls in registers, a row is read
// once instead of four times, norms need no other wave.  Bound by its traffic (a workgroup per token and head was bound by the 65 536 workgroups of a
// 2048-token pass: mean per launch of a 4165-token prompt 31.7 -> 20.2 us).  The rolling window that the next call reads is written by the wave that read
// the one of this call: both may be the same memory.
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int PT>
__global__ __launch_bounds__(256) void gdn_pre_kernel(GdnArgs a) {
    constexpr int K = 128, KER = 4;
    static_assert(PT >= KER - 1, "only the wave of token 0 reads the window of the call before");
    const int lane = threadIdx.x & 63, item = (int)blockIdx.y * 4 + ((int)threadIdx.x >> 6), t0 = (int)blockIdx.x * PT;
    const int nk = a.NV / a.vpg;
    if (item >= 2 * nk + a.NV) return;
    const int conv_dim = 2 * a.key_dim + a.NV * K;
    const int c = item * K + 2 * lane;                   // channels: q heads, k heads, v heads
    const float* conv_state = a.conv_pool + ((size_t)a.slot * a.gdn_layers + a.layer_idx) * 2 * conv_dim * (KER - 1);
    const float* cs_in = conv_state + (size_t)(a.start_pos & 1) * conv_dim * (KER - 1);
    const float* pc = a.proj + c;
    f32x2 x[KER - 1 + PT];                           // inputs at tokens t0 - 3 ...
#pragma unroll
    for (int i = 0; i < KER - 1 + PT; ++i) x[i] = *(const f32x2*)(pc + (size_t)min(max(t0 + i - (KER - 1), 0), a.S - 1) * a.proj_stride);
    const f32x4 w0 = *(const f32x4*)(a.conv_w + (size_t)c * KER), w1 = *(const f32x4*)(a.conv_w + (size_t)(c + 1) * KER);
    if (t0 == 0) {
#pragma unroll
        for (int i = 0; i < KER - 1; ++i) x[i] = (f32x2){cs_in[c * (KER - 1) + i], cs_in[(c + 1) * (KER - 1) + i]};
        float* cs_out = a.conv_pool + ((size_t)a.slot * a.gdn_layers + a.layer_idx) * 2 * conv_dim * (KER - 1) +
                        (size_t)((a.start_pos + a.S) & 1) * conv_dim * (KER - 1);
#pragma unroll
        for (int i = 0; i < KER - 1; ++i) {              // (prompts of 16 tokens or more: the window lies in this pass)
            const f32x2 v = *(const f32x2*)(pc + (size_t)(a.S - (KER - 1) + i) * a.proj_stride);
            cs_out[c * (KER - 1) + i] = v[0]; cs_out[(c + 1) * (KER - 1) + i] = v[1];
        }
    }
    const int kind = item < nk ? 0 : item < 2 * nk ? 1 : 2;
    float* dst = kind == 0 ? a.pre_q + c : kind == 1 ? a.pre_k + (c - a.key_dim) : a.pre_v + (c - 2 * a.key_dim);
    const size_t ldd = kind == 2 ? (size_t)a.NV * K : (size_t)a.key_dim;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        f32x2 y = {silu_f(x[i][0] * w0[0] + x[i + 1][0] * w0[1] + x[i + 2][0] * w0[2] + x[i + 3][0] * w0[3]),
                   silu_f(x[i][1] * w1[0] + x[i + 1][1] * w1[1] + x[i + 2][1] * w1[2] + x[i + 3][1] * w1[3])};
        if (kind < 2) {                                  // (a wave's own branch)
            const float n = sqrtf(wave_sum(y[0] * y[0] + y[1] * y[1]) + 1e-6f);
            y[0] = y[0] / n; y[1] = y[1] / n;
            if (kind == 0) { y[0] *= 0.08838834764831845f; y[1] *= 0.08838834764831845f; }      // 1 / sqrt(128)
        }
        if (t0 + i < a.S) *(f32x2*)(dst + (size_t)(t0 + i) * ldd) = y;
    }
    if (kind == 2 && lane < PT && t0 + lane < a.S) { // beta and decay of the value head, a token per lane
        const int h = item - 2 * nk, t = t0 + lane;
        const float* pr = a.proj + (size_t)t * a.proj_stride;
        const float beta = 1.0f / (1.0f + expf(-pr[conv_dim + a.NV * K + h]));
        const float av = pr[conv_dim + a.NV * K + a.NV + h] + a.dt_bias[h];
        const float g = -expf(a.A_log[h]) * logf(1.0f + expf(av));
        a.pre_bd[((size_t)t * a.NV + h) * 2] = beta;
        a.pre_bd[((size_t)t * a.NV + h) * 2 + 1] = expf(g);
        if (a.pre_g != nullptr) a.pre_g[(size_t)t * a.NV + h] = g;
    }
}

// grid = (NV, V / 32), block = 512: thread = (column v = 32 * blockIdx.y + tid / 16, k-slice ks = tid % 16: 8 of the 128 k).
// The recurrence is VALU-issue-bound (4 lane-ops per state element and token), so a value head is spread over 4 CUs and
// 16 lanes share a column: ~50 instructions per token and wave instead of 160 (4 lanes per column, one CU per head:
// 0.59 us per token).  The 16 partial sums of a column are one DPP row reduction.
__global__ __launch_bounds__(512) void gdn_scan_kernel(GdnArgs a) {
    constexpr int K = 128, V = 128, KS = 16, KP = K / KS, CB = 32, TB = 8;
    __shared__ __attribute__((aligned(16))) float qk[2][TB][2][K];      // double-buffered q^ / k^ of TB tokens
    __shared__ float bd[2][TB][2];
    const int h = blockIdx.x, tid = threadIdx.x, v = blockIdx.y * CB + (tid >> 4), ks = tid & 15;
    const int nk = a.NV / a.vpg;
    const int kh = a.chunked ? h % nk : h / a.vpg;
    float* Sg = a.state_pool + (((size_t)a.slot * a.gdn_layers + a.layer_idx) * a.NV + h) * K * V;
    float S[KP];
#pragma unroll
    for (int k = 0; k < KP; ++k) S[k] = Sg[(ks * KP + k) * V + v];
    // The next batch of TB tokens (q^ / k^ rows, beta / decay, this column's v values) is requested into REGISTERS before
    // the current batch is consumed and parked in LDS after it: the loads have a whole batch of compute to arrive.
    float rq[4], rbd = 0.f, vvn[TB], vv[TB];
    auto fetch = [&](int t0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + 512 * i, tt = e >> 8, which = (e >> 7) & 1, kk = e & 127;
            const int t = min(t0 + tt, a.S - 1);
            rq[i] = (which ? a.pre_k : a.pre_q)[(size_t)t * a.key_dim + kh * K + kk];
        }
        if (tid < 2 * TB) rbd = a.pre_bd[((size_t)min(t0 + (tid >> 1), a.S - 1) * a.NV + h) * 2 + (tid & 1)];
#pragma unroll
        for (int i = 0; i < TB; ++i) vvn[i] = a.pre_v[((size_t)min(t0 + i, a.S - 1) * a.NV + h) * V + v];
    };
    auto park = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + 512 * i, tt = e >> 8, which = (e >> 7) & 1, kk = e & 127;
            qk[buf][tt][which][kk] = rq[i];
        }
        if (tid < 2 * TB) bd[buf][tid >> 1][tid & 1] = rbd;
#pragma unroll
        for (int i = 0; i < TB; ++i) vv[i] = vvn[i];
    };
    fetch(0);
    park(0);
    __syncthreads();
    for (int t0 = 0; t0 < a.S; t0 += TB) {
        const int buf = (t0 / TB) & 1;
        fetch(min(t0 + TB, a.S - 1));                // unconditional (clamped): no load under a branch
        const int nt = min(TB, a.S - t0);
#pragma unroll
        for (int i = 0; i < TB; ++i) {
            if (i >= nt) break;
            const float beta = bd[buf][i][0], decay = bd[buf][i][1];
            const f32x4* kp = (const f32x4*)&qk[buf][i][1][ks * KP];
            const f32x4* qp = (const f32x4*)&qk[buf][i][0][ks * KP];
            const f32x4 ka = kp[0], kb = kp[1], qa = qp[0], qb = qp[1];
            const float kf[KP] = {ka[0], ka[1], ka[2], ka[3], kb[0], kb[1], kb[2], kb[3]};
            const float qf[KP] = {qa[0], qa[1], qa[2], qa[3], qb[0], qb[1], qb[2], qb[3]};
            float kv2[2] = {0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KP; ++k) { S[k] *= decay; kv2[k & 1] += S[k] * kf[k]; }
            const float kv = row16_sum(kv2[0] + kv2[1]);          // the 16 k-slices of this column are one DPP row
            const float delta = (vv[i] - kv) * beta;
            float y2[2] = {0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KP; ++k) { S[k] += kf[k] * delta; y2[k & 1] += S[k] * qf[k]; }
            const float y = row16_sum(y2[0] + y2[1]);
            if (ks == 0) a.out[(size_t)(t0 + i) * a.out_stride + h * V + v] = y;      // raw; gdn_post_kernel normalises
        }
        park(buf ^ 1);                               // the other buffer was consumed one iteration ago (barrier below)
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < KP; ++k) Sg[(ks * KP + k) * V + v] = S[k];
}


// ---------------------------------------------------------------------------------------------------------
// Chunk-parallel prompt scan: the gated delta rule in its WY / UT-transform form on the f32 matrix cores.
// The sequential scan above is bound by two dependent 16-lane reductions per token on 64 workgroups (240 us per layer and
// 1024 tokens on Qwen3.5-0.8B: 43 % of its prompt pass).  The reference names the chunked form as the prompt-path algorithm
// (ops/gdn/backend.rs:100-104); HF's torch_chunk_gated_delta_rule is the same algebra.  Per value head and chunk of C = 64
// tokens with state S0 [K x V] at the chunk's start (t, s index tokens of the chunk; G_t = g_1 + ... + g_t, g = log decay):
//     u_t = beta_t (v_t - e^{G_t} S0^T k_t - sum_{s<t} e^{G_t - G_s} (k_s . k_t) u_s)          (the delta rule, unrolled)
//  => (I + A) U = beta V - (beta e^G K) S0,   A[t][s] = beta_t e^{G_t - G_s} (k_t . k_s) for s < t
//  => U = U0 - W S0  with  W = (I + A)^-1 (beta e^G K),  U0 = (I + A)^-1 (beta V)              (independent of S0: all chunks in parallel)
//     Y = e^G (Q S0) + P U,   P[t][s] = e^{G_t - G_s} (q_t . k_s) for s <= t
//     S_C = e^{G_C} S0 + K^T (e^{G_C - G} U)
// gdn_chunk_prep_kernel (grid chunks x NV): A and P on v_mfma_f32_16x16x4_f32, (I + A)^-1 [.] by forward substitution (one
// thread per column of [beta e^G K | beta V], its 64 unknowns in registers: no dependency between threads) -> W, U0, P, G.
// gdn_chunk_scan_kernel (grid NV x V/16): the only sequential part -- U and the state's update, two small matrix products per chunk
// over a 128 x 16 slice of the state (columns of S are independent); for prompts of more than a few chunks it leaves U and the state in front of every chunk to
// gdn_chunk_out_kernel (grid chunks x NV), which forms Y and its gated norm for all chunks at once.  (Y inside the scan is half of
// its products and most of its registers: 2048 tokens, 16 heads, all kernels but gdn_pre_kernel: 145.2 us with it there, 118.3 apart.)  Everything stays f32 (f32 MFMA: products and sums in f32), logs of the
// decays are summed, never multiplied (a decay of e^-80 per token underflows a running product after two tokens).
// Same results as the sequential scan to f32 summation order (tests: prompts through both, logits < 1e-4).
// ---------------------------------------------------------------------------------------------------------
constexpr int CKP = 132;          // LDS row stride (floats) of a 128-wide row: 16-byte aligned, rows 4 banks apart
constexpr int CTP = 68;           // ... of a 64-wide row

// workgroup barrier for LDS hand-offs only: waits for this wave's LDS operations, NOT for its outstanding global loads
// (__syncthreads() carries a workgroup-scope fence that drains vmcnt as well -- it would retire the register prefetch of the
// next chunk at every barrier)
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ f32x4 mfma4(const f32x4& av, const f32x4& bv, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(av[0], bv[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(av[1], bv[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(av[2], bv[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(av[3], bv[3], c, 0, 0, 0);
    return c;
}

// Where Y is formed.  A launch for the outputs of all chunks costs its start and one chunk's chain of products whatever their number, Y inside the scan a
// part of every chunk: short prompts, while the scan's NV x 8 workgroups fit on the chip at once, keep it inside.  us a layer, scan and outputs apart
// minus together, prompts of 2 / 3 / 4 / 5 / 6 / 8 chunks: 16 heads 5.4 / 4.3 / 3.5 / 1.5 / -0.2 / -3.8, 32 heads 6.4 / 2.8 / 0.9 / 0.0 / -1.5 / -4.1, 48 heads (384
// workgroups) -1.7 / -5.2 / -8.4 / -11.0 / -6.2 / -14.3
static bool gdn_out_in_scan(int chunks, int NV) { return chunks <= 5 && NV * 8 <= 256; }

constexpr int ATP = 20;           // ... of a row of a 16 x 16 tile of A
size_t gdn_chunk_prep_lds() { return (size_t)(2 * GDN_CK * CKP + 10 * 16 * ATP + 3 * GDN_CK) * sizeof(float); }
size_t gdn_chunk_scan_lds(bool out) { return (size_t)(16 * CKP + (out ? 2 : 1) * 16 * CTP) * sizeof(float); }

// A keeps the tiles on and under its diagonal only, 81 152 bytes in all: two workgroups fit on a CU and one's products run under the other's chains (the whole of A,
// one workgroup, V requested after the products, a row's decay exponentiated by every column: 50.1 us a launch of 32 chunks and 16 heads, 33.2 now; 48 heads 146.3, 83.9).
// The waves' shares of the triangle are five tiles of A or of P each.
__global__ __launch_bounds__(256, 2) void gdn_chunk_prep_kernel(GdnArgs a) {
    constexpr int K = 128, V = 128, C = GDN_CK;
    extern __shared__ __attribute__((aligned(16))) float cl[];
    float (*Ks)[CKP] = (float (*)[CKP])cl;
    float (*Qs)[CKP] = (float (*)[CKP])(cl + C * CKP);
    float (*Am)[16][ATP] = (float (*)[16][ATP])(cl + 2 * C * CKP);      // tile (I, L), L <= I, at I (I + 1) / 2 + L
    float* lg = cl + 2 * C * CKP + 10 * 16 * ATP;
    float* bt = lg + C;
    float* be = bt + C;                                                 // beta e^G
    const int c = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nk = a.NV / a.vpg, kh = a.chunked ? h % nk : h / a.vpg;
    const int t0 = c * C, nt = min(C, a.S - t0);
    const bool isk = tid < K;
    float* ck = a.ck + ((size_t)c * a.NV + h) * GDN_CK_FLOATS;
    float* Wg = ck, *U0g = ck + C * 128, *Pg = ck + 2 * C * 128, *Gg = ck + 2 * C * 128 + C * C;
    float b[C];                                        // this thread's column of [beta e^G K | beta V]
    {
        f32x4 kv[8], qv[8];                            // k^ and q^ rows of the chunk (rows past the prompt: zero)
        float g = a.pre_g[(size_t)(t0 + min(lane, nt - 1)) * a.NV + h], beta = a.pre_bd[((size_t)(t0 + min(lane, nt - 1)) * a.NV + h) * 2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = tid + 256 * i, row = min(e >> 5, nt - 1), c4 = (e & 31) << 2;
            kv[i] = *(const f32x4*)(a.pre_k + (size_t)(t0 + row) * a.key_dim + kh * K + c4);
            qv[i] = *(const f32x4*)(a.pre_q + (size_t)(t0 + row) * a.key_dim + kh * K + c4);
        }
        if (!isk) {                                    // (requested behind the rows that are needed first)
#pragma unroll
            for (int t = 0; t < C; ++t) b[t] = a.pre_v[((size_t)min(t0 + t, a.S - 1) * a.NV + h) * V + (tid - K)];
        }
        if (wave == 0) {                               // cumulative log decay of the chunk (inclusive), beta
            if (lane >= nt) { g = 0.f; beta = 0.f; }
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) { const float o = __shfl_up(g, d); if (lane >= d) g += o; }
            lg[lane] = g;
            bt[lane] = beta;
            be[lane] = beta * expf(g);
            Gg[lane] = g;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = tid + 256 * i, row = e >> 5, c4 = (e & 31) << 2;
            *(f32x4*)&Ks[row][c4] = row < nt ? kv[i] : (f32x4){0.f, 0.f, 0.f, 0.f};
            *(f32x4*)&Qs[row][c4] = row < nt ? qv[i] : (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    }
    lds_barrier();
    {   // A = tril(beta e^{G_t - G_s} K K^T, -1) -> LDS; P = tril(e^{G_t - G_s} Q K^T) -> scratch.  Even waves A, odd ones P; waves 0 and 1 the rows of
        // tiles 3 and 0, waves 2 and 3 those of 2 and 1: tile n of a wave's five is (hi, n) or (lo, n - n0)
        const int r = lane & 15, kq = lane >> 4;
        const bool isp = wave & 1;
        const int hi = wave < 2 ? 3 : 2, lo = 3 - hi, n0 = hi + 1;
        const float (*As)[CKP] = isp ? Qs : Ks;
        f32x4 acc[5];
#pragma unroll
        for (int n = 0; n < 5; ++n) acc[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const f32x4 ah = *(const f32x4*)&As[16 * hi + r][16 * j + 4 * kq], al = *(const f32x4*)&As[16 * lo + r][16 * j + 4 * kq];
#pragma unroll
            for (int n = 0; n < 5; ++n) {
                const bool up = n < n0;
                acc[n] = mfma4(up ? ah : al, *(const f32x4*)&Ks[16 * (up ? n : n - n0) + r][16 * j + 4 * kq], acc[n]);
            }
        }
#pragma unroll
        for (int n = 0; n < 5; ++n) {
            const int I = n < n0 ? hi : lo, L = n < n0 ? n : n - n0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = 16 * I + 4 * kq + i, s2 = 16 * L + r;
                const float e = s2 <= t ? expf(lg[t] - lg[s2]) : 0.f;
                if (isp) Pg[t * C + s2] = e * acc[n][i];
                else Am[I * (I + 1) / 2 + L][4 * kq + i][r] = s2 < t ? bt[t] * e * acc[n][i] : 0.f;
            }
        }
        if (isp)
#pragma unroll
            for (int n = 0; n < 3; ++n) {              // P over its diagonal: the tiles that neither row of the wave multiplies
                const int I = n < 3 - hi ? hi : lo, L = n < 3 - hi ? n0 + n : lo + 1 + n - (3 - hi);
#pragma unroll
                for (int i = 0; i < 4; ++i) Pg[(16 * I + 4 * kq + i) * C + 16 * L + r] = 0.f;
            }
    }
    lds_barrier();
    // ---- X = (I + A)^-1 [beta e^G K | beta V] by BLOCKED forward substitution (16-token blocks): the off-diagonal part
    // R_I = B_I - sum_{L<I} A_IL X_L on the matrix cores, the 16 x 16 diagonal solves one thread per column (120 FMAs each).
    // (All 64 rows per thread as scalar FMAs were LDS-bound: every thread reads every A[t][s] -- 512 broadcast reads per thread.)
    // X lives in LDS where k^ / q^ were ([64][264] = the same floats): every thread first forms its column of B in registers.
    {
        if (isk) {
#pragma unroll
            for (int t = 0; t < C; ++t) b[t] = be[t] * Ks[t][tid];
        } else {
#pragma unroll
            for (int t = 0; t < C; ++t) b[t] = t < nt ? bt[t] * b[t] : 0.f;
        }
        lds_barrier();                                  // every read of Ks / Qs is done: the region becomes X
        constexpr int XP = 2 * CKP;                    // 264
        float (*X)[XP] = (float (*)[XP])cl;
#pragma unroll
        for (int t = 0; t < C; ++t) X[t][tid] = b[t];
        const int r = lane & 15, kq = lane >> 4;
        auto store = [&](int I) __attribute__((always_inline)) {        // 16 rows of W and of U0, a lane of the scan's own values in one piece
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int j = wave + 4 * i;
                f32x4 u;
#pragma unroll
                for (int n = 0; n < 4; ++n) u[n] = X[16 * I + 4 * kq + n][128 + 16 * j + r];
                *(f32x4*)(Wg + (I * 8 + j) * 256 + lane * 4) = *(const f32x4*)&X[16 * I + r][16 * j + 4 * kq];
                *(f32x4*)(U0g + (I * 8 + j) * 256 + lane * 4) = u;
            }
        };
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            lds_barrier();
            if (I > 0) store(I - 1);
            if (I > 0) {                               // R_I: wave w owns column tiles 4 w .. 4 w + 3
                f32x4 acc[4];
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int L = 0; L < I; ++L) {
                    const f32x4 av = *(const f32x4*)&Am[I * (I + 1) / 2 + L][r][4 * kq];
#pragma unroll
                    for (int n = 0; n < 4; ++n) {
                        f32x4 bv;
#pragma unroll
                        for (int i = 0; i < 4; ++i) bv[i] = X[16 * L + 4 * kq + i][16 * (4 * wave + n) + r];
                        acc[n] = mfma4(av, bv, acc[n]);
                    }
                }
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) X[16 * I + 4 * kq + i][16 * (4 * wave + n) + r] -= acc[n][i];
                lds_barrier();
            }
            float x[16];                               // diagonal block: x_t = r_t - sum_{s<t, same block} A[t][s] x_s
#pragma unroll
            for (int t = 0; t < 16; ++t) x[t] = X[16 * I + t][tid];
#pragma unroll
            for (int t = 1; t < 16; ++t) {
                float p0 = 0.f, p1 = 0.f;
#pragma unroll
                for (int s4 = 0; s4 < t; s4 += 4) {
                    const f32x4 av = *(const f32x4*)&Am[I * (I + 3) / 2][t][s4];
                    p0 += av[0] * x[s4];
                    if (s4 + 1 < t) p1 += av[1] * x[s4 + 1];
                    if (s4 + 2 < t) p0 += av[2] * x[s4 + 2];
                    if (s4 + 3 < t) p1 += av[3] * x[s4 + 3];
                }
                x[t] -= p0 + p1;
            }
#pragma unroll
            for (int t = 0; t < 16; ++t) X[16 * I + t][tid] = x[t];
        }
        lds_barrier();
        store(3);
    }
}

// OUT: Y of every chunk too (raw rows for gdn_post_kernel), nothing left for gdn_chunk_out_kernel
template <bool OUT>
__global__ __launch_bounds__(256, OUT ? 1 : 2) void gdn_chunk_scan_kernel(GdnArgs a) {
    constexpr int K = 128, V = 128, C = GDN_CK, VB = 16;
    extern __shared__ __attribute__((aligned(16))) float cl[];
    float (*St)[CKP] = (float (*)[CKP])cl;                              // state slice, transposed: [column][k]
    float (*Vt)[CTP] = (float (*)[CTP])(cl + VB * CKP);                 // e^{G_C - G_t} U of the chunk, transposed: [column][t]
    float (*Ut)[CTP] = (float (*)[CTP])(cl + VB * CKP + VB * CTP);      // OUT: U of the chunk, transposed: [column][t]
    const int h = blockIdx.x, cb = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int nk = a.NV / a.vpg, kh = a.chunked ? h % nk : h / a.vpg;
    float* Sg = a.state_pool + (((size_t)a.slot * a.gdn_layers + a.layer_idx) * a.NV + h) * K * V;
    float s0[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = tid + 256 * i, k = e >> 4, col = e & 15;
        s0[i] = Sg[k * V + VB * cb + col];
    }
    asm volatile("" ::: "memory");
    const int nchunks = (a.S + C - 1) / C;
    // One or two waves per SIMD: little hides a load but the wave's own work, so the operands of a chunk are requested two chunks ahead into two alternating
    // register sets, each where the one before it in the set is consumed -- unconditionally (rows / chunks past the end are clamped and never
    // consumed, or multiplied by U rows that are zero); each request stands under the products that follow it.  The k^ rows go to registers too: a wave multiplies its own 32 of their columns only, lane r
    // columns 2 r, 2 r + 1 of them, so the two state tiles hold even and odd rows and a lane's eight new state values are neighbours.  Bound by its f32 products
    // (64 a wave and chunk, 14.3 ns each: 0.92 us) and the two hand-offs through LDS.  Us per chunk of 64 tokens: 2.4 with k^ rows staged in LDS one chunk
    // ahead and three barriers; 2.4 from registers with the requests bunched behind the products; 1.8 with them between; 1.66 with W, U0, U and the state
    // stored in the order of the scan's lanes, a request 1 KB in one piece.  32 chunks, 16 heads 80.4 -> 56.6 us, 48 heads 141.1 -> 106.6.
    constexpr int NQ = OUT ? 8 : 1;
    struct Set { f32x4 w[8], q[NQ], p[4], g, u0; f32x2 k[16]; float gC; } sa, sb;
    auto part = [&](int c) __attribute__((always_inline)) { return (const char*)(a.ck + ((size_t)(min(c, nchunks - 1)) * a.NV + h) * GDN_CK_FLOATS); };
    const uint32_t wof = (uint32_t)(wave * 2048 + lane * 4) * 4, kof = (uint32_t)(32 * wave + 2 * r) * 4;
    auto fetch_w = [&](int c, int j, Set& o) __attribute__((always_inline)) {       // 16 columns of the W rows (OUT: and of the q^ rows)
        o.w[j] = *(const f32x4*)(part(c) + wof + 1024 * j);
        if constexpr (OUT) o.q[j] = *(const f32x4*)(a.pre_q + (size_t)min(min(c, nchunks - 1) * C + 16 * wave + r, a.S - 1) * a.key_dim + kh * K + 16 * j + 4 * kq);
    };
    auto fetch_u = [&](int c, Set& o) __attribute__((always_inline)) {  // U0 values and cumulative log decays (OUT: and P rows)
        const char* ck = part(c);
        o.g = *(const f32x4*)(ck + (uint32_t)(2 * C * 128 + C * C + 16 * wave + 4 * kq) * 4);
        o.u0 = *(const f32x4*)(ck + (uint32_t)(C * 128 + (wave * 8 + cb) * 256 + lane * 4) * 4);
        o.gC = *(const float*)(ck + (2 * C * 128 + C * C + C - 1) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (OUT) o.p[i] = *(const f32x4*)(ck + (uint32_t)(2 * C * 128 + (16 * wave + r) * C + 16 * i + 4 * kq) * 4);
        }
    };
    auto fetch_k = [&](int c, int j, Set& o) __attribute__((always_inline)) {       // this wave's columns of four of every 16 k^ rows
        const int t0 = (min(c, nchunks - 1)) * C, last = a.S - 1 - t0;
        const char* kr = (const char*)(a.pre_k + (size_t)t0 * a.key_dim + kh * K);
        int q4 = 4 * kq;
        asm volatile("" : "+v"(q4));                   // (row numbers are added up here, not kept in 16 registers over the whole scan: those spilled)
#pragma unroll
        for (int i = 0; i < 4; ++i)                    // (24-bit products: 64 rows of a few thousand floats)
            o.k[4 * j + i] = *(const f32x2*)(kr + (__umul24(min(q4 + (16 * j + i), last), 4 * a.key_dim) + kof));
    };
    f32x4 st[2];                                       // this lane's state values: column r, rows k = 32 wave + 8 kq + 2 i + m in st[m][i]
    auto chunk = [&](int c, Set& o) __attribute__((always_inline)) {
        char* ck = (char*)(a.ck + ((size_t)c * a.NV + h) * GDN_CK_FLOATS);
        // ---- U = U0 - W S0 (OUT: and Q S0): wave w owns token rows 16 w .. 16 w + 15 ----
        f32x4 accU = {0.f, 0.f, 0.f, 0.f}, accV = accU, accQ = accU, accP = accU, pc[4];
        float eg[4], ed[4];
        const float eC = expf(o.gC);
        f32x4 s[8];                                    // (all of them requested before the first product waits for one, here and below)
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] = *(const f32x4*)&St[r][16 * j + 4 * kq];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                accU = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[j][i], s[j][i], accU, 0, 0, 0);
                accV = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[j + 1][i], s[j + 1][i], accV, 0, 0, 0);
                if constexpr (OUT) accQ = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[j + i / 2][2 * (i & 1)], s[j + i / 2][2 * (i & 1)], accQ, 0, 0, 0);
                if constexpr (OUT) accQ = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[j + i / 2][2 * (i & 1) + 1], s[j + i / 2][2 * (i & 1) + 1], accQ, 0, 0, 0);
            }
            if (!OUT && j == 0) {                        // (stores and requests lie under products: bunched in front of a barrier they hold it up)
                char* sd = ck + (uint32_t)(GDN_CK_ST + (cb * 8 + 2 * wave) * 256 + lane * 4) * 4;
                *(f32x4*)sd = (f32x4){st[0][0], st[1][0], st[0][1], st[1][1]};
                *(f32x4*)(sd + 1024) = (f32x4){st[0][2], st[1][2], st[0][3], st[1][3]};
            }
            ed[j / 2] = expf(o.gC - o.g[j / 2]);
            fetch_w(c + 2, j, o);
            fetch_w(c + 2, j + 1, o);
        }
        f32x4 u, ud;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            u[i] = o.u0[i] - (accU[i] + accV[i]);
            ud[i] = u[i] * ed[i];
            if constexpr (OUT) { eg[i] = expf(o.g[i]); pc[i] = o.p[i]; }
        }
        *(f32x4*)&Vt[r][16 * wave + 4 * kq] = ud;
        if constexpr (OUT) *(f32x4*)&Ut[r][16 * wave + 4 * kq] = u;
        lds_barrier();                                 // Vt is whole, every read of St is done
        if constexpr (OUT) {                           // ---- Y = e^G (Q S0) + P U ----
#pragma unroll
            for (int j = 0; j < 4; ++j) accP = mfma4(pc[j], *(const f32x4*)&Ut[r][16 * j + 4 * kq], accP);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = c * C + 16 * wave + 4 * kq + i;
                if (t < a.S) a.out[(size_t)t * a.out_stride + h * V + VB * cb + r] = eg[i] * accQ[i] + accP[i];
            }
        }
        // ---- S_C = e^{G_C} S0 + K^T (e^{G_C - G} U): wave w owns state rows k = 32 w .. 32 w + 31 ----
        f32x4 accS[2], bv[4];
#pragma unroll
        for (int m = 0; m < 2; ++m) accS[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[j] = *(const f32x4*)&Vt[r][16 * j + 4 * kq];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int m = 0; m < 2; ++m) accS[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[4 * j + i][m], bv[j][i], accS[m], 0, 0, 0);
            if (j == 0) {
                if constexpr (!OUT) *(f32x4*)(ck + (uint32_t)(GDN_CK_UT + (cb * 4 + wave) * 256 + lane * 4) * 4) = u;
                fetch_u(c + 2, o);
            }
            fetch_k(c + 2, j, o);
        }
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) st[m][i] = eC * st[m][i] + accS[m][i];
        *(f32x4*)&St[r][32 * wave + 8 * kq] = (f32x4){st[0][0], st[1][0], st[0][1], st[1][1]};
        *(f32x4*)&St[r][32 * wave + 8 * kq + 4] = (f32x4){st[0][2], st[1][2], st[0][3], st[1][3]};
        lds_barrier();                                 // St is whole, every read of Vt is done
    };
    // (in the loop's order: its waits count the loads behind the one they wait for, over both ways into it)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        Set& o = i ? sb : sa;
#pragma unroll
        for (int j = 0; j < 8; ++j) fetch_w(i, j, o);
        asm volatile("" ::: "memory");
        fetch_u(i, o);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < 4; ++j) fetch_k(i, j, o);
        asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = tid + 256 * i, k = e >> 4, col = e & 15;
        St[col][k] = s0[i];
    }
    lds_barrier();
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) st[m][i] = St[r][32 * wave + 8 * kq + 2 * i + m];
    int c = 0;
    for (; c + 1 < nchunks; c += 2) {
        chunk(c, sa);
        chunk(c + 1, sb);
    }
    if (c < nchunks) chunk(c, sa);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = tid + 256 * i, k = e >> 4, col = e & 15;
        Sg[k * V + VB * cb + col] = St[col][k];
    }
}

// Y = e^G (Q S0) + P U of every chunk and the gated norm of its rows (gdn_post_kernel's), from the states and U rows the scan leaves.  Eight waves:
// 16 token rows x 64 columns each.  Bound by its f32 matrix products (192 per wave, 32 cycles each) and the 150 KB a (chunk, head) reads; U and the
// state share one LDS region, one after the other, so that two workgroups fit on a CU and one loads while the other multiplies (both at once: 29.2
// for 24.1 us)
constexpr size_t gdn_chunk_out_lds = (size_t)(128 * CKP + 128) * sizeof(float);
__global__ __launch_bounds__(512, 4) void gdn_chunk_out_kernel(GdnArgs a) {
    constexpr int K = 128, V = 128, C = GDN_CK;
    extern __shared__ __attribute__((aligned(16))) float cl[];
    float (*St)[CKP] = (float (*)[CKP])cl;                              // S0 transposed: [column][k]
    float (*Ut)[CTP] = (float (*)[CTP])cl;                              // in front of it: U transposed: [column][t]
    float (*red)[C] = (float (*)[C])(cl + 128 * CKP);                   // sums of squares of a row's two halves
    const int c = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, kq = lane >> 4, rt = wave & 3, hf = wave >> 2;
    const int nk = a.NV / a.vpg, kh = a.chunked ? h % nk : h / a.vpg;
    const int t0 = c * C, nt = min(C, a.S - t0);
    const float* ck = a.ck + ((size_t)c * a.NV + h) * GDN_CK_FLOATS;
    f32x4 p[4], q[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) { p[n] = (f32x4){0.f, 0.f, 0.f, 0.f}; q[n] = p[n]; }
    f32x4 s[8];
    {
        f32x4 u[4], ap[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = *(const f32x4*)(ck + GDN_CK_UT + (tid + 512 * i) * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) ap[j] = *(const f32x4*)(ck + 2 * C * 128 + (16 * rt + r) * C + 16 * j + 4 * kq);
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] = *(const f32x4*)(ck + GDN_CK_ST + (tid + 512 * i) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) { const int e = tid + 512 * i, l = e & 63; *(f32x4*)&Ut[(e >> 8) * 16 + (l & 15)][((e >> 6) & 3) * 16 + (l >> 4) * 4] = u[i]; }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < 4; ++n) p[n] = mfma4(ap[j], *(const f32x4*)&Ut[64 * hf + 16 * n + r][16 * j + 4 * kq], p[n]);
    }
    f32x4 aq[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) aq[j] = *(const f32x4*)(a.pre_q + (size_t)min(t0 + 16 * rt + r, a.S - 1) * a.key_dim + kh * K + 16 * j + 4 * kq);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = tid + 512 * i, l = e & 63;
        *(f32x4*)&St[(e >> 9) * 16 + (l & 15)][((e >> 7) & 3) * 32 + (l >> 4) * 8 + ((e >> 6) & 1) * 4] = s[i];
    }
    lds_barrier();
    // the gate's inputs, while the products run
    const int conv_dim = 2 * a.key_dim + a.NV * V;
    const f32x4 g = *(const f32x4*)(ck + 2 * C * 128 + C * C + 16 * rt + 4 * kq);
    float z[4][4], gw[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const int v = 64 * hf + 16 * n + r;
        gw[n] = a.gnorm_w[v];
#pragma unroll
        for (int i = 0; i < 4; ++i) z[n][i] = a.proj[(size_t)min(t0 + 16 * rt + 4 * kq + i, a.S - 1) * a.proj_stride + conv_dim + h * V + v];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int n = 0; n < 4; ++n) q[n] = mfma4(aq[j], *(const f32x4*)&St[64 * hf + 16 * n + r][16 * j + 4 * kq], q[n]);
    float y[4][4], ss[4] = {0.f, 0.f, 0.f, 0.f};                        // [row][column tile]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float eg = expf(g[i]);
#pragma unroll
        for (int n = 0; n < 4; ++n) { y[i][n] = eg * q[n][i] + p[n][i]; ss[i] = fmaf(y[i][n], y[i][n], ss[i]); }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) ss[i] += __shfl_xor(ss[i], o);
        if (r == 0) red[hf][16 * rt + 4 * kq + i] = ss[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = 16 * rt + 4 * kq + i;
        if (t >= nt) continue;
        const float rms = 1.0f / sqrtf((red[0][t] + red[1][t]) / (float)V + a.eps);
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const float v = y[i][n] * rms * gw[n] * silu_f(z[n][i]);
            const size_t at = (size_t)(t0 + t) * a.out_stride + h * V + 64 * hf + 16 * n + r;
            if (a.out_hi == nullptr) { a.out[at] = v; continue; }
            // neighbouring columns make a word: the even lane stores the first terms of both, the odd one the second
            const float o = __shfl_xor(v, 1), e0 = r & 1 ? o : v, e1 = r & 1 ? v : o;
            const uint32_t hi = pack_bf16x2(e0, e1);
            if (!(r & 1)) *(uint32_t*)(a.out_hi + at) = hi;
            else if (a.out_lo != nullptr) *(uint32_t*)(a.out_lo + at - 1) = pack_bf16x2(e0 - bf16_lo(hi), e1 - bf16_hi(hi));
        }
    }
}

__global__ __launch_bounds__(128) void gdn_post_kernel(GdnArgs a) {
    constexpr int V = 128;
    __shared__ float red[2];
    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int conv_dim = 2 * a.key_dim + a.NV * V;
    const float y = a.out[(size_t)t * a.out_stride + h * V + tid];
    const float sy = wave_sum(y * y);
    if (lane == 0) red[wave] = sy;
    __syncthreads();
    const float rms = 1.0f / sqrtf((red[0] + red[1]) / (float)V + a.eps);
    const float z = a.proj[(size_t)t * a.proj_stride + conv_dim + h * V + tid];
    gdn_put(a, (size_t)t * a.out_stride + h * V + tid, y * rms * a.gnorm_w[tid] * silu_f(z));
}

// prompts: three passes (needs the scratch rows of ensure_prefill_buffers); decode steps and short tails: fused
bool gdn_in_passes(const GdnArgs& a) { return a.st == nullptr && a.pre_q != nullptr && a.S >= 16 && a.n_seq <= 1; }

void launch_gdn(const GdnArgs& a, hipStream_t s) {
    if (gdn_in_passes(a)) {
        const int nk = a.NV / a.vpg;
        const unsigned heads = (unsigned)((2 * nk + a.NV + 3) / 4);
        // (four tokens per wave where eight leave too few waves: 1.0 us a layer at 17 .. 449 tokens, none from 769 on)
        if (a.S < 512) hipLaunchKernelGGL(gdn_pre_kernel<4>, dim3((unsigned)((a.S + 3) / 4), heads), dim3(256), 0, s, a);
        else hipLaunchKernelGGL(gdn_pre_kernel<8>, dim3((unsigned)((a.S + 7) / 8), heads), dim3(256), 0, s, a);
        // prompts of a chunk or more: the chunk-parallel scan on the f32 matrix cores (CM_GDN_CHUNKED=0: the sequential scan, A/B)
        static const int ck_env = getenv("CM_GDN_CHUNKED") ? atoi(getenv("CM_GDN_CHUNKED")) : 1;
        if (a.ck != nullptr && a.pre_g != nullptr && ck_env != 0 && a.S >= GDN_CK) {
            static DevOnce attr;
            attr.run([&] {
                (void)hipFuncSetAttribute((const void*)gdn_chunk_prep_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gdn_chunk_prep_lds());
                (void)hipFuncSetAttribute((const void*)gdn_chunk_scan_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gdn_chunk_scan_lds(false));
                (void)hipFuncSetAttribute((const void*)gdn_chunk_scan_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gdn_chunk_scan_lds(true));
                (void)hipFuncSetAttribute((const void*)gdn_chunk_out_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gdn_chunk_out_lds);
            });
            const int chunks = (a.S + GDN_CK - 1) / GDN_CK;
            hipLaunchKernelGGL(gdn_chunk_prep_kernel, dim3(chunks, a.NV), dim3(256), gdn_chunk_prep_lds(), s, a);
            if (gdn_out_in_scan(chunks, a.NV)) {
                hipLaunchKernelGGL(gdn_chunk_scan_kernel<true>, dim3(a.NV, 128 / 16), dim3(256), gdn_chunk_scan_lds(true), s, a);
                hipLaunchKernelGGL(gdn_post_kernel, dim3(a.S, a.NV), dim3(128), 0, s, a);
            } else {
                hipLaunchKernelGGL(gdn_chunk_scan_kernel<false>, dim3(a.NV, 128 / 16), dim3(256), gdn_chunk_scan_lds(false), s, a);
                hipLaunchKernelGGL(gdn_chunk_out_kernel, dim3(chunks, a.NV), dim3(512), gdn_chunk_out_lds, s, a);
            }
            return;
        }
        hipLaunchKernelGGL(gdn_scan_kernel, dim3(a.NV, 4), dim3(512), 0, s, a);
        hipLaunchKernelGGL(gdn_post_kernel, dim3(a.S, a.NV), dim3(128), 0, s, a);
        return;
    }
    if (a.st != nullptr && a.S == 1 && a.gdn_scratch != nullptr && a.gdn_ticket != nullptr) {     // decode step: 4 workgroups per value head
        hipLaunchKernelGGL(gdn_decode_kernel, dim3(a.NV, 4, a.n_seq > 0 ? a.n_seq : 1), dim3(256), 0, s, a);
        return;
    }
    hipLaunchKernelGGL(gdn_kernel, dim3(a.NV, a.n_seq > 0 ? a.n_seq : 1), dim3(128), 0, s, a);
}

__global__ void bf16_to_f32_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst, size_t n, float add) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = bf16_to_f32(src[i]) + add;
}
void launch_bf16_to_f32(const uint16_t* src, float* dst, size_t n, float add, hipStream_t s) {
    int blocks = (int)std::min<size_t>((n + 255) / 256, 1024);
    hipLaunchKernelGGL(bf16_to_f32_kernel, dim3(blocks < 1 ? 1 : blocks), dim3(256), 0, s, src, dst, n, add);
}

}  // namespace cm
