// Decode steps of ONE row through layers with element-wise tanh norms and mixtures of experts, bfloat16 format: the norms and the router inside the
// products that read them.
//
// Such a step is a chain of launches that move 1 .. 15 MB each and wait for each other: launch, first loads, reduction, end.  A norm without a statistic is a
// few operations per element, so every block of the next product makes the whole row for itself (rows of 1024 .. 4096 elements out of the L2) while its
// weights are on their way; so is a router of some tens of logits.  What leaves a launch besides its product is written by one block, into a buffer that
// no other block of the launch reads: the residual goes from x to x2 in front of the mixer and back in front of the experts.
// Every sum is made in the order of the launches that these replace (lay_add_tanh_norm_kernel, lgemv_kernel, lay_router_decode_kernel, lay_attn_merge_kernel): the
// same bits.
// Measured (us, width 1024, 14 experts of 768, 4 per token, and one of 512): norm + router + gate-and-up 18.9 in three launches, 8.3 here; norm and input
// projection 7.8 in two, 4.1 here; the second product 5.3, 4.2 (its matrices follow from the choices, not from the sorted rows); output projection behind
// five attention shares 9.0 with a merging launch, 4.3 here.
#include <algorithm>

#include "dev_common.h"
#include "kernels.h"
#include "layered.h"
#include "layered_dev.h"

namespace cm {

namespace {

// the row through residual update and norm: h[k] for all k in LDS (f32), the new residual to xout where this block writes it
template <int NIT>
__device__ __forceinline__ void step_norm(const LStepNorm& a, float* __restrict__ h, bool writes) {
    float2 x[NIT], nw[NIT], nb[NIT];
    const int k0 = (int)threadIdx.x * 2;
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        x[i] = *(const float2*)(a.x + k0 + i * 512);
        nw[i] = *(const float2*)(a.w + k0 + i * 512);
        nb[i] = *(const float2*)(a.b + k0 + i * 512);
    }
    if (a.y) {
        float2 sum[NIT];
#pragma unroll
        for (int i = 0; i < NIT; ++i) sum[i] = make_float2(0.f, 0.f);
#pragma unroll 4
        for (int k = 0; k < a.nsum; ++k) {
            const float f = a.wsel ? a.wsel[k] : 1.f;
#pragma unroll
            for (int i = 0; i < NIT; ++i) {
                const float2 y = *(const float2*)(a.y + (size_t)k * (NIT * 512) + k0 + i * 512);
                sum[i].x = fmaf(f, y.x, sum[i].x); sum[i].y = fmaf(f, y.y, sum[i].y);
            }
        }
#pragma unroll
        for (int i = 0; i < NIT; ++i) { x[i].x = fmaf(a.mult, sum[i].x, x[i].x); x[i].y = fmaf(a.mult, sum[i].y, x[i].y); }
    }
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        if (writes) *(float2*)(a.xout + k0 + i * 512) = x[i];
        *(float2*)(h + k0 + i * 512) = make_float2(fmaf(tanhf(a.alpha * x[i].x), nw[i].x, nb[i].x), fmaf(tanhf(a.alpha * x[i].y), nw[i].y, nb[i].y));
    }
}
// a lane's eight elements of h, as they are
__device__ __forceinline__ void step_row(const float* h, int k, float (&x)[8]) {
    const f32x4 a = *(const f32x4*)(h + k), b = *(const f32x4*)(h + k + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { x[i] = a[i]; x[4 + i] = b[i]; }
}
__device__ __forceinline__ float step_dot(float acc, const u32x4& w, const float (&x)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) { acc = fmaf(bf16_lo(w[i]), x[2 * i], acc); acc = fmaf(bf16_hi(w[i]), x[2 * i + 1], acc); }
    return acc;
}

// C = act(norm(x) W^T + bias), two columns per wave; columns of queries, keys and values through their convolution, whose inputs and weights are on their way meanwhile
template <int NIT>
__global__ __launch_bounds__(256) void lay_step_in_kernel(LStepNorm a, LStepProj p, LStepConv cv) {
    constexpr int K = NIT * 512;
    __shared__ __attribute__((aligned(16))) float h[K];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = min((int)(blockIdx.x * 4 + wave) * 2, p.N - 1), n1 = min(n0 + 1, p.N - 1);
    u32x4 w0[NIT], w1[NIT];
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        w0[i] = ld_nt16(p.W + (size_t)n0 * K + lane * 8 + i * 512);
        w1[i] = ld_nt16(p.W + (size_t)n1 * K + lane * 8 + i * 512);
    }
    const int n = (int)(blockIdx.x * 4 + wave) * 2 + lane;
    const bool conv = lane < 2 && n < cv.C;
    float in[LAY_STEP_TAPS], cw[LAY_STEP_TAPS];            // taps in front of the first one: weight 0
#pragma unroll
    for (int j = 0; j < LAY_STEP_TAPS; ++j) {
        const int t = j - (LAY_STEP_TAPS - cv.taps);
        cw[j] = conv && t >= 0 ? cv.cw[(size_t)t * cv.C + n] : 0.f;
        in[j] = conv && t >= 0 && t < cv.taps - 1 ? cv.tail[(size_t)t * cv.C + n] : 0.f;
    }
    step_norm<NIT>(a, h, blockIdx.x == 0);
    __syncthreads();
    float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        float x[8];
        step_row(h, lane * 8 + i * 512, x);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = bf16_round(x[j]);
        acc0 = step_dot(acc0, w0[i], x);
        acc1 = step_dot(acc1, w1[i], x);
    }
    acc0 = wave_sum(acc0); acc1 = wave_sum(acc1);
    if (lane < 2 && n < p.N) {
        float v = lane ? acc1 : acc0;
        if (p.bias) v += p.bias[n];
        v = lay_act(v, n < p.act_split ? p.act : p.act2, p.act_param);
        if (conv) {
            in[LAY_STEP_TAPS - 1] = v;
            v = 0.f;
#pragma unroll
            for (int j = 0; j < LAY_STEP_TAPS; ++j) v = fmaf(cw[j], in[j], v);
#pragma unroll
            for (int j = 1; j < LAY_STEP_TAPS; ++j) {
                const int t = j - 1 - (LAY_STEP_TAPS - cv.taps);
                if (t >= 0) cv.tail[(size_t)t * cv.C + n] = in[j];
            }
        }
        p.C[n] = v;
    }
}

// C = (attention rows merged from their shares) W^T, two columns per wave: lay_attn_merge_kernel's sums in every block
template <int NIT>
__global__ __launch_bounds__(256) void lay_step_out_kernel(LAttnArgs a, int nsplit, const uint16_t* __restrict__ W, float* __restrict__ C, int N) {
    constexpr int K = NIT * 512;
    __shared__ __attribute__((aligned(16))) float h[K];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = min((int)(blockIdx.x * 4 + wave) * 2, N - 1), n1 = min(n0 + 1, N - 1);
    u32x4 w0[NIT], w1[NIT];
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        w0[i] = ld_nt16(W + (size_t)n0 * K + lane * 8 + i * 512);
        w1[i] = ld_nt16(W + (size_t)n1 * K + lane * 8 + i * 512);
    }
    const int nrep = a.H / a.G, e = a.e;
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        const int k = (int)threadIdx.x * 2 + i * 512, head = k / e, c = k - head * e, g = head / nrep;      // (e is even)
        const size_t p0 = (size_t)g * nsplit * 16 + (head - g * nrep);
        const float gate = a.gbuf[head];
        // eight shares requested at once (a loop over their number would wait for each): past the last one it again, with weight 0
        constexpr int AT = 8;
        float2 ml[AT], po[AT];
        auto request = [&](int z0) __attribute__((always_inline)) {
#pragma unroll
            for (int z = 0; z < AT; ++z) {
                const size_t pr = p0 + (size_t)min(z0 + z, nsplit - 1) * 16;
                ml[z] = *(const float2*)(a.part_ml + pr * 2); po[z] = *(const float2*)(a.part_o + pr * e + c);
            }
        };
        request(0);
        float M = -INFINITY, L = 0.f;
#pragma unroll
        for (int z = 0; z < AT; ++z) M = fmaxf(M, ml[z].x);
        for (int z = AT; z < nsplit; ++z) M = fmaxf(M, a.part_ml[(p0 + (size_t)z * 16) * 2]);
        float2 acc = make_float2(0.f, 0.f);
        for (int z0 = 0; z0 < nsplit; z0 += AT) {
            if (z0 > 0) request(z0);
#pragma unroll
            for (int z = 0; z < AT; ++z) {
                const float w = ml[z].x == -INFINITY || z0 + z >= nsplit ? 0.f : expf(ml[z].x - M);
                L = z0 + z < nsplit ? fmaf(ml[z].y, w, L) : L;
                acc.x = z0 + z < nsplit ? fmaf(po[z].x, w, acc.x) : acc.x;
                acc.y = z0 + z < nsplit ? fmaf(po[z].y, w, acc.y) : acc.y;
            }
        }
        *(float2*)(h + k) = make_float2(bf16_round(acc.x * gate / L * a.out_scale), bf16_round(acc.y * gate / L * a.out_scale));
    }
    __syncthreads();
    float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
        float x[8];
        step_row(h, lane * 8 + i * 512, x);
        acc0 = step_dot(acc0, w0[i], x);
        acc1 = step_dot(acc1, w1[i], x);
    }
    acc0 = wave_sum(acc0); acc1 = wave_sum(acc1);
    const int n = (int)(blockIdx.x * 4 + wave) * 2 + lane;
    if (lane < 2 && n < N) C[n] = lane ? acc1 : acc0;
}

// norm, router, choice, and act(h W_e^T) * (h W2_e^T) of the chosen experts and the one of every token.  blockIdx.y: the choice, the last the expert of every token.  A last block
// of the first choice writes the choices and their weights, which the others do not wait for (one wave's choice for
// the block and all of them through it 9.3 us a launch, each its own 8.3)
template <int NIT>
__global__ __launch_bounds__(256) void lay_step_moe_kernel(LStepNorm a, LStepMoe m) {
    constexpr int K = NIT * 512, NR = NIT <= 2 ? 4 : NIT == 4 ? 2 : 1;     // router outputs of a wave whose weights are requested together
    __shared__ __attribute__((aligned(16))) float h[K];
    __shared__ float zs[2 * 64 + 2 + 64], swt[65];            // lay_router_choose: logits, scores, one group, choices
    __shared__ int32_t ss[64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, slot = blockIdx.y;
    const bool every = slot == m.top, first = blockIdx.x == 0 && slot == 0, writes = blockIdx.x == gridDim.x - 1;
    const int N = every ? m.sh_ff : m.ff;
    if (writes ? slot != 0 : (int)blockIdx.x * 8 >= N) return;
    const int logits = m.experts + (m.rs.shared_gate ? 1 : 0);
    u32x4 rw[NR][NIT];
    auto request = [&](int e0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NR; ++j)
#pragma unroll
            for (int i = 0; i < NIT; ++i) rw[j][i] = ld16(m.router + (size_t)min(e0 + 4 * j, logits - 1) * K + lane * 8 + i * 512);
    };
    if (!every) request(wave);
    step_norm<NIT>(a, h, first);
    __syncthreads();
    int e = 0;
    if (!every) {
        for (int e0 = wave; e0 < logits; e0 += 4 * NR) {
            float acc[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) acc[j] = 0.f;
#pragma unroll
            for (int i = 0; i < NIT; ++i) {
                float x[8];
                step_row(h, lane * 8 + i * 512, x);
#pragma unroll
                for (int j = 0; j < NR; ++j) acc[j] = step_dot(acc[j], rw[j][i], x);
            }
            if (e0 + 4 * NR < logits) request(e0 + 4 * NR);
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const float z = wave_sum(acc[j]);
                if (lane == 0 && e0 + 4 * j < logits) zs[e0 + 4 * j] = z;
            }
        }
        __syncthreads();
        e = writes ? -1 : lay_router_choice(zs, lane, slot, m.experts, m.rs);
        if (e < 0) {                           // (every wave has it from the same logits: uniform in the block)
            __syncthreads();                   // lay_router_choose writes over logits that a slower wave may still read
            if (wave == 0) lay_router_choose(zs, 0, lane, ss, swt, m.experts, m.top, m.rs, nullptr, m.slots);
            __syncthreads();
            e = ss[slot];
            if (writes) {
                for (int k = threadIdx.x; k < m.top; k += 256) m.sel[k] = ss[k];
                for (int k = threadIdx.x; k < m.slots; k += 256) m.wsel[k] = swt[k];
                return;
            }
        }
        e = __builtin_amdgcn_readfirstlane(e);
    }
    const uint16_t* W = every ? m.sh_gate : m.gate + (size_t)e * m.ff * K;
    const uint16_t* W2 = every ? m.sh_up : m.up + (size_t)e * m.ff * K;
    const int n0 = min((int)(blockIdx.x * 4 + wave) * 2, N - 1), n1 = min(n0 + 1, N - 1);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    constexpr int NB = NIT < 4 ? NIT : 4;                                  // k pieces requested together: 4 NB loads of 16 bytes per lane
#pragma unroll
    for (int i0 = 0; i0 < NIT; i0 += NB) {
        u32x4 w[NB][4];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const size_t k = (size_t)lane * 8 + (i0 + i) * 512;
            w[i][0] = ld_nt16(W + (size_t)n0 * K + k); w[i][1] = ld_nt16(W + (size_t)n1 * K + k);
            w[i][2] = ld_nt16(W2 + (size_t)n0 * K + k); w[i][3] = ld_nt16(W2 + (size_t)n1 * K + k);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            float x[8];
            step_row(h, lane * 8 + (i0 + i) * 512, x);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = bf16_round(x[j]);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] = step_dot(acc[c], w[i][c], x);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = wave_sum(acc[c]);
    const int n = (int)(blockIdx.x * 4 + wave) * 2 + lane;
    if (lane < 2 && n < N) {
        const float v = lane ? acc[1] : acc[0], u = lane ? acc[3] : acc[2];
        float* out = every ? m.hs : m.hh + (size_t)slot * m.ff;
        out[n] = lay_act(v, LACT_SILU) * u;
    }
}

// the second product of the chosen experts and the one of every token: ys[slot] = inner row of the slot times its matrix
__global__ __launch_bounds__(256) void lay_step_down_kernel(LStepMoe m, float* __restrict__ ys, int W) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, slot = blockIdx.y;
    const bool every = slot == m.top;
    const int K = every ? m.sh_ff : m.ff;
    const float* x = every ? m.hs : m.hh + (size_t)slot * m.ff;
    const int n0 = min((int)(blockIdx.x * 4 + wave) * 2, W - 1), n1 = min(n0 + 1, W - 1);
    const uint16_t* D = every ? m.sh_down : m.down + (size_t)m.sel[slot] * W * m.ff;
    float acc0 = 0.f, acc1 = 0.f;
#pragma unroll 4
    for (int k = lane * 8; k < K; k += 512) {
        const u32x4 w0 = ld_nt16(D + (size_t)n0 * K + k), w1 = ld_nt16(D + (size_t)n1 * K + k);
        float v[8];
        step_row(x, k, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = bf16_round(v[j]);
        acc0 = step_dot(acc0, w0, v);
        acc1 = step_dot(acc1, w1, v);
    }
    acc0 = wave_sum(acc0); acc1 = wave_sum(acc1);
    const int n = (int)(blockIdx.x * 4 + wave) * 2 + lane;
    if (lane < 2 && n < W) ys[(size_t)slot * W + n] = lane ? acc1 : acc0;
}

}  // namespace

// All widths and numbers of logits that the kernels are made for pay, although every block repeats norm and router.  us a layer behind 24 tokens, single launches / here
// (width, experts, per token, columns): 512, 8, 2, 512 41.1 / 31.0; 512, 63, 4, 512 49.4 / 35.1; 1024, 14, 4, 768 51.7 / 39.1; 1024, 63, 8, 768 63.5 / 49.7; 2048, 16, 4, 1024
// 68.6 / 54.5; 2048, 63, 8, 1024 92.8 / 80.7; 4096, 8, 2, 2048 94.4 / 86.7; 4096, 16, 4, 2048 110.7 / 107.0; 4096, 63, 4, 1024 117.3 / 99.6
bool lay_step_fits(int W, const LayerSpec& sp) {
    const int logits = sp.experts + (sp.router.shared_gate ? 1 : 0);
    return (W == 512 || W == 1024 || W == 2048 || W == 4096) && sp.mlp == LMLP_MOE && !sp.scale_input && sp.router.identity == 0 && sp.router.groups == 1 &&
           !sp.router.correction && sp.expert_act == LACT_SILU && logits <= 64 && sp.top <= 63 && sp.ff % 8 == 0 && sp.shared_ff % 8 == 0;
}
#define CM_STEP_W(CALL) switch (W) { case 512: CALL(1); break; case 1024: CALL(2); break; case 2048: CALL(4); break; default: CALL(8); }
void launch_lay_step_in(const LStepNorm& a, const LStepProj& p, const LStepConv& c, int W, hipStream_t s) {
#define CM_CALL(I) hipLaunchKernelGGL(lay_step_in_kernel<I>, dim3((unsigned)((p.N + 7) / 8)), dim3(256), 0, s, a, p, c)
    CM_STEP_W(CM_CALL)
#undef CM_CALL
}
// Every block merges the whole row, shares x K sums out of the L2, eight shares of K / 512 elements per thread requested at once: that has to cost less than the
// launch that merges once -- one batch of eight at K 2048, two at 1024, four at 512.  us a layer, merged there / here: K 1024, 2 / 5 / 8 / 11 / 14 shares 42.0 / 37.9, 43.7 / 37.7, 42.1 /
// 37.9, 43.5 / 41.7, 44.7 / 43.8; K 2048, 2 / 4 / 6 / 8 / 11 / 14 47.9 / 45.8, 49.0 / 45.4, 50.0 / 46.5, 48.9 / 47.3, 50.4 / 54.6, 51.3 / 58.4, on a width of 4096 2 / 8 / 14 62.9 / 62.6, 63.9 /
// 64.0, 66.7 / 74.3; K 4096, 2 / 6 / 14 72.1 / 77.2, 73.7 / 78.2, 74.7 / 101.1
bool lay_step_out_fits(const LAttnArgs& a) {
    const int K = a.H * a.e;
    // (a key head's queries in one tile of 16: the kernel finds a head's shares by its place in the first)
    return a.nsplit > 1 && (long long)((a.nsplit + 7) / 8) * K <= 2048 && a.H <= 16 * a.G && (K == 512 || K == 1024 || K == 2048) && a.e % 2 == 0 &&
           a.gate == LGATE_HEAD;
}
void launch_lay_step_out(const LAttnArgs& a, const uint16_t* Wm, float* C, int N, hipStream_t s) {
    const dim3 grid((unsigned)((N + 7) / 8));
    const int K = a.H * a.e;
    if (K == 512) hipLaunchKernelGGL(lay_step_out_kernel<1>, grid, dim3(256), 0, s, a, a.nsplit, Wm, C, N);
    else if (K == 1024) hipLaunchKernelGGL(lay_step_out_kernel<2>, grid, dim3(256), 0, s, a, a.nsplit, Wm, C, N);
    else hipLaunchKernelGGL(lay_step_out_kernel<4>, grid, dim3(256), 0, s, a, a.nsplit, Wm, C, N);
}
void launch_lay_step_moe(const LStepNorm& a, const LStepMoe& m, float* ys, int W, hipStream_t s) {
    const unsigned slots = (unsigned)(m.top + (m.sh_ff > 0 ? 1 : 0));
    const dim3 grid((unsigned)((std::max(m.ff, m.sh_ff) + 7) / 8 + 1), slots);
#define CM_CALL(I) hipLaunchKernelGGL(lay_step_moe_kernel<I>, grid, dim3(256), 0, s, a, m)
    CM_STEP_W(CM_CALL)
#undef CM_CALL
    hipLaunchKernelGGL(lay_step_down_kernel, dim3((unsigned)((W + 7) / 8), slots), dim3(256), 0, s, m, ys, W);
}
#undef CM_STEP_W

}  // namespace cm
