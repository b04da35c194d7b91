// Attention of the vision tower: every patch of a frame against every patch of the same frame, head_dim 64, no mask.  Q, K and V are bf16 hi + lo
// planes of f32 values (three products each: s = kh.qh + kh.ql + kl.qh, o += vh.ph + vh.pl + vl.ph); K / V rows lie as
// [64 patches][heads][patch][64] blocks.  ONE launch for all frames and images of a pass: a workgroup looks its (frame, rows) up in a table.
//
// What bounds it: matrix and vector work, which share the SIMDs and overlap little (two waves on each: 96 products and 270 vector instructions per
// wave and key tile, 16 x 96 and 4.5 x 270 cycles of the 3400 measured), and CUs that get one workgroup where others get two.  So: the planes of a
// key tile go from memory into LDS without passing registers (the next tile's while this one is worked on; 64 keys x 128 bytes per plane, 16-byte
// chunks moved by an XOR of the row on the source address so that neither the 16-row fragment reads of K nor the transposed reads of V meet in a
// bank: 0 conflicts); a wave owns 32 rows where there are enough of them and uses every fragment twice; two 16-key groups of P^T go into one
// 16 x 16 x 32 product, which takes as long as a 16 x 16 x 16 one (the order of the keys inside the product is the same permutation on both
// operands).  All frames in one launch instead of one launch per frame with two runs of keys and a merge: 42 x 64 and 22 x 22 patches, 16 heads
// 174 -> 114 us per block of the tower (two runs of keys and their merge; 127 in one run), six images of 22 x 22 patches: tower 10.6 -> 8.2 ms.  Measured and no better: the next tile's scores issued
// between this tile's exponentials (registers), eight waves of 16 rows (registers).
#include "dev_common.h"
#include "kernels.h"

namespace cm {

namespace {

constexpr int D = 64, KT = 64;

// four probabilities as bf16 hi and lo pairs
__device__ __forceinline__ void split_p(const float (&p)[4], uint32_t* hi, uint32_t* lo) {
    hi[0] = pack_bf16x2(p[0], p[1]); hi[1] = pack_bf16x2(p[2], p[3]);
    lo[0] = pack_bf16x2(p[0] - bf16_lo(hi[0]), p[1] - bf16_hi(hi[0]));
    lo[1] = pack_bf16x2(p[2] - bf16_lo(hi[1]), p[3] - bf16_hi(hi[1]));
}

__device__ __forceinline__ void store4(uint16_t* hi, uint16_t* lo, size_t at, const float (&v)[4]) {
    uint32_t h[2], l[2];
    split_p(v, h, l);
    *(u32x2*)(hi + at) = (u32x2){h[0], h[1]};
    *(u32x2*)(lo + at) = (u32x2){l[0], l[1]};
}

// grid (heads x tiles, runs), heads first: the workgroups of a head follow each other by `heads`, so that its K / V stay in one XCD's L2 where heads % 8 == 0
template <int NQ>
__global__ __launch_bounds__(256, 2) void vit_attn_kernel(VitAttnArgs a) {
    constexpr int PLANE = KT * D, STAGE = 4 * PLANE;                   // K hi, K lo, V hi, V lo
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * STAGE];
    constexpr float L2E = 1.4426950408889634f;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = lane & 15, g = lane >> 4;
    const int heads = a.heads, h = (int)blockIdx.x % heads;
    const int4 tl = a.tiles[(int)blockIdx.x / heads];                               // first and end row of the frame, first query row
    const int lo = tl.x, end = tl.y;
    bf16x8 qh[NQ][2], ql[NQ][2];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const size_t at = ((size_t)min(tl.z + (wave * NQ + n) * 16 + sub, end - 1) * heads + h) * D + g * 8;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            qh[n][ks] = *(const bf16x8*)(a.q_hi + at + ks * 32);
            ql[n][ks] = *(const bf16x8*)(a.q_lo + at + ks * 32);
        }
    }
    f32x4 o[NQ][4];
    float m_run[NQ], l_run[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        m_run[n] = -INFINITY; l_run[n] = 0.f;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) o[n][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const int all = (end - lo + KT - 1) / KT, full = (end - lo) / KT, per = (all + a.runs - 1) / a.runs;
    const int t0 = (int)blockIdx.y * per, t1 = min(all, t0 + per);     // this workgroup's run of key tiles (may be empty)
    // wave w brings plane w of a tile: eight requests of eight rows.  A row's address moves on by one 64-row block per tile
    const uint16_t* const plane = (wave < 2 ? a.k : a.v) + (wave & 1 ? a.lo_off : 0);
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + (uint32_t)wave * PLANE * 2u;
    const int prow = lane >> 3, pslot = lane & 7;
    auto source = [&](int row, int i) __attribute__((always_inline)) -> uint32_t {      // element of the plane that slot pslot of tile row 8 i + prow holds
        const int tr = 8 * i + prow, f = wave < 2 ? (tr >> 1) & 7 : ((tr >> 1) & 3) << 1;
        return (uint32_t)(((row >> 6) * heads + h) * 64 + (row & 63)) * D + (uint32_t)((pslot ^ f) << 3);
    };
    uint32_t src[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) src[i] = source(lo + 8 * i + prow, i);
    auto request = [&](int t) __attribute__((always_inline)) {
        const uint32_t dst = lds0 + (uint32_t)((t & 1) * STAGE) * 2u;
        if (t < full) {
            const uint16_t* p = plane + (size_t)t * heads * (64 * D);
#pragma unroll
            for (int i = 0; i < 8; ++i) lds_load16(p + src[i], dst + i * 1024u);
        } else {                                                       // the ragged end: its last row again
#pragma unroll
            for (int i = 0; i < 8; ++i) lds_load16(plane + source(min(lo + t * KT + 8 * i + prow, end - 1), i), dst + i * 1024u);
        }
    };
    const int kf = (sub >> 1) & 7, vf = (2 * g + (sub >> 3)) & 3;
    const int vrow = (g * 4 + (sub >> 2)) * D + (sub & 1) * 4;
    auto tile = [&](int t, auto masked_c) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked_c)::value;
        const uint16_t* S = lds + (t & 1) * STAGE;
        f32x4 s[NQ][4];
#pragma unroll
        for (int n = 0; n < NQ; ++n)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) s[n][tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int kc = ((ks * 4 + g) ^ kf) << 3;
            bf16x8 kh[4], kl[4];
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                kh[tt] = *(const bf16x8*)&S[(tt * 16 + sub) * D + kc];
                kl[tt] = *(const bf16x8*)&S[PLANE + (tt * 16 + sub) * D + kc];
            }
#pragma unroll
            for (int p = 0; p < 3; ++p)                                // products of one accumulator stand apart
#pragma unroll
                for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                    for (int n = 0; n < NQ; ++n) s[n][tt] = mma_k32<KV_BF16>(p == 2 ? kl[tt] : kh[tt], p == 1 ? ql[n][ks] : qh[n][ks], s[n][tt]);
        }
        u32x4 ph[NQ][2], pl[NQ][2];                                    // keys 4 g + r of groups 2 u and 2 u + 1
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            float mt = -INFINITY;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (MASKED) { if (lo + t * KT + tt * 16 + g * 4 + r >= end) s[n][tt][r] = -INFINITY; }
                    mt = fmaxf(mt, s[n][tt][r]);
                }
            mt = rows_max(mt);
            const float m_new = fmaxf(m_run[n], mt);                   // finite: every tile holds a patch of the frame
            const float alpha = __builtin_amdgcn_exp2f((m_run[n] - m_new) * L2E), nm = -m_new * L2E;
            float psum = 0.f;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                float p[4];
                uint32_t hi[2], lw[2];
#pragma unroll
                for (int r = 0; r < 4; ++r) { p[r] = __builtin_amdgcn_exp2f(fmaf(s[n][tt][r], L2E, nm)); psum += p[r]; }
                split_p(p, hi, lw);
                ph[n][tt >> 1][(tt & 1) * 2] = hi[0]; ph[n][tt >> 1][(tt & 1) * 2 + 1] = hi[1];
                pl[n][tt >> 1][(tt & 1) * 2] = lw[0]; pl[n][tt >> 1][(tt & 1) * 2 + 1] = lw[1];
            }
            l_run[n] = l_run[n] * alpha + psum;
            m_run[n] = m_new;
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) { o[n][nt][0] *= alpha; o[n][nt][1] *= alpha; o[n][nt][2] *= alpha; o[n][nt][3] *= alpha; }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            bf16x8 vh[4], vl[4];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const int at = 2 * PLANE + u * 32 * D + vrow + ((((nt ^ vf) << 1) + ((sub & 3) >> 1)) << 3);
                auto frag = [&](const uint16_t* V) __attribute__((always_inline)) {
                    const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)V));
                    const u32x2 y = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)(V + 16 * D)));
                    return __builtin_bit_cast(bf16x8, (u32x4){x[0], x[1], y[0], y[1]});
                };
                vh[nt] = frag(S + at); vl[nt] = frag(S + PLANE + at);
            }
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                    for (int n = 0; n < NQ; ++n) {
                        const bf16x8 pv = __builtin_bit_cast(bf16x8, p == 1 ? pl[n][u] : ph[n][u]);
                        o[n][nt] = mma_k32<KV_BF16>(p == 2 ? vl[nt] : vh[nt], pv, o[n][nt]);
                    }
        }
    };
    if (t0 < t1) request(t0);
    for (int t = t0; t < t1; ++t) {
        // tile t has landed and every wave has read tile t - 1, whose stage the next one goes to
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (t + 1 < t1) request(t + 1);
        if (t < full) tile(t, std::false_type{}); else tile(t, std::true_type{});
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        float l = l_run[n];
        l = rows_sum(l);
        const int row = tl.z + (wave * NQ + n) * 16 + sub;
        if (row >= end) continue;
        if (a.runs > 1) {                                              // un-normalised; an empty run: maximum -inf, sum 0
            const size_t at = ((size_t)blockIdx.y * a.rows + row) * heads + h;
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) *(f32x4*)(a.part_o + at * D + nt * 16 + g * 4) = o[n][nt];
            if (g == 0) { a.part_ml[at * 2] = m_run[n]; a.part_ml[at * 2 + 1] = l; }
        } else {
            const float inv = 1.0f / l;
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const float v[4] = {o[n][nt][0] * inv, o[n][nt][1] * inv, o[n][nt][2] * inv, o[n][nt][3] * inv};
                store4(a.out_hi, a.out_lo, ((size_t)row * heads + h) * D + nt * 16 + g * 4, v);
            }
        }
    }
}

// out = sum_z e^(m_z - M) o_z / sum_z e^(m_z - M) l_z of the runs.  One thread per (row, head, 4 dims)
__global__ __launch_bounds__(256) void vit_attn_merge_kernel(VitAttnArgs a) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, zs = (size_t)a.rows * a.heads;
    if (i >= zs * (D / 4)) return;
    const size_t row = i / (D / 4);
    const int d4 = (int)(i % (D / 4)) * 4;
    float M = -INFINITY;
    for (int z = 0; z < a.runs; ++z) M = fmaxf(M, a.part_ml[(z * zs + row) * 2]);
    float L = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < a.runs; ++z) {
        const float mz = a.part_ml[(z * zs + row) * 2];
        const float w = mz > -INFINITY ? expf(mz - M) : 0.f;
        L += w * a.part_ml[(z * zs + row) * 2 + 1];
        const f32x4 p = *(const f32x4*)(a.part_o + (z * zs + row) * D + d4);
        acc[0] += w * p[0]; acc[1] += w * p[1]; acc[2] += w * p[2]; acc[3] += w * p[3];
    }
    const float inv = 1.0f / L;
    const float v[4] = {acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
    store4(a.out_hi, a.out_lo, row * D + d4, v);
}

}  // namespace

void launch_vit_attn(const VitAttnArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)a.heads * (unsigned)a.ntiles, (unsigned)a.runs);
    if (a.wide) hipLaunchKernelGGL(vit_attn_kernel<2>, grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(vit_attn_kernel<1>, grid, dim3(256), 0, s, a);
    if (a.runs > 1) {
        const size_t n = (size_t)a.rows * a.heads * (D / 4);
        hipLaunchKernelGGL(vit_attn_merge_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    }
}

}  // namespace cm
