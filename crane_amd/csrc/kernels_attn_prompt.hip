// Prompt attention of the dense decoders over 2-byte pages, head_dim 128, where there are many query tiles: attn_prefill_fast_kernel's sums (kernels_prefill.hip), one query head per four
// waves and two of a key head per workgroup.
//
// What bounds it: the chain of a tile -- fragments out of the LDS, 32 products, a maximum over the lanes, exponentials, 32 products: 1.7 us for 0.43 of products -- which only other
// waves of the SIMD hide.  That kernel holds two tiles in 64 registers on their way to the LDS and 69 KB of LDS for four waves, so two waves share a SIMD; here rows go from memory into
// the LDS directly, eight waves share 64 KB of it and stay within 128 registers, so four do, and the sums are scaled only when a maximum in the wave has moved.  The order of
// every sum is that kernel's.
// Measured (us a launch, that kernel / here, 32 heads on 8): 2048 rows 114 / 85, behind 2048 tokens 269 / 188; 1400 rows behind 2048 tokens 192 / 165; where that kernel's places fill again as the short walks end it
// is ahead: 1000 rows 35 / 39, 16 heads 2048 rows 60 / 70.  The line stands beside launch_prefill_fast.
// Two heads in every wave (its fragments shared, two chains, 250 registers): 99 / 191 us in the place of 85 / 188; matrix and vector instructions of the two put side by side by hand: 98 / 195;
// the waves 4-7 half a tile behind the others (174 registers): 120 / 260.
//
// LDS: two stages of a key and a value tile, rows of 256 bytes.  Slot p of key row r holds chunk p ^ (r & 15): the 16 rows of a fragment read fall on 16 slots; of value row r chunk
// p ^ 2 (r & 7): so do the pairs of chunks that a transposing read takes of 8 rows.
#include <type_traits>

#include "dev_common.h"
#include "kernels.h"

namespace cm {

template <int KVT>
__global__ __launch_bounds__(512, 4) void attn_prompt_pair_kernel(AttnPreArgs a_in) {
    constexpr int D = 128, KT = 64, NKS = 4, NTT = 4, NNT = 8, TILE = KT * D, STAGE = 2 * TILE;      // elements
    constexpr float L2E = 1.4426950408889634f;
    AttnPreArgs a = a_in;
    int qt_seg = -1;
    if (a.tiles != nullptr) {         // several sequences: this workgroup's (sequence, query tile), longest first
        const int2 tq = a.tiles[gridDim.y - 1 - blockIdx.y];
        const PrefillSegDev sg = a.segs[tq.x];
        const size_t r0 = (size_t)sg.row0 * a.Hq * D;
        a.S = sg.S; a.start_pos = sg.start_pos; a.block_table += sg.bt_off;
        a.q_hi += r0; a.q_lo += r0; a.out_hi += r0;
        if (a.out_lo != nullptr) a.out_lo += r0;
        if (a.out_f32 != nullptr) a.out_f32 += r0;
        qt_seg = tq.y;
    }
    extern __shared__ __attribute__((aligned(16))) uint16_t ldsp[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = lane & 15, g = lane >> 4;
    const int h = (int)blockIdx.x * 2 + (wave >> 2), kvh = h / a.nrep;
    // (long tiles first, descending, then the short ones ascending: the two workgroups of a CU are a long and a short one)
    const int ny = (int)gridDim.y, yy = (int)blockIdx.y, nlong = (ny + 1) / 2;
    const int qb = (qt_seg >= 0 ? qt_seg : (yy < nlong ? ny - 1 - yy : yy - nlong)) * 64;
    const int qrow = qb + (wave & 3) * 16 + sub, qrow_c = qrow < a.S ? qrow : a.S - 1, qpos = a.start_pos + qrow;
    bf16x8 qh[NKS], ql[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const size_t off = ((size_t)qrow_c * a.Hq + h) * D + ks * 32 + g * 8;
        qh[ks] = *(const bf16x8*)(a.q_hi + off);
        ql[ks] = *(const bf16x8*)(a.q_lo + off);
    }
    f32x4 o[NNT];
    float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
    for (int nt = 0; nt < NNT; ++nt) o[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int last_q = min(qb + 63, a.S - 1), kv_end = a.start_pos + last_q + 1, ntile = (kv_end + KT - 1) / KT;
    const int nfull = (a.start_pos + qb + 1) / KT;          // tiles every query of the block sees completely (and that end before kv_end)
    // page ids of 64 tiles in one register (a page is whole tiles)
    const int tpp = a.page / KT, npg = (kv_end + a.page - 1) / a.page;
    int pgs_grp = 0;
    int pgs = a.block_table[min(lane / tpp, npg - 1)];
    auto tile_base = [&](int t) __attribute__((always_inline)) -> size_t {
        if ((t >> 6) != pgs_grp) {                           // (uniform; every 64 tiles)
            pgs_grp = t >> 6;
            pgs = a.block_table[min((pgs_grp * 64 + lane) / tpp, npg - 1)];
        }
        const int pg = __builtin_amdgcn_readlane(pgs, t & 63);
        return ((size_t)(pg * a.Hkv + kvh) * a.page + (t * KT) % a.page) * (D * 2);
    };
    // requests: a wave's instruction i brings the rows 32 i + 4 wave .. + 3
    const int r0 = wave * 4 + (lane >> 4);
    const uint32_t kchunk = (uint32_t)((lane & 15) ^ (r0 & 15)) << 4, vchunk = (uint32_t)((lane & 15) ^ ((r0 & 7) << 1)) << 4;
    const uint32_t lds0 = (uint32_t)(uintptr_t)ldsp + (uint32_t)wave * 1024u;
    auto ask = [&](int t) __attribute__((always_inline)) {
        const size_t b = tile_base(t);
        const char* const kb = (const char*)a.kpool + b;
        const char* const vb = (const char*)a.vpool + b;
        const uint32_t to = lds0 + (uint32_t)((t & 1) * STAGE) * 2u;
        const int lim = kv_end - 1 - t * KT;                 // rows behind the last key: that one again (what a page holds there may be no number)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t row = (uint32_t)min(32 * i + r0, lim) * (D * 2);
            lds_load16_at(kb, row + kchunk, to + (uint32_t)i * 8192u);
            lds_load16_at(vb, row + vchunk, to + (uint32_t)(TILE * 2 + i * 8192));
        }
    };
    const int vr = (g & 1) * 4 + (sub >> 2);                 // row of the transposing reads, modulo 8
    auto tile = [&](int t, auto masked_c) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked_c)::value;
        const int t0 = t * KT;
        // this wave's rows of the tile are here; behind the barrier all are, and the other stage has been read
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < ntile) ask(t + 1);
        const uint16_t* Kb = ldsp + (t & 1) * STAGE + sub * D;
        const uint16_t* Vb = ldsp + (t & 1) * STAGE + TILE + (g * 4 + (sub >> 2)) * D + (sub & 1) * 4;
        f32x4 s[NTT];
#pragma unroll
        for (int tt = 0; tt < NTT; ++tt) s[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            bf16x8 kh[NTT];
#pragma unroll
            for (int tt = 0; tt < NTT; ++tt) kh[tt] = *(const bf16x8*)&Kb[tt * 16 * D + (((ks * 4 + g) ^ sub) << 3)];
#pragma unroll
            for (int tt = 0; tt < NTT; ++tt) s[tt] = mma_k32<KVT>(kh[tt], qh[ks], s[tt]);
#pragma unroll
            for (int tt = 0; tt < NTT; ++tt) s[tt] = mma_k32<KVT>(kh[tt], ql[ks], s[tt]);
        }
        float mt = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (MASKED) { if (t0 + tt * 16 + g * 4 + r > qpos) s[tt][r] = -INFINITY; }
                mt = fmaxf(mt, s[tt][r]);
            }
        mt = rows_max(mt);
        const float m_new = fmaxf(m_run, mt);               // finite: token 0 is visible to every query
        const float nm = -m_new * L2E;
        float alpha = 1.f;
        if (__any(m_new != m_run)) {                        // (uniform; else every factor is 1)
            alpha = __builtin_amdgcn_exp2f((m_run - m_new) * L2E);
#pragma unroll
            for (int nt = 0; nt < NNT; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[nt][r] *= alpha;
        }
        m_run = m_new;
        float psum = 0.f;
        // O^T += V^T . P^T, the 32 keys of a product two score tiles side by side
#pragma unroll
        for (int tt = 0; tt < NTT; tt += 2) {
            bf16x4 ph[2], pl[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) { p[r] = __builtin_amdgcn_exp2f(fmaf(s[tt + k][r], L2E, nm)); psum += p[r]; }
                p_split4<KVT>(p, ph[k], pl[k]);
            }
            const bf16x8 p8h = __builtin_shufflevector(ph[0], ph[1], 0, 1, 2, 3, 4, 5, 6, 7), p8l = __builtin_shufflevector(pl[0], pl[1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int nt = 0; nt < NNT; ++nt) {
                bf16x4 v2[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint16_t* vp = &Vb[(tt + k) * 16 * D + (((nt ^ vr) * 2 + ((sub & 3) >> 1)) << 3)];
                    v2[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
                }
                const bf16x8 vh = __builtin_shufflevector(v2[0], v2[1], 0, 1, 2, 3, 4, 5, 6, 7);
                o[nt] = mma_k32<KVT>(vh, p8h, o[nt]);
                o[nt] = mma_k32<KVT>(vh, p8l, o[nt]);
            }
        }
        l_run = fmaf(l_run, alpha, psum);
    };
    ask(0);
    int t = 0;
    for (; t < nfull; ++t) tile(t, std::false_type{});
    for (; t < ntile; ++t) tile(t, std::true_type{});       // the diagonal and the ragged end
    float l = l_run;
    l = rows_sum(l);
    if (qrow >= a.S) return;
    const float inv = 1.0f / l;
    const size_t at = ((size_t)qrow * a.Hq + h) * D + g * 4;
#pragma unroll
    for (int nt = 0; nt < NNT; ++nt) {
        const float v[4] = {o[nt][0] * inv, o[nt][1] * inv, o[nt][2] * inv, o[nt][3] * inv};
        if (a.out_f32 != nullptr) *(f32x4*)(a.out_f32 + at + nt * 16) = (f32x4){v[0], v[1], v[2], v[3]};
        else split_store4(a.out_hi, a.out_lo, at + nt * 16, v);
    }
}

// The same for head_dim 256 (the hybrid family's gated attention), at every number of query tiles: four query groups of 16 rows, and the keys of a tile in two halves, each with waves,
// sums and a maximum of its own; the halves meet in the LDS behind the walk.
// What bounds it: the chain of a tile, as above; eight heads of 2048 rows are one query tile per CU, so a kernel of four waves a tile had one wave on a SIMD.  A query group's fragments and sums
// are 128 registers, its tiles 64 KB a stage: eight waves of 256 registers and 128 KB of LDS are what a CU holds.  Behind the chain stands the LDS: every wave reads a fragment for two products.
// Measured (8 heads on 2, us a launch, four waves with tiles through registers / here): 2048 rows 125 / 70, behind 2048 tokens 262 / 145; 69 rows behind 4096 28 / 20 (16 shares).  Prompts of
// Qwen3.5-2B, 31 ... 4165 tokens: 0.8 ... 3.7 % of the whole, none slower.
// LDS: two stages of a key and a value tile of 64 rows of 512 bytes, chunks moved as above.
template <int KVT>
__global__ __launch_bounds__(512, 2) void attn_prompt_wide_kernel(AttnPreArgs a_in) {
    constexpr int D = 256, KT = 64, NKS = 8, NNT = 16, TILE = KT * D, STAGE = 2 * TILE;      // elements
    constexpr float L2E = 1.4426950408889634f;
    AttnPreArgs a = a_in;
    int qt_seg = -1;
    if (a.tiles != nullptr) {         // several sequences: this workgroup's (sequence, query tile), longest first
        const int2 tq = a.tiles[gridDim.y - 1 - blockIdx.y];
        const PrefillSegDev sg = a.segs[tq.x];
        const size_t r0 = (size_t)sg.row0 * a.Hq * D;
        a.S = sg.S; a.start_pos = sg.start_pos; a.block_table += sg.bt_off;
        a.q_hi += r0; a.q_lo += r0; a.out_hi += r0;
        if (a.out_lo != nullptr) a.out_lo += r0;
        if (a.out_f32 != nullptr) a.out_f32 += r0;
        if (a.gate != nullptr) a.gate += (size_t)sg.row0 * a.gate_stride;
        qt_seg = tq.y;
    }
    extern __shared__ __attribute__((aligned(16))) uint16_t ldsp[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2, grp = wave & 3;
    const int sub = lane & 15, g = lane >> 4;
    const int h = (int)blockIdx.x, kvh = h / a.nrep;
    const int qb = (qt_seg >= 0 ? qt_seg : (int)(gridDim.y - 1 - blockIdx.y)) * 64;          // longest first
    const int qrow = qb + grp * 16 + sub, qrow_c = qrow < a.S ? qrow : a.S - 1, qpos = a.start_pos + qrow;
    bf16x8 qh[NKS], ql[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const size_t off = ((size_t)qrow_c * a.Hq + h) * D + ks * 32 + g * 8;
        qh[ks] = *(const bf16x8*)(a.q_hi + off);
        ql[ks] = *(const bf16x8*)(a.q_lo + off);
    }
    f32x4 o[NNT];
    float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
    for (int nt = 0; nt < NNT; ++nt) o[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int last_q = min(qb + 63, a.S - 1), kv_end = a.start_pos + last_q + 1, ntile = (kv_end + KT - 1) / KT;
    const int nfull = (a.start_pos + qb + 1) / KT;          // tiles every query of the block sees completely (and that end before kv_end)
    const int tps = (ntile + a.nsplit - 1) / a.nsplit, tbeg = (int)blockIdx.z * tps, tend = min(ntile, tbeg + tps);      // this share's tiles (may be none)
    // page ids of 64 tiles in one register (a page is whole tiles)
    const int tpp = a.page / KT, npg = (kv_end + a.page - 1) / a.page;
    int pgs_grp = tbeg >> 6;
    int pgs = a.block_table[min((pgs_grp * 64 + lane) / tpp, npg - 1)];
    auto tile_base = [&](int t) __attribute__((always_inline)) -> size_t {
        if ((t >> 6) != pgs_grp) {                           // (uniform; every 64 tiles)
            pgs_grp = t >> 6;
            pgs = a.block_table[min((pgs_grp * 64 + lane) / tpp, npg - 1)];
        }
        const int pg = __builtin_amdgcn_readlane(pgs, t & 63);
        return ((size_t)(pg * a.Hkv + kvh) * a.page + (t * KT) % a.page) * (D * 2);
    };
    // requests: a wave's instruction i brings the rows 16 i + 2 wave and the next
    const int r0 = wave * 2 + (lane >> 5);
    const uint32_t kchunk = (uint32_t)((lane & 31) ^ r0) << 4, vchunk = (uint32_t)((lane & 31) ^ ((r0 & 7) << 1)) << 4;
    const uint32_t lds0 = (uint32_t)(uintptr_t)ldsp + (uint32_t)wave * 1024u;
    auto ask = [&](int t) __attribute__((always_inline)) {
        const size_t b = tile_base(t);
        const char* const kb = (const char*)a.kpool + b;
        const char* const vb = (const char*)a.vpool + b;
        const uint32_t to = lds0 + (uint32_t)((t & 1) * STAGE) * 2u;
        const int lim = kv_end - 1 - t * KT;                 // rows behind the last key: that one again (what a page holds there may be no number)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t row = (uint32_t)min(16 * i + r0, lim) * (D * 2);
            lds_load16_at(kb, row + kchunk, to + (uint32_t)i * 8192u);
            lds_load16_at(vb, row + vchunk, to + (uint32_t)(TILE * 2 + i * 8192));
        }
    };
    const int vr = (g & 1) * 4 + (sub >> 2);                 // row of the transposing reads, modulo 8
    auto tile = [&](int t, auto masked_c) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked_c)::value;
        const int t0 = t * KT + half * 32;
        // this wave's rows of the tile are here; behind the barrier all are, and the other stage has been read
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < tend) ask(t + 1);
        const uint16_t* Kb = ldsp + (t & 1) * STAGE + (half * 32 + sub) * D;
        const uint16_t* Vb = ldsp + (t & 1) * STAGE + TILE + (half * 32 + g * 4 + (sub >> 2)) * D + (sub & 1) * 4;
        f32x4 s[2], u[2];                                    // products with the hi and the lo plane: four chains
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) s[tt] = u[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            bf16x8 kh[2];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) kh[tt] = *(const bf16x8*)&Kb[tt * 16 * D + (((ks * 4 + g) ^ sub) << 3)];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                s[tt] = mma_k32<KVT>(kh[tt], qh[ks], s[tt]);
                u[tt] = mma_k32<KVT>(kh[tt], ql[ks], u[tt]);
            }
        }
        float mt = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[tt][r] += u[tt][r];
                if (MASKED) { if (t0 + tt * 16 + g * 4 + r > qpos) s[tt][r] = -INFINITY; }
                mt = fmaxf(mt, s[tt][r]);
            }
        mt = rows_max(mt);
        const float m_new = fmaxf(m_run, mt);               // (-inf: nothing seen so far, in a half or a share that starts behind the query)
        const float nm = (MASKED && m_new == -INFINITY ? 0.f : -m_new) * L2E;
        float alpha = 1.f;
        if (__any(m_new != m_run)) {                        // (uniform; else every factor is 1)
            alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * L2E);
#pragma unroll
            for (int nt = 0; nt < NNT; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[nt][r] *= alpha;
        }
        m_run = m_new;
        float psum = 0.f;
        // O^T += V^T . P^T, the 32 keys of a product two score tiles side by side
        bf16x4 ph[2], pl[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) { p[r] = __builtin_amdgcn_exp2f(fmaf(s[k][r], L2E, nm)); psum += p[r]; }
            p_split4<KVT>(p, ph[k], pl[k]);
        }
        const bf16x8 p8h = __builtin_shufflevector(ph[0], ph[1], 0, 1, 2, 3, 4, 5, 6, 7), p8l = __builtin_shufflevector(pl[0], pl[1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int n0 = 0; n0 < NNT; n0 += 4) {
            bf16x8 vh[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                bf16x4 v2[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint16_t* vp = &Vb[k * 16 * D + ((((n0 + n) ^ vr) * 2 + ((sub & 3) >> 1)) << 3)];
                    v2[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
                }
                vh[n] = __builtin_shufflevector(v2[0], v2[1], 0, 1, 2, 3, 4, 5, 6, 7);
            }
#pragma unroll
            for (int n = 0; n < 4; ++n) o[n0 + n] = mma_k32<KVT>(vh[n], p8h, o[n0 + n]);
#pragma unroll
            for (int n = 0; n < 4; ++n) o[n0 + n] = mma_k32<KVT>(vh[n], p8l, o[n0 + n]);
        }
        l_run = fmaf(l_run, alpha, psum);
    };
    if (tbeg < tend) ask(tbeg);
    int t = tbeg;
    for (const int mid = min(nfull, tend); t < mid; ++t) tile(t, std::false_type{});
    for (; t < tend; ++t) tile(t, std::true_type{});        // the diagonal and the ragged end
    // the halves of the keys: each wave gives the sums of eight of its sixteen column groups to the other half's wave of the same rows and finishes the other eight
    float l = rows_sum(l_run);
    f32x4* const X = (f32x4*)ldsp;
    float2* const ML = (float2*)(ldsp + 8 * 8 * 64 * 8);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");        // every wave has read its last tile
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) X[(wave * 8 + nt) * 64 + lane] = half ? o[nt] : o[8 + nt];
    ML[wave * 64 + lane] = make_float2(m_run, l);
    __syncthreads();
    if (qrow >= a.S) return;
    const float2 other = ML[(wave ^ 4) * 64 + lane];
    const float M = fmaxf(m_run, other.x), mu = M == -INFINITY ? 0.f : M;
    const float w0 = __builtin_amdgcn_exp2f((m_run - mu) * L2E), w1 = __builtin_amdgcn_exp2f((other.x - mu) * L2E);
    l = fmaf(other.y, w1, l * w0);
    const float inv = a.nsplit > 1 ? 1.f : 1.f / l;
    const size_t row = ((size_t)blockIdx.z * (a.nsplit > 1 ? a.S : 0) + qrow) * a.Hq + h;
    if (a.nsplit > 1 && half == 0 && g == 0) *(float2*)(a.ws + (size_t)a.nsplit * a.S * a.Hq * D + row * 2) = make_float2(M, l);
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        const f32x4 mine = half ? o[8 + nt] : o[nt], his = X[((wave ^ 4) * 8 + nt) * 64 + lane];
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fmaf(his[r], w1, mine[r] * w0) * inv;
        const int col = (half * 8 + nt) * 16 + g * 4;
        const size_t at = row * D + col;
        if (a.nsplit > 1) { *(f32x4*)(a.ws + at) = (f32x4){v[0], v[1], v[2], v[3]}; continue; }       // attn_prefill_merge_kernel takes it from here
        if (a.gate != nullptr) {            // Qwen3.5: y * sigmoid(gate) (qwen3_5/modeling.rs:556-561)
            const f32x4 gv = *(const f32x4*)(a.gate + (size_t)qrow * a.gate_stride + h * D + col);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= 1.0f / (1.0f + expf(-gv[r]));
        }
        if (a.out_f32 != nullptr) *(f32x4*)(a.out_f32 + at) = (f32x4){v[0], v[1], v[2], v[3]};
        else split_store4(a.out_hi, a.out_lo, at, v);
    }
}

void launch_attn_prompt_pair(const AttnPreArgs& a, int kvt, hipStream_t s) {
    constexpr size_t lds = (size_t)2 * 2 * 64 * 128 * sizeof(uint16_t);
    const dim3 grid(a.Hq / 2, a.tiles != nullptr ? a.ntiles : (a.S + 63) / 64);
    if (kvt == KV_F16) hipLaunchKernelGGL(attn_prompt_pair_kernel<KV_F16>, grid, dim3(512), lds, s, a);
    else hipLaunchKernelGGL(attn_prompt_pair_kernel<KV_BF16>, grid, dim3(512), lds, s, a);
}

void launch_attn_prompt_wide(const AttnPreArgs& a, int kvt, hipStream_t s) {
    constexpr size_t lds = (size_t)2 * 2 * 64 * 256 * sizeof(uint16_t);
    static DevOnce attr;
    attr.run([] {
        (void)hipFuncSetAttribute((const void*)attn_prompt_wide_kernel<KV_F16>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        (void)hipFuncSetAttribute((const void*)attn_prompt_wide_kernel<KV_BF16>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    const dim3 grid(a.Hq, a.tiles != nullptr ? a.ntiles : (a.S + 63) / 64, a.nsplit);
    if (kvt == KV_F16) hipLaunchKernelGGL(attn_prompt_wide_kernel<KV_F16>, grid, dim3(512), lds, s, a);
    else hipLaunchKernelGGL(attn_prompt_wide_kernel<KV_BF16>, grid, dim3(512), lds, s, a);
}

}  // namespace cm
