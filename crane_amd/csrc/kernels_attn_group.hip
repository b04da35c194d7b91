// Decode attention of groups of sequences over 16-bit pages, head_dim 128: a block takes one sequence's keys of one key head whole (or one of nsplit shares).
//
// The NREP query heads of the key head are columns of the matrix-core tiles, as in attn_decode_mfma_kernel:
//   S^T[64 tokens x columns] = K Q^T    A = cached key rows straight from the page, 16 bytes per lane; B = the queries
//   O^T[128 x columns]      += V^T P^T  V rows through the wave's own LDS tile, turned by ds_read_b64_tr_b16; P stays in the scores' registers
// Queries and weights keep their 24 bits as three parts in the pages' type, and the parts of up to four heads are columns side by side of one
// product: column c is part c / NREP (mod 4, the fourth is zero) of head c % NREP.  A head's scores are the sum over its columns (two rotations within 16
// lanes), after which each of them forms the weights and keeps its own part.  binary16 parts have 11 bits and little exponent, so a query
// row is scaled by the power of two that takes its largest element to 2^13 and weights by 2^14, both taken out again exactly: the third part ends
// at 2^-38 of the row's largest element.  bfloat16 parts need no scale.
//
// What bounds it: the chain of one wave -- page number, keys, scores, exponentials, weights, values -- and not the bytes.  So a wave takes 64 tokens at a time
// (16 in attn_decode_mfma_kernel: four times the chains), requests the next tile's keys as soon as this one's are multiplied, and every wave of
// the block has tiles of its own; they meet in LDS once.  A sequence whole in a block needs no partial sums in memory; the shares
// of one are merged by the block that arrives last (a launch for that: 4.2 us and its gap; 20 sequences up to 700 tokens, three shares: 19.5 us a layer, 15.9 in one).  The loops over the scores are rolled: unrolled, sixteen expf are longer to fetch than to run.  The key head is the fastest grid dimension: with the
// share there, the shares that short sequences don't have fall on the same XCDs (20 sequences up to 700 tokens, 4 shares: 22.1 us for 17.1).
// Measured (us, with the merging launches there were; attn_decode_split_kernel / attn_decode_mfma_kernel / here; 32 query heads on 8, lengths spread up to the longest; error
// against 64 bits 2.0e-7 / 3.2e-7 / 2.1e-7): 8 sequences up to 1000 tokens 16.9 / 14.7 / 12.6; 20 up to 700 30.8 / 20.1 / 17.1; 32 up to 1000 50.4 / 28.1 /
// 24.0; 64 up to 500 48.7 / 25.6 / 23.0; 128 up to 4000 443 / 249 / 213 (4.9 TB/s).  Three products per tile instead of one with the parts side by side: 20.2
// and 27.4 at the second and third; blocks of eight waves: 17.4 and 24.5, 212 and more at the last.
#include <algorithm>

#include "dev_common.h"
#include "kernels.h"

namespace cm {

namespace {

constexpr int D = 128, KT = 64, QLD = D + 8, VLD = D + 16, NKS = D / 32, NNT = D / 16, VPL = KT * D / 8 / 64;
constexpr int DW = 4;             // waves of a block: two blocks on a CU

template <int KVT> __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    if constexpr (KVT == KV_F16) return __builtin_bit_cast(uint32_t, (cm_f16x2){(_Float16)lo, (_Float16)hi});
    else return pack_bf16x2(lo, hi);
}
// over the four columns NREP apart that hold a head's parts, every one of them gets the same sum
template <int NREP> __device__ __forceinline__ float parts_sum(float v) {
    v += dpp_mov<0x120 + 2 * NREP>(v);        // row_ror
    return v + dpp_mov<0x120 + NREP>(v);
}

// two finished columns of a row: as bfloat16 hi + lo planes where the next product reads those, else f32
__device__ __forceinline__ void put_pair(const AttnDecArgs& a, int bq, int col, float x, float y) {
    if (a.out1_hi) {
        const uint32_t h = pack_bf16x2(x, y);
        *(uint32_t*)(a.out1_hi + (size_t)bq * a.out1_cols + col) = h;
        *(uint32_t*)(a.out1_lo + (size_t)bq * a.out1_cols + col) = pack_bf16x2(x - bf16_lo(h), y - bf16_hi(h));
    } else *(float2*)(a.out1 + (size_t)bq * a.out1_stride + col) = make_float2(x, y);
}
// the Q8_0 block of 32 columns with the largest magnitude am: scale amax / 127 as it is stored (binary16), its inverse for the codes
__device__ __forceinline__ float q8_scale(float am, float& id) {
    const float dq = am / 127.0f;
    id = dq != 0.f ? 1.0f / dq : 0.f;
    return (float)(_Float16)dq;
}

// the shares of a sequence's head merged by one wave, two columns per lane, always in their order
__device__ __forceinline__ void merge_head(const AttnDecArgs& a, int bq, int h, int nh, int nsplit, int shares, int lane) {
    constexpr int AT = 8;                                         // shares requested at once
    const size_t p0 = ((size_t)bq * nh + h) * nsplit;
    const float* po = a.part_o + p0 * D + 2 * lane;
    float2 v[AT];
#pragma unroll
    for (int k = 0; k < AT; ++k) v[k] = get_through(po + (size_t)min(k, shares - 1) * D);
    const float2 ml = get_through(a.part_ml + (p0 + min(lane, shares - 1)) * 2);      // (at most 64 shares)
    const float M = wave_max(ml.x), w = lane < shares ? expf(ml.x - M) : 0.f;
    const float inv = 1.0f / wave_sum(w * ml.y);
    float x = 0.f, y = 0.f;
    for (int k0 = 0; k0 < shares; k0 += AT) {
#pragma unroll
        for (int k = 0; k < AT; ++k) {
            const float wk = __shfl(w, min(k0 + k, 63));          // 0 behind the last share
            x = fmaf(wk, v[k].x, x); y = fmaf(wk, v[k].y, y);
        }
        if (k0 + AT < shares) {
#pragma unroll
            for (int k = 0; k < AT; ++k) v[k] = get_through(po + (size_t)min(k0 + AT + k, shares - 1) * D);
        }
    }
    x *= inv; y *= inv;
    const int col = h * D + 2 * lane;
    if (a.gate) {
        const float2 g = *(const float2*)(a.gate + (size_t)bq * a.qkv_stride + col);
        x *= 1.0f / (1.0f + expf(-g.x)); y *= 1.0f / (1.0f + expf(-g.y));
    }
    put_pair(a, bq, col, x, y);
    if (!a.out1_q) return;
    float id;
    const float dq = q8_scale(row16_max(fmaxf(fabsf(x), fabsf(y))), id);      // 16 lanes: 32 columns
    *(uint16_t*)(a.out1_q + (size_t)bq * a.out1_cols + col) = (uint16_t)(((uint32_t)(int)roundf(x * id) & 0xFFu) | (((uint32_t)(int)roundf(y * id) & 0xFFu) << 8));
    if ((lane & 15) == 0) a.out1_qd[(size_t)(col >> 5) * QGEMM_MAXM + bq] = dq;
}

template <int NREP, int KVT>
__global__ __launch_bounds__(DW * 64, 2) void attn_decode_group_kernel(AttnDecArgs a) {
    constexpr float PUP = KVT == KV_F16 ? 16384.f : 1.f;           // scale of the weights
    extern __shared__ __attribute__((aligned(16))) uint16_t gsm[];
    uint16_t* const Qs = gsm + DW * KT * VLD;                     // [3 parts][NREP][QLD]
    uint16_t* const knew = Qs + 3 * NREP * QLD;                   // [D] this step's key and value, rounded as the pages hold them
    uint16_t* const vnew = knew + D;
    __shared__ float qinv[NREP], red_m[DW][16], red_w[DW][16], red_l[DW][16];
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint16_t* const Vw = gsm + wave * KT * VLD;                   // this wave's tile
    const int kvh = blockIdx.x, bq = blockIdx.y, split = blockIdx.z, nsplit = gridDim.z;
    const StepState* st = a.st + bq;
    const int32_t* bt = a.block_table + (size_t)bq * a.bt_stride;
    const float* qkv = a.qkv + (size_t)bq * a.qkv_stride;
    const int pos = st->pos, rpos = pos + st->rsv[0];
    const int psh = __builtin_ctz(a.page), ntile = pos / KT + 1;  // (page: a power of two and whole tiles) tokens 0 .. pos, the last one this step's own
    const int shares = min(nsplit, (ntile + DW - 1) / DW);        // blocks that this sequence keeps busy
    if (split >= shares) return;
    const int t_first = split * DW + wave, t_step = DW * nsplit;
    const bool owner = (ntile - 1) / DW % nsplit == split;        // appends this step's token

    int pgs_grp = 0;                                              // lane i: page of this wave's tile 64 grp + i
    auto load_pages = [&](int grp) __attribute__((always_inline)) { return bt[(min(t_first + (grp * 64 + lane) * t_step, ntile - 1) * KT) >> psh]; };
    int pgs = load_pages(0);
    auto base_of = [&](int i, int t) __attribute__((always_inline)) {
        if ((i >> 6) != pgs_grp) { pgs_grp = i >> 6; pgs = load_pages(pgs_grp); }      // (uniform)
        return ((size_t)(__builtin_amdgcn_readlane(pgs, i & 63) * a.Hkv + kvh) * a.page + (t * KT & (a.page - 1))) * D;
    };
    u32x4 kr[4][NKS], vr[VPL];
    // rows behind the cached ones repeat the last of them (row 0 of a tile that has none: in the page, and replaced by knew / vnew below)
    auto fetch_k = [&](int i) __attribute__((always_inline)) {
        const int t = t_first + i * t_step;
        if (t >= ntile) return;                                   // (uniform)
        const uint16_t* kp = (const uint16_t*)a.kpool + base_of(i, t);
        const int last = max(pos - 1 - t * KT, 0);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) kr[tt][ks] = ld16(kp + (uint32_t)(min(tt * 16 + lr, last) * D + lg * 8) + ks * 32);
    };
    auto fetch_v = [&](int i) __attribute__((always_inline)) {
        const int t = t_first + i * t_step;
        if (t >= ntile) return;
        const uint16_t* vp = (const uint16_t*)a.vpool + base_of(i, t);
        const int last = max(pos - 1 - t * KT, 0);
#pragma unroll
        for (int k = 0; k < VPL; ++k) vr[k] = ld16(vp + (uint32_t)(min(lg + k * 4, last) * D + lr * 8));
    };
    // ---- the heads' queries (norm, rotation, 1 / sqrt(D), three parts), this step's key and value (the owner appends them).  Everything they need is
    // requested in front of the first tile: answers come in order, so none of it waits for the tile
    constexpr int IT = (NREP + 2 + DW - 1) / DW;
    float x0[IT], x1[IT], n0[IT], n1[IT], p0[IT][7], p1[IT][7];
    const float c = a.cos[(size_t)rpos * 64 + lane], sn = a.sin[(size_t)rpos * 64 + lane];
    auto source = [&](int item) __attribute__((always_inline)) { return qkv + (item < NREP ? a.q_off + (kvh * NREP + item) * D : (item == NREP ? a.k_off : a.v_off) + kvh * D); };
#pragma unroll
    for (int k = 0; k < IT; ++k) {
        const int item = min(wave + k * DW, NREP + 1);
        const float* src = source(item);
        const float* nw = item < NREP ? a.qnw : item == NREP ? a.knw : nullptr;
        x0[k] = src[lane]; x1[k] = src[lane + 64];
        n0[k] = nw ? nw[lane] : 1.f; n1[k] = nw ? nw[lane + 64] : 1.f;
    }
    if (a.qkv_ns > 1) {                                           // slices of a product whose depth is split (2 .. 8), added in their order below
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            const float* src = source(min(wave + k * DW, NREP + 1));
#pragma unroll
            for (int sl = 1; sl < 8; ++sl) {
                const float* ps = src + (size_t)(sl < a.qkv_ns ? sl : 0) * a.qkv_slice;
                p0[k][sl - 1] = ps[lane]; p1[k][sl - 1] = ps[lane + 64];
            }
        }
    }
    fetch_k(0);
    fetch_v(0);
    // (the sums behind every request: with an item's in front of the next one's the first keys were asked for two trips to memory later)
    if (a.qkv_ns > 1) {
#pragma unroll
        for (int k = 0; k < IT; ++k)
#pragma unroll
            for (int sl = 1; sl < 8; ++sl)
                if (sl < a.qkv_ns) { x0[k] += p0[k][sl - 1]; x1[k] += p1[k][sl - 1]; }
    }
#pragma unroll
    for (int k = 0; k < IT; ++k) {
        const int item = wave + k * DW;
        if (item >= NREP + 2) break;
        float y0 = x0[k], y1 = x1[k];
        if ((item < NREP ? a.qnw : item == NREP ? a.knw : nullptr) != nullptr) {
            const float rr = 1.0f / sqrtf(wave_sum(y0 * y0 + y1 * y1) / (float)D + a.eps);
            y0 = y0 * rr * n0[k]; y1 = y1 * rr * n1[k];
        }
        if (item <= NREP) {                                       // rotate-half: element i with element i + D / 2, both in this lane
            const float lo = y0, hi = y1;
            y0 = lo * c - hi * sn;
            y1 = lo * sn + hi * c;
        }
        if (item < NREP) {
            y0 *= a.scale; y1 *= a.scale;
            if (KVT == KV_F16) {                                  // largest element to 2^13 (infinities and NaN pass through unscaled)
                const uint32_t E = __float_as_uint(wave_max(fmaxf(fabsf(y0), fabsf(y1)))) >> 23;
                const uint32_t f = E == 255u ? 127u : min(267u - E, 253u);
                const float up = __uint_as_float(f << 23);
                if (lane == 0) qinv[item] = __uint_as_float((254u - f) << 23);
                y0 *= up; y1 *= up;
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const uint32_t pk = pack2<KVT>(y0, y1);
                y0 -= kv16_lo<KVT>(pk); y1 -= kv16_hi<KVT>(pk);
                Qs[(q * NREP + item) * QLD + lane] = (uint16_t)(pk & 0xFFFFu);
                Qs[(q * NREP + item) * QLD + lane + 64] = (uint16_t)(pk >> 16);
            }
        } else {
            uint16_t* dst = item == NREP ? knew : vnew;
            const uint16_t b0 = kv16_from_f32<KVT>(y0), b1 = kv16_from_f32<KVT>(y1);
            dst[lane] = b0; dst[lane + 64] = b1;
            if (owner) {
                uint16_t* row = (uint16_t*)(item == NREP ? a.kpool : a.vpool) + ((size_t)(bt[pos >> psh] * a.Hkv + kvh) * a.page + (pos & (a.page - 1))) * D;
                row[lane] = b0; row[lane + 64] = b1;
            }
        }
    }
    __syncthreads();

    const int head = lr % NREP, part = lr / NREP & 3;             // this lane's column
    const float qi = KVT == KV_F16 ? qinv[head] : 1.f, pup = part < 3 ? PUP : 0.f;
    bf16x8 qf[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        u32x4 v = *(const u32x4*)&Qs[(min(part, 2) * NREP + head) * QLD + ks * 32 + lg * 8];
        if (part == 3) v = (u32x4){0u, 0u, 0u, 0u};
        qf[ks] = __builtin_bit_cast(bf16x8, v);
    }
    float m = -INFINITY, l = 0.f;
    f32x4 o[NNT];
#pragma unroll
    for (int n = 0; n < NNT; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int i = 0, t = t_first; t < ntile; ++i, t += t_step) {
        const int own = pos - t * KT;                             // row of this step's token, past the tile for all but the last
        if (own < KT) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks)
                    if (tt * 16 + lr >= own) kr[tt][ks] = *(const u32x4*)&knew[ks * 32 + lg * 8];
#pragma unroll
            for (int k = 0; k < VPL; ++k)
                if (lg + k * 4 >= own) vr[k] = *(const u32x4*)&vnew[lr * 8];
        }
        f32x4 s[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) s[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) s[tt] = mma_k32<KVT>(__builtin_bit_cast(bf16x8, kr[tt][ks]), qf[ks], s[tt]);
        fetch_k(i + 1);
#pragma unroll
        for (int k = 0; k < VPL; ++k) *(u32x4*)&Vw[(lg + k * 4) * VLD + lr * 8] = vr[k];
        fetch_v(i + 1);
        float mt = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {                         // scores of keys 16 tt + 4 lg + r
                const float sc = parts_sum<NREP>(s[tt][r]) * qi;
                s[tt][r] = tt * 16 + lg * 4 + r <= own ? sc : -INFINITY;
                mt = fmaxf(mt, s[tt][r]);
            }
        mt = rows_max(mt);
        const float mn = fmaxf(m, mt);
        const float corr = expf(m - mn);
        l *= corr;
#pragma unroll
        for (int n = 0; n < NNT; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[n][r] *= corr;
        m = mn;
        bf16x8 p[2];
        p[1] = __builtin_bit_cast(bf16x8, (u32x4){0u, 0u, 0u, 0u});
#pragma unroll 1
        for (int h = 0; h < 2; ++h) {                             // p[h]: this lane's part for keys 32 h + 4 lg + 0 .. 3, then 32 h + 16 + 4 lg + 0 .. 3
            u32x4 pk;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float p0 = expf(s[q >> 1][2 * (q & 1)] - mn), p1 = expf(s[q >> 1][2 * (q & 1) + 1] - mn);
                l += p0 + p1;
                p0 *= pup; p1 *= pup;
#pragma unroll
                for (int k = 0; k < 2; ++k) {                     // what the parts in front of this one leave
                    const uint32_t f = pack2<KVT>(p0, p1);
                    p0 -= part > k ? kv16_lo<KVT>(f) : 0.f; p1 -= part > k ? kv16_hi<KVT>(f) : 0.f;
                }
                pk[q] = pack2<KVT>(p0, p1);
            }
            p[0] = p[1]; p[1] = __builtin_bit_cast(bf16x8, pk);
            s[0] = s[2]; s[1] = s[3];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // the wave's own tile is in LDS
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int n = 0; n < NNT; ++n) {
                bf16x4 v2[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint16_t* vp = &Vw[((2 * h + k) * 16 + lg * 4 + (lr >> 2)) * VLD + n * 16 + (lr & 3) * 4];
                    v2[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
                }
                const bf16x8 vf = __builtin_shufflevector(v2[0], v2[1], 0, 1, 2, 3, 4, 5, 6, 7);
                o[n] = mma_k32<KVT>(vf, p[h], o[n]);
            }
    }
    l = rows_sum(l);
    if (lg == 0) red_m[wave][lr] = m;
    __syncthreads();                                              // every wave's tile has been read: its place holds the sums
#pragma unroll
    for (int n = 0; n < NNT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][r] = parts_sum<NREP>(o[n][r]);
    float* po = (float*)gsm;                                      // [wave][NNT][4 lg][NREP][4]
    if (lr < NREP) {
#pragma unroll
        for (int n = 0; n < NNT; ++n) *(f32x4*)&po[(((wave * NNT + n) * 4 + lg) * NREP + lr) * 4] = o[n];
    }
    float M = -INFINITY, L = 0.f, cw[DW];
#pragma unroll
    for (int k = 0; k < DW; ++k) M = fmaxf(M, red_m[k][lr]);
    if (lg == 0) {                                                // a wave without a tile: weight 0
        const float w = m == -INFINITY ? 0.f : expf(m - M);
        red_w[wave][lr] = w; red_l[wave][lr] = w * l;
    }
    __syncthreads();
    if (shares == 1 && lr >= NREP) return;
#pragma unroll
    for (int k = 0; k < DW; ++k) { cw[k] = red_w[k][lr]; L += red_l[k][lr]; }
    const int hq = kvh * NREP + lr;
    const float inv = shares == 1 ? 1.0f / L : 1.f;
    for (int b = wave; b < NNT / 2 && lr < NREP; b += DW) {       // 32 columns: two tiles of sixteen
        f32x4 v[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            v[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < DW; ++k) {
                const f32x4 pk = *(const f32x4*)&po[(((k * NNT + b * 2 + j) * 4 + lg) * NREP + lr) * 4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[j][r] = fmaf(pk[r], cw[k], v[j][r]);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) v[j][r] *= inv * (1.f / PUP);
        }
        if (shares > 1) {
            const size_t ph = ((size_t)bq * a.Hkv * NREP + hq) * nsplit + split;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; r += 2) put_through(a.part_o + ph * D + (b * 2 + j) * 16 + lg * 4 + r, v[j][r], v[j][r + 1]);
            if (b == 0 && lg == 0) put_through(a.part_ml + ph * 2, M, L);
            continue;
        }
        float am = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = hq * D + (b * 2 + j) * 16 + lg * 4;
            if (a.gate) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[j][r] *= 1.0f / (1.0f + expf(-a.gate[(size_t)bq * a.qkv_stride + col + r]));
            }
            put_pair(a, bq, col, v[j][0], v[j][1]);
            put_pair(a, bq, col + 2, v[j][2], v[j][3]);
#pragma unroll
            for (int r = 0; r < 4; ++r) am = fmaxf(am, fabsf(v[j][r]));
        }
        if (!a.out1_q) continue;
        am = rows_max(am);
        float id;
        const float dq = q8_scale(am, id);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t c = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) c |= ((uint32_t)(int)roundf(v[j][r] * id) & 0xFFu) << (8 * r);
            *(uint32_t*)(a.out1_q + (size_t)bq * a.out1_cols + hq * D + (b * 2 + j) * 16 + lg * 4) = c;
        }
        if (lg == 0) a.out1_qd[(size_t)(hq * (D / 32) + b) * QGEMM_MAXM + bq] = dq;
    }
    if (shares == 1) return;
    // the last share to arrive merges them (a launch for it: 4 us and the gap in front of it)
    __shared__ int last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int32_t* done = a.done + (size_t)bq * a.Hkv + kvh;
    if (threadIdx.x == 0) last = atomicAdd(done, 1) == shares - 1;
    __syncthreads();
    if (!last) return;
    if (threadIdx.x == 0) __hip_atomic_store(done, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int k = wave; k < NREP; k += DW) merge_head(a, bq, kvh * NREP + k, a.Hkv * NREP, nsplit, shares, lane);
}

template <int NREP, int KVT>
void go(const AttnDecArgs& a, int nsplit, int n_seq, hipStream_t s) {
    constexpr size_t lds = (size_t)(DW * KT * VLD + 3 * NREP * QLD + 2 * D) * sizeof(uint16_t);
    static_assert((size_t)DW * NNT * 4 * NREP * 4 * sizeof(float) <= (size_t)DW * KT * VLD * sizeof(uint16_t), "the waves' sums");
    static DevOnce attr;
    attr.run([&] { (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_decode_group_kernel<NREP, KVT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
    hipLaunchKernelGGL((attn_decode_group_kernel<NREP, KVT>), dim3((unsigned)a.Hkv, (unsigned)n_seq, (unsigned)nsplit), dim3(DW * 64), lds, s, a);
}
}  // namespace

bool attn_decode_group_fits(int head_dim, int nrep, int kv_mode, int page, int rot_dim) {
    return head_dim == D && rot_dim == D && (kv_mode == KV_F16 || kv_mode == KV_BF16) && page >= KT && (page & (page - 1)) == 0 &&
           (nrep == 1 || nrep == 2 || nrep == 4);
}

// Whether a group is this kernel's.  For it: every wave has 64 tokens, so few launches' blocks are short of work; the slices of a split qkv product are added here, a
// launch less.  Against it: parts for four heads whatever NREP is, and the merging (a launch of 4 us when these were measured, about 2 inside the
// kernel now) where a sequence is more than four tiles.  us a layer (width 1024, 32 query
// heads on 8 unless said; qkv product, attention, o_proj, feed-forward), older kernels / this one, lengths spread up to the longest:
//   slices to add: 9 sequences up to 300 / 700 / 4000 tokens 50.4 / 48.2, 54.9 / 47.9, 64.2 / 59.5; 16 up to 400 54.5 / 48.5; 8 heads on 2, 9 up to 200 / 1000 / 4000
//     42.2 / 38.4, 44.7 / 43.7, 48.6 / 47.9, 16 up to 300 45.0 / 44.2; 4 on 1, 33 up to 300 45.1 / 45.2; 16 on 8, 9 up to 200 / 300 / 400 44.0 / 42.2, 45.1 / 46.0, 45.7 / 45.7,
//     16 up to 300 47.8 / 46.6; 8 on 8, 9 up to 200 / 300 / 700 40.1 / 39.2, 41.0 / 43.1, 44.9 / 43.5, 16 up to 300 / 400 43.6 / 44.0, 45.6 / 44.4, 33 up to 300 57.9 / 48.8
//   none: 2 .. 8 sequences up to 200 39.3 / 37.9 .. 54.8 / 52.6, 8 up to 250 55.0 / 55.7; 3 / 6 / 8 up to 300 49.9 / 51.8, 53.9 / 55.3, 55.7 / 56.2; 5 / 6 / 8 up to 500 54.3 /
//     54.8, 55.1 / 55.2, 57.1 / 56.1, up to 1000 55.3 / 54.9, 56.0 / 55.4, 57.3 / 56.4, 6 / 7 / 8 up to 1500 57.5 / 56.0, 58.6 / 59.6, 59.6 / 60.5, 5 / 6 / 8
//     up to 4000 64.2 / 65.2, 65.6 / 65.9, 68.6 / 70.2; 16 heads on 8, 6 up to 100 / 200 46.9 / 46.5, 46.5 / 47.4; 8 on 8, 6 up to 100 43.7 / 44.2
bool attn_decode_group_pays(int pairs, int nrep, int64_t longest, bool slices, int num_cu) {
    const int heads = pairs * nrep;
    if (pairs >= num_cu) return true;
    if (slices) return heads > 160 || longest <= 200 || longest > 448;
    if (nrep == 4) return heads >= 512 || longest <= 200 || (pairs >= 48 && longest > 448 && longest <= 1024);
    return nrep == 2 && longest <= 128;
}

// shares of a sequence, given the tokens of the longest and the (sequence, key head) pairs: a tile per wave, as far as that makes two blocks per CU; pairs that
// fill the chip by themselves are taken whole, and half as many where two shares would do (32 sequences up to 1000 tokens in 1 / 2 / 4 shares merged by the last: 24.6 / 25.6 / 27.3 us:
// all blocks ask for their first tiles at once, and the memory takes as long for them either way).  us with merging launches, 1 / 2 / 3 / 4 / 8 shares:
// 8 sequences up to 1000 tokens 19.6 / 16.3 / 16.5 / 12.6 / -, up to 4000 58.7 / 37.7 / 31.1 / 26.0 / 25.8; 20 up to 500 14.4 / 15.3, up to 700 17.8 / 17.7 /
// 17.1, up to 1000 22.2 / 24.5 / 21.8 / 19.6, up to 4000 61.7 / 63.1 / 50.8 / 53.5 / 51.1; 32 up to 2000 38.7 / 43.3 / 43.0 / 42.2 / 41.8 -- lengths spread evenly.
// One long context beside short ones (100 tokens) would like more: us a layer, the kernels that single sequences use / 1 / 2 / 4 / 8 / 16 shares, 32 sequences with one of 1000
// 65.7 / 59.7 / 61.5 / 56.2 / 56.2 / 56.4, of 4000 97.9 / 95.3 / 95.6 / 72.1 / 61.1 / 64.0; 64 with one of 4000 145.7 / 102.8 / 89.4 / 84.0 / 78.6 / 73.9
int attn_decode_group_split(int64_t longest, int pairs, int num_cu, int most) {
    const int64_t tiles = (longest + KT - 1) / KT, want = (tiles + DW - 1) / DW;
    if (pairs >= num_cu || (want == 2 && 2 * pairs > num_cu)) return 1;
    return (int)std::max<int64_t>(1, std::min<int64_t>({want, (2 * num_cu + pairs - 1) / std::max(1, pairs), most, 64}));
}

bool launch_attn_decode_group(const AttnDecArgs& a, int nrep, int kv_mode, int nsplit, int n_seq, hipStream_t s) {
#define CM_GRP(N) case N: if (kv_mode == KV_F16) go<N, KV_F16>(a, nsplit, n_seq, s); else go<N, KV_BF16>(a, nsplit, n_seq, s); return true;
    switch (nrep) {
        CM_GRP(1) CM_GRP(2) CM_GRP(4)
        default: return false;
    }
#undef CM_GRP
}

}  // namespace cm
