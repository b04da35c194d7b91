// Window attention of prompt passes over bfloat16 pages, layer-list decoders (launch_lay_attn_tile): the masks, distance terms, sink,
// block rows and gates of lay_attn_kernel (kernels_layered.hip) for key and value sizes that are multiples of 16 up to 128 and pages of
// whole 64-key tiles.
//
// What bounds it: per 64-key tile and 16 query rows 48 matrix-core instructions (768 cycles), about as many vector cycles for 16 scores
// per lane, and 32 KB of key and value fragments out of LDS.  The layout takes everything else away:
//   * S^T = K Q^T (A = 16 cached key rows, B = 16 queries): a lane holds the scores of ONE query, so running maximum and sum are one
//     number per lane and the weights leave the scores' registers as the B operand of O^T += V^T P^T: no pass of the weights through
//     LDS, no transposed copy of the values (ds_read_b64_tr_b16 turns the row-major tile), 16-byte LDS stores only.
//   * the 32 keys of one P V product are two 16-key score tiles side by side (the k index of a product is any order the two operands agree
//     on), so both products run on the 32-deep instruction.
//   * a key tile is 64 consecutive positions from a multiple of 64: it lies in one page (one table entry per tile, 64 of them in a
//     register), and only tiles on the edge of somebody's mask are masked.
//   * rows are staged once per block, two LDS buffers, requested two tiles ahead, one barrier per tile.
// Measured (us per launch): 2048 tokens, 32 query heads of 128 on 8 key heads, causal: 106 (325 TFLOP/s; the form with transposed stores and
// the weights through LDS: 1590); a mixed batch of 24 single tokens and 300 prompt rows, 8 heads on 2, window 1024: 27 (174).  Blocks of
// 128 rows (two query groups per wave, half the fragment reads per product): 100 at the first size, 3 % slower at 1024 tokens; not kept.
// Rounding points are the older form's: q rounded to bfloat16 once, scores, running maximum / sum and weights f32, the weights as a
// bfloat16 hi + lo pair (two products), exp2 and log on the hardware units.
#include <algorithm>

#include "dev_common.h"
#include "kernels.h"
#include "layered.h"

namespace cm {

namespace {

constexpr int KT = 64;
constexpr float L2E = 1.4426950408889634f;

__device__ __forceinline__ void lds_barrier() {        // LDS hand-off only: requests for later tiles stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// DP / EP: key / value size the registers and LDS rows are laid out for (64 or 128; the key rows' padding is zero).  A block takes 64 query
// rows, 16 per wave, row qi = (position in the portion) * nrep + (query head in the group).  POOL: the walk starts with the mean rows of
// position blocks.
template <int DP, int EP, bool POOL>
__global__ __launch_bounds__(256, 2) void lay_attn_tile_kernel(LAttnArgs a, bool qvec, bool ovec) {
    constexpr int KLD = DP + 8, VLD = EP + 16, NKS = DP / 32, NNT = EP / 16;
    constexpr int KC = DP / 8, VC = EP / 8, KPT = KT * KC / 256, VPT = KT * VC / 256;   // 16-byte chunks per row / per thread
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    uint16_t* const Ks = smem;                         // [2][64][KLD]
    uint16_t* const Vs = smem + 2 * KT * KLD;          // [2][64][VLD]
    const int g = blockIdx.x;
    const int2 tile_id = a.tiles[blockIdx.y];
    const LaySegDev sg = a.segs[tile_id.x];
    const int nrep = a.H / a.G, d = a.d, e = a.e;
    const int q0 = tile_id.y, nq = min(64, sg.n * nrep - q0);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lg = lane >> 4;
    const int win = (int)min(a.win, 1ll << 30), keep = (int)min(a.keep, 1ll << 30), chunk = (int)min(a.chunk, 1ll << 30);
    const int pool = POOL ? (int)min(a.pool, 1ll << 30) : 0;

    const int qr = wave * 16 + lr;
    const bool qok = qr < nq;
    const int qi = q0 + (qok ? qr : 0), lp = qi / nrep, qhead = g * nrep + (qi - lp * nrep), qrow = sg.row0 + lp;
    const int qpos = qok ? sg.start_pos + lp : -1;     // -1: sees nothing where masks are applied
    const int qclo = chunk > 0 && qok ? qpos / chunk * chunk : 0;
    const float r1 = a.bias != LBIAS_NONE ? a.r1[qhead] * L2E : 0.f, r2 = a.bias == LBIAS_LOG ? a.r2[qhead] : 0.f;
    float m = -INFINITY, l = 0.f;
    if (a.sink && qok) { m = a.sink[qhead] * L2E; l = lg == 0 ? 1.f : 0.f; }       // the four lane groups' sums meet at the end
    bf16x8 qf[NKS];
    const float* src = a.proj + (size_t)qrow * a.ldp + a.q_off + qhead * d;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const int c = ks * 32 + lg * 8;
        u32x4 pk = {0u, 0u, 0u, 0u};
        if (qok && c < d) {
            float x[8];
            if (qvec) {
                const f32x4 x0 = *(const f32x4*)(src + c), x1 = *(const f32x4*)(src + c + 4);
#pragma unroll
                for (int i = 0; i < 4; ++i) { x[i] = x0[i]; x[4 + i] = x1[i]; }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = src[c + i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) pk[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
        }
        qf[ks] = __builtin_bit_cast(bf16x8, pk);
    }
    // the key walk: `front` tiles of block rows (POOL) or of the kept first tokens that lie in front of the window's first tile, then the
    // window from a multiple of 64 on
    const int pmin = sg.start_pos + q0 / nrep, pmax = sg.start_pos + (q0 + nq - 1) / nrep;
    int main_lo = max(0, pmin - win + 1);
    if (chunk > 0) main_lo = max(main_lo, pmin / chunk * chunk);
    const int main0 = main_lo / KT * KT;
    const int blocks = POOL ? max(0, (pmax - win + 1) / pool) : 0;
    const int front = POOL ? (blocks + KT - 1) / KT : min((keep + KT - 1) / KT, main0 / KT);
    const int ntile = front + (pmax - main0) / KT + 1;
    const int vis_lo = max(pmax - win + 1, chunk > 0 ? pmax / chunk * chunk : 0);      // everybody sees [vis_lo, pmin]
    auto first_of = [&](int t) __attribute__((always_inline)) { return t < front ? t * KT : main0 + (t - front) * KT; };

    // page of every position tile; lane i holds that of tile 64 grp + i
    int pgs_grp = 0;
    auto load_pages = [&](int grp) __attribute__((always_inline)) {
        const int j = min(first_of(min(grp * 64 + lane, ntile - 1)), pmax);
        return a.bt[sg.bt_off + j / a.page];
    };
    int pgs = load_pages(0);
    struct Rows { u32x4 k[KPT], v[VPT]; };
    const int Gv = a.v_div > 1 ? a.G / a.v_div : a.G, gv = a.v_div > 1 ? g / a.v_div : g;
    auto fetch = [&](int t_, Rows& rg) __attribute__((always_inline)) {
        const int t = min(t_, ntile - 1);              // past the end: the last tile again, parked into a buffer nobody reads
        const int j0 = first_of(t);
        if ((t >> 6) != pgs_grp) { pgs_grp = t >> 6; pgs = load_pages(pgs_grp); }      // (uniform)
        if (POOL && t < front) {
#pragma unroll
            for (int i = 0; i < KPT; ++i) {
                const int idx = tid + 256 * i, b = min(j0 + idx / KC, blocks - 1), c = (idx % KC) * 8;
                const int lpg = (b * pool + pool - 1) / a.page;
                const size_t row = ((size_t)a.bt[sg.bt_off + lpg] * a.G + g) * a.pool_rows + (b - (int)(((long long)lpg * a.page) / pool));
                rg.k[i] = (u32x4){0u, 0u, 0u, 0u};
                if (c < d) rg.k[i] = ld16((const uint16_t*)a.pk_pool + row * d + c);
            }
#pragma unroll
            for (int i = 0; i < VPT; ++i) {
                const int idx = tid + 256 * i, b = min(j0 + idx / VC, blocks - 1), c = (idx % VC) * 8;
                const int lpg = (b * pool + pool - 1) / a.page;
                const size_t row = ((size_t)a.bt[sg.bt_off + lpg] * a.G + g) * a.pool_rows + (b - (int)(((long long)lpg * a.page) / pool));
                rg.v[i] = (u32x4){0u, 0u, 0u, 0u};
                if (c < e) rg.v[i] = a.pv_pool ? ld16((const uint16_t*)a.pv_pool + row * e + c) : ld16((const uint16_t*)a.pk_pool + row * d + c);
            }
            return;
        }
        const int pg = __builtin_amdgcn_readlane(pgs, t & 63), r0 = j0 % a.page, last = pmax - j0;      // rows past the newest position: that one again
        const uint16_t* kp = (const uint16_t*)a.kpool + (((size_t)pg * a.G + g) * a.page + r0) * d;
        const uint16_t* vp = a.vpool ? (const uint16_t*)a.vpool + (((size_t)pg * Gv + gv) * a.page + r0) * e : kp;
        const int ldv = a.vpool ? e : d;
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            const int idx = tid + 256 * i, row = min(idx / KC, last), c = (idx % KC) * 8;
            rg.k[i] = (u32x4){0u, 0u, 0u, 0u};
            if (c < d) rg.k[i] = ld16(kp + (size_t)row * d + c);
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int idx = tid + 256 * i, row = min(idx / VC, last), c = (idx % VC) * 8;
            rg.v[i] = (u32x4){0u, 0u, 0u, 0u};
            if (c < e) rg.v[i] = ld16(vp + (size_t)row * ldv + c);
        }
    };
    auto park = [&](int buf, const Rows& rg) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KPT; ++i) { const int idx = tid + 256 * i; *(u32x4*)&Ks[(buf * KT + idx / KC) * KLD + (idx % KC) * 8] = rg.k[i]; }
#pragma unroll
        for (int i = 0; i < VPT; ++i) { const int idx = tid + 256 * i; *(u32x4*)&Vs[(buf * KT + idx / VC) * VLD + (idx % VC) * 8] = rg.v[i]; }
    };

    f32x4 o[NNT];
#pragma unroll
    for (int n = 0; n < NNT; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const float scale = a.scale * L2E;                 // scores in units of log 2

    auto tile = [&](int t, Rows& rg_new, const Rows& rg_next) __attribute__((always_inline)) {
        fetch(t + 2, rg_new);
        const uint16_t* Kb = Ks + (t & 1) * KT * KLD;
        const uint16_t* Vb = Vs + (t & 1) * KT * VLD;
        f32x4 s[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            s[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const bf16x8 kf = *(const bf16x8*)&Kb[(tt * 16 + lr) * KLD + ks * 32 + lg * 8];
                s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], s[tt], 0, 0, 0);
            }
        }
        const int j0 = first_of(t);
        const bool blk = POOL && t < front;
        const bool full = t >= front && j0 >= vis_lo && j0 + KT - 1 <= pmin;
        float mt = -INFINITY;
        if (full && a.bias == LBIAS_NONE) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) { s[tt][r] *= scale; mt = fmaxf(mt, s[tt][r]); }
        } else {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = j0 + tt * 16 + lg * 4 + r, dist = qpos - j;
                    const bool vis = blk ? j < blocks && (j + 1) * pool <= qpos - win + 1
                                         : dist >= 0 && ((dist < win && j >= qclo) || j < keep);
                    float sc = s[tt][r] * scale;
                    if (!blk) sc -= a.bias == LBIAS_LOG ? r1 * __logf(1.f + r2 * (float)max(dist, 0)) : r1 * (float)dist;
                    s[tt][r] = vis ? sc : -INFINITY;
                    mt = fmaxf(mt, s[tt][r]);
                }
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16));
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float mn = fmaxf(m, mt), ms = mn == -INFINITY ? 0.f : mn;    // nothing seen so far: every weight is exp2(-inf) = 0
        if (__any(mn > m)) {                           // a new maximum somewhere in the wave
            const float corr = __builtin_amdgcn_exp2f(m - ms);
            l *= corr;
#pragma unroll
            for (int n = 0; n < NNT; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[n][r] *= corr;
            m = mn;
        }
        bf16x8 ph[2], pl[2];
        float psum = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 hi, lo;
#pragma unroll
            for (int q = 0; q < 4; ++q) {              // keys 16 (2 h) + 4 lg + {0, 1}, {2, 3}, then 16 (2 h + 1) + ...
                const float p0 = __builtin_amdgcn_exp2f(s[2 * h + (q >> 1)][2 * (q & 1)] - ms);
                const float p1 = __builtin_amdgcn_exp2f(s[2 * h + (q >> 1)][2 * (q & 1) + 1] - ms);
                psum += p0 + p1;
                hi[q] = pack_bf16x2(p0, p1);
                lo[q] = pack_bf16x2(p0 - bf16_lo(hi[q]), p1 - bf16_hi(hi[q]));
            }
            ph[h] = __builtin_bit_cast(bf16x8, hi);
            pl[h] = __builtin_bit_cast(bf16x8, lo);
        }
        l += psum;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int n = 0; n < NNT; ++n) {
                bf16x4 v2[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint16_t* vp = &Vb[((2 * h + k) * 16 + lg * 4 + (lr >> 2)) * VLD + n * 16 + (lr & 3) * 4];
                    v2[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
                }
                const bf16x8 vf = __builtin_shufflevector(v2[0], v2[1], 0, 1, 2, 3, 4, 5, 6, 7);
                o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph[h], o[n], 0, 0, 0);
                o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl[h], o[n], 0, 0, 0);
            }
        park((t + 1) & 1, rg_next);                    // that buffer was last read one tile ago, behind that tile's barrier
        lds_barrier();
    };
    Rows ra, rb;
    fetch(0, ra);
    fetch(1, rb);
    park(0, ra);
    lds_barrier();
    for (int t = 0; t < ntile; t += 2) {
        tile(t, ra, rb);
        if (t + 1 < ntile) tile(t + 1, rb, ra);
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (!qok) return;
    const float* gp = a.gbuf + (size_t)qrow * a.ldg + (a.gate == LGATE_ELEM ? qhead * e : qhead);
    const float inv = (a.gate == LGATE_HEAD ? gp[0] : 1.f) / l * a.out_scale;
    float* out = a.out + (size_t)qrow * a.ldo + qhead * e;
#pragma unroll
    for (int n = 0; n < NNT; ++n) {
        const int c = n * 16 + lg * 4;
        if (c >= e) continue;
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = o[n][r] * inv * (a.gate == LGATE_ELEM ? gp[c + r] : 1.f);
        if (ovec) *(f32x4*)(out + c) = v;
        else {
#pragma unroll
            for (int r = 0; r < 4; ++r) out[c + r] = v[r];
        }
    }
}

template <int DP, int EP, bool POOL>
void go(const LAttnArgs& a, bool qvec, bool ovec, hipStream_t s) {
    constexpr size_t lds = (size_t)2 * KT * (DP + 8 + EP + 16) * sizeof(uint16_t);
    static DevOnce attr;
    attr.run([&] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&lay_attn_tile_kernel<DP, EP, POOL>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    hipLaunchKernelGGL((lay_attn_tile_kernel<DP, EP, POOL>), dim3((unsigned)a.G, (unsigned)a.ntiles), dim3(256), lds, s, a, qvec, ovec);
}
template <int DP, int EP>
void go_sizes(const LAttnArgs& a, bool qvec, bool ovec, hipStream_t s) {
    if (a.pool > 0) go<DP, EP, true>(a, qvec, ovec, s);
    else go<DP, EP, false>(a, qvec, ovec, s);
}

}  // namespace

bool lay_attn_tile_fits(int d, int e, bool own_v, int page) {
    return d > 0 && e > 0 && d % 16 == 0 && e % 16 == 0 && d <= 128 && e <= 128 && (own_v || e <= d) && page % KT == 0;
}

void launch_lay_attn_tile(const LAttnArgs& a0, hipStream_t s) {
    if (a0.ntiles <= 0) return;
    LAttnArgs a = a0;
    if (!a.gbuf) { a.gbuf = a.proj + a.g_off; a.ldg = a.ldp; }
    if (a.e <= 0) a.e = a.d;
    const bool qvec = a.ldp % 4 == 0 && a.q_off % 4 == 0 && ((uintptr_t)a.proj & 15) == 0;
    const bool ovec = a.ldo % 4 == 0 && ((uintptr_t)a.out & 15) == 0;
    if (a.d <= 64) { if (a.e <= 64) go_sizes<64, 64>(a, qvec, ovec, s); else go_sizes<64, 128>(a, qvec, ovec, s); }
    else { if (a.e <= 64) go_sizes<128, 64>(a, qvec, ovec, s); else go_sizes<128, 128>(a, qvec, ovec, s); }
}

}  // namespace cm
