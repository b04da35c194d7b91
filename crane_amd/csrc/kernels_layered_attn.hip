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
// the weights through LDS: 1590); a mixed batch of 24 single tokens and 300 prompt rows, 8 heads on 2, window 1024: 24 (174).  Blocks of
// 128 rows (two query groups per wave, half the fragment reads per product): 100 at the first size, 3 % slower at 1024 tokens; not kept.
// Rounding points are the older form's: q rounded to bfloat16 once, scores, running maximum / sum and weights f32, the weights as a
// bfloat16 hi + lo pair (two products), exp2 and log on the hardware units.
#include <algorithm>

#include "dev_common.h"
#include "kernels.h"
#include "layered.h"
#include "layered_dev.h"

namespace cm {

namespace {

constexpr int KT = 64;
// a decode step whose queries' parts fit side by side (lay_attn_few_kernel)
bool lay_attn_packed(const LAttnArgs& a) { return a.single && a.H <= 4 * a.G; }
// over the four columns of a row of sixteen lanes that are four apart; each of them gets the same sum
__device__ __forceinline__ float parts_sum(float v) {
    v += dpp_mov<0x128>(v);        // row_ror 8
    return v + dpp_mov<0x124>(v);  // row_ror 4
}
constexpr float L2E = 1.4426950408889634f;

__device__ __forceinline__ void lds_barrier() {        // LDS hand-off only: requests for later tiles stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The key walk of query rows [q0, q0 + nq) of a portion: `front` tiles of block rows (POOL) or of the kept first tokens that lie in front of the
// window's first tile, then the window from a multiple of 64 on.
struct Walk : LAttnWalk {                                     // (everybody sees [vis_lo, pmin])
    template <bool POOL>
    __host__ __device__ __forceinline__ void init(const LAttnArgs& a, const LaySegDev& sg, int q0, int nq, int nrep) {
        auto word = [](long long v) { return (int)(v < (1ll << 30) ? v : 1ll << 30); };
        auto lower = [](int x, int y) { return x < y ? x : y; };
        auto upper = [](int x, int y) { return x > y ? x : y; };
        win = word(a.win); keep = word(a.keep); chunk = word(a.chunk);
        pool = POOL ? word(a.pool) : 0;
        pmin = sg.start_pos + q0 / nrep; pmax = sg.start_pos + (q0 + nq - 1) / nrep;
        int main_lo = upper(0, pmin - win + 1);
        if (chunk > 0) main_lo = upper(main_lo, pmin / chunk * chunk);
        main0 = main_lo / KT * KT;
        blocks = POOL ? upper(0, (pmax - win + 1) / pool) : 0;
        front = POOL ? (blocks + KT - 1) / KT : lower((keep + KT - 1) / KT, main0 / KT);
        ntile = front + (pmax - main0) / KT + 1;
        vis_lo = upper(pmax - win + 1, chunk > 0 ? pmax / chunk * chunk : 0);
    }
    __device__ __forceinline__ int first(int t) const { return t < front ? t * KT : main0 + (t - front) * KT; }
};
// cached row of block b's mean (keys' row index; the values' follows the same count)
__device__ __forceinline__ size_t block_row(const LAttnArgs& a, const LaySegDev& sg, int g, int b, int pool) {
    const int lpg = (b * pool + pool - 1) / a.page;
    return ((size_t)a.bt[sg.bt_off + lpg] * a.G + g) * a.pool_rows + (b - (int)(((long long)lpg * a.page) / pool));
}

// elements c .. c + 7 of a query row in f32 (zero outside)
__device__ __forceinline__ void query8(const float* src, int c, int d, bool ok, bool qvec, float (&x)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = 0.f;
    if (!ok || c >= d) return;
    if (qvec) {
        const f32x4 x0 = *(const f32x4*)(src + c), x1 = *(const f32x4*)(src + c + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) { x[i] = x0[i]; x[4 + i] = x1[i]; }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = src[c + i];
    }
}

// a lane's query (column lane % 16 of the transposed scores) and its running softmax.  PARTS: bfloat16 parts of a weight.  Two parts (prompt
// passes): scores in units of log 2, exp2 and log of the hardware units.  Three (decode steps): lay_attn_kernel's functions -- expf, and log1pf,
// which keeps the low bits of a small r2 * distance that 1 + x drops (r1 = 1e6, r2 = 1e-7: weights 5 % off with the hardware's log of 1 + x)
// PACK: column lane % 16 holds part (lane % 16) / 4 (the fourth: nothing) of query min(lane % 4, ..); the scores come as sums over the parts, a lane keeps its
// own part of the weights
template <int PARTS, bool PACK = false>
struct Query {
    static constexpr bool EXACT = PARTS == 3;
    static constexpr int KEPT = PACK ? 1 : PARTS;
    static constexpr float UNIT = EXACT ? 1.f : L2E;
    // the scores' loops take what lies in front and move the rest up: rolled where the functions are long.  A decode launch has about one key tile per
    // wave and waits for its own code: with sixteen expf in a row it is 4 us longer than with sixteen v_exp_f32, with eight in a loop of two 0.9 (8 heads on
    // 2 of 128, context 1000: 13.3 us against 12.4)
    static constexpr int ROLL = EXACT ? 1 : 4;
    static __device__ __forceinline__ float ex(float x) { return EXACT ? expf(x) : __builtin_amdgcn_exp2f(x); }
    bool ok;
    int pos, head, row, clo;
    float r1, r2, m, l;
    // pos -1: sees nothing where masks are applied
    __device__ __forceinline__ void init(const LAttnArgs& a, const LaySegDev& sg, int g, int qr, int q0, int nq, int nrep, int chunk) {
        ok = qr < nq;
        const int qi = q0 + (ok ? qr : 0), lp = qi / nrep;
        head = g * nrep + (qi - lp * nrep);
        row = sg.row0 + lp;
        pos = ok ? sg.start_pos + lp : -1;
        clo = chunk > 0 && ok ? pos / chunk * chunk : 0;
        begin(a);
    }
    // queries of one row in all (LAttnPrep)
    __device__ __forceinline__ void init_alone(const LAttnArgs& a, int g, int j) {
        ok = true; head = g * a.prep.nrep + j; row = 0; pos = a.prep.walk.pmax; clo = a.prep.clo;
        begin(a);
    }
    __device__ __forceinline__ void begin(const LAttnArgs& a) {
        r1 = a.bias != LBIAS_NONE ? a.r1[head] * UNIT : 0.f;
        r2 = a.bias == LBIAS_LOG ? a.r2[head] : 0.f;
        m = -INFINITY; l = 0.f;
    }
    // the wave that starts the running pair from the sink (behind its first requests: the sink's arrival is no reason to hold them back)
    __device__ __forceinline__ void start(const LAttnArgs& a, float sink, int lg, bool first) {
        if (a.sink && ok && first) { m = sink * UNIT; l = lg == 0 ? 1.f : 0.f; }     // the four lane groups' sums meet at the end
    }
    // scores of tile t (products in s, keys 16 tt + 4 lg + r) -> weights in PARTS bfloat16 parts, the running pair moved on, o rescaled when a
    // new maximum appears in the wave.  p[..][h]: keys 16 (2 h) + 4 lg + 0 .. 3, then 16 (2 h + 1) + 4 lg + 0 .. 3
    // TT groups of 16 keys from j0 on, in tile t of the walk
    template <bool POOL, int NNT, int TT>
    __device__ __forceinline__ void weights(const LAttnArgs& a, const Walk& w, int t, int j0, int lg, f32x4 (&s)[TT], bf16x8 (&p)[KEPT][TT / 2], f32x4 (&o)[NNT],
                                            int part_of = 0) {
        const float scale = a.scale * UNIT;
        const bool blk = POOL && t < w.front;
        const bool full = t >= w.front && j0 >= w.vis_lo && j0 + 16 * TT - 1 <= w.pmin;
        float mt = -INFINITY;
        if (full && a.bias == LBIAS_NONE) {
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) { s[tt][r] *= scale; mt = fmaxf(mt, s[tt][r]); }
        } else {
            // (the distance term and the kind of tile are settled outside the loops: a branch per score kept the vector units at a third)
            auto each = [&](auto penalty, auto visible) __attribute__((always_inline)) {
#pragma unroll ROLL
                for (int tt = 0; tt < TT; ++tt) {
                    f32x4 v = s[0];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int j = j0 + tt * 16 + lg * 4 + r, dist = pos - j;
                        const float sc = v[r] * scale - penalty(dist);
                        v[r] = visible(j, dist) ? sc : -INFINITY;
                        mt = fmaxf(mt, v[r]);
                    }
#pragma unroll
                    for (int k = 0; k + 1 < TT; ++k) s[k] = s[k + 1];
                    s[TT - 1] = v;
                }
            };
            // bitwise: no short-circuit branches
            const auto window = [&](int j, int dist) { return (bool)((dist >= 0) & (((dist < w.win) & (j >= clo)) | (j < w.keep))); };
            if (blk) each([](int) { return 0.f; }, [&](int j, int) { return (bool)((j < w.blocks) & ((j + 1) * w.pool <= pos - w.win + 1)); });
            else if (a.bias == LBIAS_NONE) each([](int) { return 0.f; }, window);
            else if (a.bias == LBIAS_LOG) each([&](int dist) {
                const float x = r2 * (float)max(dist, 0);
                return r1 * (EXACT ? log1pf(x) : __logf(1.f + x));
            }, window);
            else each([&](int dist) { return r1 * (float)dist; }, window);
        }
        mt = rows_max(mt);
        const float mn = fmaxf(m, mt), ms = mn == -INFINITY ? 0.f : mn;    // nothing seen so far: every weight is exp(-inf) = 0
        if (__any(mn > m)) {
            const float corr = ex(m - ms);
            l *= corr;
#pragma unroll
            for (int n = 0; n < NNT; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[n][r] *= corr;
            m = mn;
        }
        float psum = 0.f;
#pragma unroll
        for (int k = 0; k < KEPT; ++k) p[k][TT / 2 - 1] = __builtin_bit_cast(bf16x8, (u32x4){0u, 0u, 0u, 0u});
#pragma unroll ROLL
        for (int h = 0; h < TT / 2; ++h) {
            u32x4 part[KEPT];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float p0 = ex(s[q >> 1][2 * (q & 1)] - ms);
                float p1 = ex(s[q >> 1][2 * (q & 1) + 1] - ms);
                psum += p0 + p1;
                if (PACK) {
#pragma unroll
                    for (int k = 0; k < PARTS - 1; ++k) {          // what the parts in front of this lane's leave
                        const uint32_t pk = pack_bf16x2(p0, p1);
                        p0 -= part_of > k ? bf16_lo(pk) : 0.f; p1 -= part_of > k ? bf16_hi(pk) : 0.f;
                    }
                    part[0][q] = part_of < PARTS ? pack_bf16x2(p0, p1) : 0u;
                } else {
#pragma unroll
                    for (int k = 0; k < KEPT; ++k) {
                        const uint32_t pk = pack_bf16x2(p0, p1);
                        part[k][q] = pk;
                        p0 -= bf16_lo(pk); p1 -= bf16_hi(pk);
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < KEPT; ++k) { p[k][0] = p[k][TT / 2 - 1]; p[k][TT / 2 - 1] = __builtin_bit_cast(bf16x8, part[k]); }
            if constexpr (TT == 4) { s[0] = s[2]; s[1] = s[3]; }
        }
        l += psum;
    }
};
// O^T += V^T P^T of one tile from its rows in LDS
template <int VLD, int PARTS, int NNT, int NH>
__device__ __forceinline__ void values(const uint16_t* Vb, int lr, int lg, const bf16x8 (&p)[PARTS][NH], f32x4 (&o)[NNT]) {
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int n = 0; n < NNT; ++n) {
            bf16x4 v2[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint16_t* vp = &Vb[((2 * h + k) * 16 + lg * 4 + (lr >> 2)) * VLD + n * 16 + (lr & 3) * 4];
                v2[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
            }
            const bf16x8 vf = __builtin_shufflevector(v2[0], v2[1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int k = 0; k < PARTS; ++k) o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p[k][h], o[n], 0, 0, 0);
        }
}
__device__ __forceinline__ const float* gate_of(const LAttnArgs& a, int row, int head) { return a.gbuf + (size_t)row * a.ldg + (a.gate == LGATE_ELEM ? head * a.e : head); }
// four output elements c .. c + 3 of a query: v times inv times the gate; head_gate: the gate of the whole head (LGATE_HEAD)
__device__ __forceinline__ void put4(const LAttnArgs& a, int row, int head, int c, const f32x4& o, float l, bool ovec, float head_gate) {
    const float* gp = gate_of(a, row, head);
    const float inv = (a.gate == LGATE_HEAD ? head_gate : 1.f) / l * a.out_scale;
    float* out = a.out + (size_t)row * a.ldo + head * a.e + c;
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = o[r] * inv * (a.gate == LGATE_ELEM ? gp[c + r] : 1.f);
    if (ovec) *(f32x4*)out = v;
    else {
#pragma unroll
        for (int r = 0; r < 4; ++r) out[r] = v[r];
    }
    if (a.out16 == nullptr) return;
    uint16_t* o16 = a.out16 + (size_t)row * a.ldo + head * a.e + c;
    if (ovec) *(u32x2*)o16 = (u32x2){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    else {
#pragma unroll
        for (int r = 0; r < 4; ++r) o16[r] = f32_to_bf16(v[r]);
    }
}

// ---- prompt passes.  DP / EP: key / value size the registers and LDS rows are laid out for (64 or 128).  A block
// takes 64 query rows, 16 per wave, row qi = (position in the portion) * nrep + (query head in the group).  POOL: the walk starts with the mean
// rows of position blocks.  KS: groups of four waves that share the key tiles (each with buffers of its own; their sums meet in LDS)
template <int DP, int EP, bool POOL, int KS>
__global__ __launch_bounds__(256 * KS, KS == 1 ? 2 : 1) void lay_attn_tile_kernel(LAttnArgs a, bool qvec, bool ovec) {
    constexpr int KLD = DP + 8, VLD = EP + 16, NKS = DP / 32, NNT = EP / 16;
    constexpr int KC = DP / 8, VC = EP / 8, KPT = KT * KC / 256, VPT = KT * VC / 256;   // 16-byte chunks per row / per thread
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    const int tid = threadIdx.x & 255, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int grp = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8), wave = tid >> 6;
    uint16_t* const Ks = smem + grp * 2 * KT * (KLD + VLD);       // [2][64][KLD]
    uint16_t* const Vs = Ks + 2 * KT * KLD;                       // [2][64][VLD]
    const int g = blockIdx.x;
    const int2 tile_id = a.tiles[blockIdx.y];
    const LaySegDev sg = a.segs[KS == 2 ? lay_share_seg(tile_id.x) : tile_id.x];
    const int share = KS == 2 ? lay_share_no(tile_id.x) : 0, shares = KS == 2 ? lay_shares(tile_id.x) : 1;
    const int nrep = a.H / a.G, d = a.d, e = a.e;
    const int q0 = tile_id.y, nq = min(64, sg.n * nrep - q0);
    Walk w;
    w.init<POOL>(a, sg, q0, nq, nrep);
    // this block's key tiles [t0, t1)
    const int per = (w.ntile + shares - 1) / shares, t0 = share * per, t1 = min(w.ntile, t0 + per), t_last = min(max(t0, t1 - 1), w.ntile - 1);      // (a share may be empty)
    Query<2> q;
    q.init(a, sg, g, wave * 16 + lr, q0, nq, nrep, w.chunk);
    const float sink = a.sink ? a.sink[q.head] : 0.f;
    const float head_gate = a.gate == LGATE_HEAD ? *gate_of(a, q.row, q.head) : 1.f;       // (here, not behind the walk: a trip to memory less)
    bf16x8 qf[NKS];                                    // rounded once
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        float x[8];
        query8(a.proj + (size_t)q.row * a.ldp + a.q_off + q.head * d, ks * 32 + lg * 8, d, q.ok, qvec, x);
        u32x4 pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
        qf[ks] = __builtin_bit_cast(bf16x8, pk);
    }

    // page of every position tile; lane i holds that of tile 64 grp + i
    int pgs_grp = 0;
    auto load_pages = [&](int grp64) __attribute__((always_inline)) {
        const int j = min(w.first(min(grp64 * 64 + lane, w.ntile - 1)), w.pmax);
        return a.bt[sg.bt_off + j / a.page];
    };
    pgs_grp = t0 >> 6;
    int pgs = load_pages(pgs_grp);
    struct Rows { u32x4 k[KPT], v[VPT]; };
    const int Gv = a.v_div > 1 ? a.G / a.v_div : a.G, gv = a.v_div > 1 ? g / a.v_div : g, ldv = a.vpool ? e : d;
    // this thread's rows and 16-byte column of a tile.  Columns of the padding hold column 0 (their queries' are zero): no load under a branch
    static_assert(256 % KC == 0 && 256 % VC == 0, "one column per thread");
    const int kr0 = tid / KC, vr0 = tid / VC;
    const int kc = (tid % KC) * 8 < d ? (tid % KC) * 8 : 0, vc = (tid % VC) * 8 < e ? (tid % VC) * 8 : 0;
    auto fetch = [&](int t_, Rows& rg) __attribute__((always_inline)) {
        const int t = min(t_, t_last);                 // past the end: the last tile again, parked into a buffer nobody reads
        const int j0 = w.first(t);
        if ((t >> 6) != pgs_grp) { pgs_grp = t >> 6; pgs = load_pages(pgs_grp); }      // (uniform)
        if (POOL && t < w.front) {
            const uint16_t* vpool = a.pv_pool ? (const uint16_t*)a.pv_pool : (const uint16_t*)a.pk_pool;
#pragma unroll
            for (int i = 0; i < KPT; ++i)
                rg.k[i] = ld16((const uint16_t*)a.pk_pool + block_row(a, sg, g, min(j0 + kr0 + i * (256 / KC), w.blocks - 1), w.pool) * d + kc);
#pragma unroll
            for (int i = 0; i < VPT; ++i)
                rg.v[i] = ld16(vpool + block_row(a, sg, g, min(j0 + vr0 + i * (256 / VC), w.blocks - 1), w.pool) * ldv + vc);
            return;
        }
        const int pg = __builtin_amdgcn_readlane(pgs, t & 63), r0 = j0 % a.page, last = w.pmax - j0;   // rows past the newest position: that one again
        const uint16_t* kp = (const uint16_t*)a.kpool + (((size_t)pg * a.G + g) * a.page + r0) * d;
        const uint16_t* vp = a.vpool ? (const uint16_t*)a.vpool + (((size_t)pg * Gv + gv) * a.page + r0) * e : kp;
#pragma unroll
        for (int i = 0; i < KPT; ++i) rg.k[i] = ld16(kp + min(kr0 + i * (256 / KC), last) * d + kc);
#pragma unroll
        for (int i = 0; i < VPT; ++i) rg.v[i] = ld16(vp + min(vr0 + i * (256 / VC), last) * ldv + vc);
    };
    auto park = [&](int buf, const Rows& rg) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KPT; ++i) *(u32x4*)&Ks[(buf * KT + kr0 + i * (256 / KC)) * KLD + (tid % KC) * 8] = rg.k[i];
#pragma unroll
        for (int i = 0; i < VPT; ++i) *(u32x4*)&Vs[(buf * KT + vr0 + i * (256 / VC)) * VLD + (tid % VC) * 8] = rg.v[i];
    };

    f32x4 o[NNT];
#pragma unroll
    for (int n = 0; n < NNT; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // step i: tile KS i + grp of this group; the rows of step i + 2 are requested at its top, those of step i + 1 parked at its bottom
    auto step = [&](int i, Rows& rg_new, const Rows& rg_next) __attribute__((always_inline)) {
        const int t = t0 + KS * i + grp;
        fetch(t + 2 * KS, rg_new);
        if (KS == 1 || t < t1) {                  // (uniform) the last step of an odd walk: the other group's only
            const uint16_t* Kb = Ks + (i & 1) * KT * KLD;
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
            bf16x8 p[2][2];
            q.template weights<POOL>(a, w, t, w.first(t), lg, s, p, o);
            values<VLD>(Vs + (i & 1) * KT * VLD, lr, lg, p, o);
        }
        park((i + 1) & 1, rg_next);                    // that buffer was last read one step ago, behind that step's barrier
        lds_barrier();
    };
    Rows ra, rb;
    fetch(t0 + grp, ra);
    fetch(t0 + grp + KS, rb);
    park(0, ra);
    lds_barrier();
    q.start(a, sink, lg, grp == 0 && share == 0);
    const int steps = (max(0, t1 - t0) + KS - 1) / KS;
    for (int i = 0; i < steps; i += 2) {
        step(i, ra, rb);
        if (i + 1 < steps) step(i + 1, rb, ra);
    }
    float l = q.l, c0 = 1.f;
    l = rows_sum(l);
    if (KS == 2) {                                     // group 1 leaves its sums, group 0 takes them in
        float* po = (float*)smem;                      // [4 waves][NNT][64 lanes][4], then [4 waves][64 lanes] maxima and sums
        float* pm = po + 4 * NNT * 64 * 4;
        if (grp == 1) {
#pragma unroll
            for (int n = 0; n < NNT; ++n) *(f32x4*)&po[((wave * NNT + n) * 64 + lane) * 4] = o[n];
            pm[wave * 64 + lane] = q.m;
            pm[256 + wave * 64 + lane] = l;
        }
        lds_barrier();
        if (grp == 1 && shares == 1) return;
        const float m1 = pm[wave * 64 + lane], l1 = pm[256 + wave * 64 + lane];
        const float mn = fmaxf(q.m, m1), ms = mn == -INFINITY ? 0.f : mn;
        const float c1 = __builtin_amdgcn_exp2f(m1 - ms);
        c0 = __builtin_amdgcn_exp2f(q.m - ms);
        l = l * c0 + l1 * c1;
#pragma unroll
        for (int n = 0; n < NNT; ++n) {
            const f32x4 p = *(const f32x4*)&po[((wave * NNT + n) * 64 + lane) * 4];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[n][r] = o[n][r] * c0 + p[r] * c1;
        }
        if (shares > 1) {                              // (uniform) the last share to arrive adds all of them up, in their order
            __shared__ int last;
            float* const po2 = a.part_o + (size_t)((int)blockIdx.y * a.G + g) * (4 * NNT * 256);
            float* const pm2 = a.part_ml + (size_t)((int)blockIdx.y * a.G + g) * 512;
            if (grp == 0) {
#pragma unroll
                for (int n = 0; n < NNT; ++n)
#pragma unroll
                    for (int r = 0; r < 4; r += 2) put_through(&po2[((wave * NNT + n) * 64 + lane) * 4 + r], o[n][r], o[n][r + 1]);
                put_through(&pm2[(wave * 64 + lane) * 2], mn, l);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            int32_t* const done = a.done + ((int)blockIdx.y - share) * a.G + g;
            if (threadIdx.x == 0) last = atomicAdd(done, 1) == shares - 1;
            __syncthreads();
            if (!last || grp == 1) return;
            if (threadIdx.x == 0) __hip_atomic_store(done, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const size_t stride = (size_t)a.G * (4 * NNT * 256);
            const float* p0 = po2 - share * stride, *m0 = pm2 - (size_t)share * a.G * 512;
            float M = -INFINITY;
            for (int k = 0; k < shares; ++k) M = fmaxf(M, get_through(&m0[(size_t)k * a.G * 512 + (wave * 64 + lane) * 2]).x);
            const float Ms = M == -INFINITY ? 0.f : M;
            l = 0.f;
#pragma unroll
            for (int n = 0; n < NNT; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
            for (int k = 0; k < shares; ++k) {
                const float2 ml = get_through(&m0[(size_t)k * a.G * 512 + (wave * 64 + lane) * 2]);
                f32x4 p[NNT];
#pragma unroll
                for (int n = 0; n < NNT; ++n)
#pragma unroll
                    for (int r = 0; r < 4; r += 2) {
                        const float2 v = get_through(&p0[k * stride + ((wave * NNT + n) * 64 + lane) * 4 + r]);
                        p[n][r] = v.x; p[n][r + 1] = v.y;
                    }
                const float c = __builtin_amdgcn_exp2f(ml.x - Ms);
                l = fmaf(ml.y, c, l);
#pragma unroll
                for (int n = 0; n < NNT; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[n][r] = fmaf(p[n][r], c, o[n][r]);
            }
        }
    }
    if (!q.ok) return;
#pragma unroll
    for (int n = 0; n < NNT; ++n) {
        const int c = n * 16 + lg * 4;
        if (c < e) put4(a, q.row, q.head, c, o[n], l, ovec, head_gate);
    }
}

template <int DP, int EP, bool POOL, int KS>
void go(const LAttnArgs& a, bool qvec, bool ovec, hipStream_t s) {
    constexpr size_t lds = (size_t)KS * 2 * KT * (DP + 8 + EP + 16) * sizeof(uint16_t);
    static_assert(KS == 1 || lds >= (size_t)(4 * (EP / 16) * 64 * 4 + 512) * sizeof(float), "the groups' sums");
    static DevOnce attr;
    attr.run([&] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&lay_attn_tile_kernel<DP, EP, POOL, KS>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    hipLaunchKernelGGL((lay_attn_tile_kernel<DP, EP, POOL, KS>), dim3((unsigned)a.G, (unsigned)a.ntiles), dim3(256 * KS), lds, s, a, qvec, ovec);
}

// ---- decode steps: few query rows (tiles of 16, lay_attn_kernel's), each wave on key tiles of its own.  Keys go from the pages straight into
// fragments, values through a private LDS tile (no barrier inside the walk); a tile's keys are requested as soon as the one before has been
// multiplied, its values as soon as the one before is in LDS.  The eight waves' sums meet in LDS once; gridDim.z > 1: they leave a partial
// sum for lay_attn_merge_kernel instead.  Queries and weights keep their 24 bits, as in lay_attn_kernel: three bfloat16 parts each, three
// products per tile (the launch waits for memory, not for the matrix cores), and its exponential and logarithm.
// For 128 / 128 elements a block's 161 KB of LDS leave one block on a CU; it is ahead of lay_attn_kernel all the same, for any number of sequences.  us a
// step of four layers, lay_attn_kernel / here: 8 heads on 2 of width 1024, 1 / 32 / 128 sequences behind 24 tokens 281 / 256, 514 / 460, 854 / 705,
// behind 1000 tokens 296 / 280, 830 / 525, 2126 / 853; 32 heads on 8 of width 4096, 1 / 32 / 128 sequences behind 24 tokens 515 / 487, 1187 / 1068,
// 1699 / 1552, behind 1000 tokens 536 / 522, 2523 / 1154, 4780 / 1927
// PACK: every sequence has one row and a key head at most four query heads: their parts are columns side by side of one product, as in
// attn_decode_group_kernel, and blocks of four waves fit a CU twice: one sequence behind 1000 tokens, 8 heads on 2, 13.1 -> 10.7 us.
// HALF (one sequence in all): eight waves on halves of tiles, since a wave's chain of requests, scores, weights and sums over a whole one is what the launch takes.
// PREP (HALF, and its projection convolved): convolved q | k | v come from the projection; a wave rotates and scales a query head, and the wave that has the newest tile the key.  That key and
// value take their rows' places in the wave's registers and go to the pages for the next step.
// 8 heads on 2 of 128 behind 1000 tokens, with the convolution's launch: 5.1 + 10.5 us, 10.3 in one (whole tiles 11.3; the walk's divisions on the host, single-byte flags made words and the
// sink's first use behind the first requests: 2.6 us of its chain)
template <int DP, int EP, bool POOL, bool PACK, bool HALF, bool PREP>
__global__ __launch_bounds__(PACK && !HALF ? 256 : 512, PACK && !HALF ? 2 : 1) void lay_attn_few_kernel(LAttnArgs a, bool qvec, bool ovec) {
    constexpr int DW = PACK && !HALF ? 4 : 8, QR = PACK ? 4 : 16, TT = HALF ? 2 : 4, KW = 16 * TT;          // waves, query rows of the tile, keys of a wave's step
    constexpr int QLD = DP + 8, VLD = EP + 16, NKS = DP / 32, NNT = EP / 16, VC = EP / 8, VPL = KW * VC / 64;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    __shared__ float pm[DW][16], pl_[DW][16];
    __shared__ __attribute__((aligned(16))) uint16_t newest[PREP ? DP + EP : 8];
    uint16_t* const Qs = smem + DW * KW * VLD;         // [3 parts][QR][QLD]
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint16_t* const Vw = smem + wave * KW * VLD;       // [KW][VLD] of this wave
    const int g = blockIdx.x;
    const int2 tile_id = PACK ? make_int2((int)blockIdx.y, 0) : a.tiles[blockIdx.y];
    const LaySegDev sg = PREP ? a.prep.seg : a.segs[tile_id.x];
    const int nrep = PREP ? a.prep.nrep : a.H / a.G, d = a.d, e = a.e;
    const int q0 = PREP ? 0 : tile_id.y, nq = PREP ? nrep : min(16, sg.n * nrep - q0);
    Walk w;
    if (PREP) static_cast<LAttnWalk&>(w) = a.prep.walk; else w.init<POOL>(a, sg, q0, nq, nrep);
    auto page_no = [&](int j) __attribute__((always_inline)) { return PREP ? j >> a.prep.page_shift : j / a.page; };
    auto in_page = [&](int j) __attribute__((always_inline)) { return PREP ? j & (a.page - 1) : j % a.page; };
    // steps of KW keys: tile u of the walk, or (HALF) half u & 1 of tile u / 2
    const int t_first = (int)blockIdx.z * DW + wave, t_step = DW * (int)gridDim.z;
    const int steps = HALF ? 2 * w.ntile - (w.pmax - w.first(w.ntile - 1) < 32 ? 1 : 0) : w.ntile;
    auto tile_of = [&](int u) __attribute__((always_inline)) { return HALF ? u >> 1 : u; };
    auto first_of = [&](int u) __attribute__((always_inline)) { return HALF ? w.first(u >> 1) + 32 * (u & 1) : w.first(u); };
    const int part_of = PACK ? lr >> 2 : 0;
    Query<3, PACK> q;
    if (PREP) q.init_alone(a, g, min(lr & 3, nq - 1)); else q.init(a, sg, g, PACK ? min(lr & 3, nq - 1) : lr, q0, nq, nrep, w.chunk);
    const float sink = a.sink ? a.sink[q.head] : 0.f;
    const float head_gate = a.gate == LGATE_HEAD ? *gate_of(a, q.row, q.head) : 1.f;
    // requested in front of the first tile: answers come in order
    float x[8];
    const int t_new = steps - 1;
    const bool has_new = PREP && a.prep.own && t_new >= t_first && (t_new - t_first) % t_step == 0;       // (uniform in the wave)
    float2 qp = make_float2(0.f, 0.f), kp2 = qp, vp2 = qp;
    int e0 = -1, e1 = -1, pg_new = 0;
    float turn = 0.f;
    if (PREP) {                                        // a rotated pair per lane, or two neighbours behind the rotated part
        const int hd = a.prep.dims / 2;
        if (lane < hd) { e0 = 2 * lane; e1 = e0 + 1; turn = a.prep.freq[lane]; }
        else if (a.prep.dims + 2 * (lane - hd) < d) { e0 = a.prep.dims + 2 * (lane - hd); e1 = e0 + 1; }          // (d is even)
        const float* qs = a.proj + a.q_off + (g * nrep + min(wave, nq - 1)) * d, *ks = a.proj + a.prep.k_off + g * d, *vs = a.proj + a.prep.v_off + g * e;
        if (e0 >= 0 && wave < QR) qp = make_float2(qs[e0], qs[e1]);
        if (has_new) {
            if (e0 >= 0) kp2 = make_float2(ks[e0], ks[e1]);
            if (2 * lane < e) vp2 = *(const float2*)(vs + 2 * lane);
            pg_new = a.bt[sg.bt_off + page_no(w.pmax)];
        }
    } else if (wave < NKS) query8(a.proj + (size_t)q.row * a.ldp + a.q_off + q.head * d, wave * 32 + lg * 8, d, q.ok, qvec, x);
    int pgs_grp = 0;                                   // lane i: page of this wave's tile 64 grp + i
    auto load_pages = [&](int grp) __attribute__((always_inline)) {
        const int j = min(first_of(min(t_first + (grp * 64 + lane) * t_step, steps - 1)), w.pmax);
        return a.bt[sg.bt_off + page_no(j)];
    };
    int pgs = load_pages(0);
    const int Gv = a.v_div > 1 ? a.G / a.v_div : a.G, gv = a.v_div > 1 ? g / a.v_div : g;
    u32x4 kr[TT][NKS], vr[VPL];
    auto page_of = [&](int i) __attribute__((always_inline)) {
        if ((i >> 6) != pgs_grp) { pgs_grp = i >> 6; pgs = load_pages(pgs_grp); }      // (uniform)
        return __builtin_amdgcn_readlane(pgs, i & 63);
    };
    auto fetch_k = [&](int i) __attribute__((always_inline)) {
        const int u = t_first + i * t_step, t = tile_of(u);
        if (u >= steps) return;                        // (uniform)
        const int j0 = first_of(u), pg = page_of(i), last = w.pmax - j0;
        const uint16_t* kp = (const uint16_t*)a.kpool + (((size_t)pg * a.G + g) * a.page + in_page(j0)) * d;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            const uint16_t* row = kp + min(tt * 16 + lr, last) * d;
            if (POOL && t < w.front) row = (const uint16_t*)a.pk_pool + block_row(a, sg, g, min(j0 + tt * 16 + lr, w.blocks - 1), w.pool) * d;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) kr[tt][ks] = ld16(row + (ks * 32 + lg * 8 < d ? ks * 32 + lg * 8 : 0));     // no load under a branch
        }
    };
    auto fetch_v = [&](int i) __attribute__((always_inline)) {
        const int u = t_first + i * t_step, t = tile_of(u);
        if (u >= steps) return;
        const int j0 = first_of(u), pg = page_of(i), last = w.pmax - j0, r0 = in_page(j0);
        const uint16_t* vp = a.vpool ? (const uint16_t*)a.vpool + (((size_t)pg * Gv + gv) * a.page + r0) * e
                                     : (const uint16_t*)a.kpool + (((size_t)pg * a.G + g) * a.page + r0) * d;
        const int ldv = a.vpool ? e : d, c = (lane % VC) * 8 < e ? (lane % VC) * 8 : 0;
#pragma unroll
        for (int k = 0; k < VPL; ++k) {
            const int row = lane / VC + k * (64 / VC);
            const uint16_t* src = vp + min(row, last) * ldv;
            if (POOL && t < w.front) {
                const size_t br = block_row(a, sg, g, min(j0 + row, w.blocks - 1), w.pool);
                src = a.pv_pool ? (const uint16_t*)a.pv_pool + br * e : (const uint16_t*)a.pk_pool + br * d;
            }
            vr[k] = ld16(src + c);
        }
    };
    f32x4 o[NNT];
#pragma unroll
    for (int n = 0; n < NNT; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    fetch_k(0);
    fetch_v(0);
    if (PREP) {
        float sn = 0.f, cs = 1.f;
        const int hd = a.prep.dims / 2;
        if ((wave < QR || has_new) && lane < hd) { sincosf((float)w.pmax * turn, &sn, &cs); sn *= a.prep.mag; cs *= a.prep.mag; }
        auto ready = [&](float2 v) __attribute__((always_inline)) {
#pragma clang fp contract(off)                         // (a head times its factor is rounded before it is split)
            if (lane < hd) v = lay_turn(v, cs, sn);
            float ss = fmaf(v.x, v.x, 0.f);
            ss = fmaf(v.y, v.y, ss);
            ss = group_sum(ss, 64);
            const float rs = 1.f / sqrtf(ss / (float)d + a.prep.eps);
            v.x *= rs; v.y *= rs;
            return v;
        };
        if (wave < QR) qp = ready(qp);
#pragma unroll
        for (int k = 0; k < 3 && wave < QR; ++k) {
            uint16_t* qd = &Qs[(k * QR + wave) * QLD];
            const uint32_t pk = pack_bf16x2(qp.x, qp.y);
            if (e0 >= 0) { qd[e0] = (uint16_t)pk; qd[e1] = (uint16_t)(pk >> 16); }
            if (d + lane < DP) qd[d + lane] = 0;
            qp.x -= bf16_lo(pk); qp.y -= bf16_hi(pk);
        }
        if (has_new) {                                 // (read back by this wave alone)
            kp2 = ready(kp2);
            const uint32_t kk = pack_bf16x2(kp2.x, kp2.y), vv = pack_bf16x2(vp2.x, vp2.y);
            const size_t row = ((size_t)pg_new * a.G + g) * a.page + (size_t)in_page(w.pmax);
            if (e0 >= 0) {
                newest[e0] = (uint16_t)kk; newest[e1] = (uint16_t)(kk >> 16);
                uint16_t* to = (uint16_t*)a.kpool + row * d;
                to[e0] = (uint16_t)kk; to[e1] = (uint16_t)(kk >> 16);
            }
            if (d + lane < DP) newest[d + lane] = 0;
            if (2 * lane < EP) *(uint32_t*)&newest[DP + 2 * lane] = 2 * lane < e ? vv : 0u;
            if (2 * lane < e) *(uint32_t*)((uint16_t*)a.vpool + row * e + 2 * lane) = vv;
        }
    } else if (wave < NKS) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            u32x4 pk;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pk[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
                x[2 * i] -= bf16_lo(pk[i]); x[2 * i + 1] -= bf16_hi(pk[i]);
            }
            if (lr < QR) *(u32x4*)&Qs[(k * QR + lr) * QLD + wave * 32 + lg * 8] = pk;
        }
    }
    q.start(a, sink, lg, t_first == 0);
    lds_barrier();
    for (int i = 0, u = t_first; u < steps; ++i, u += t_step) {
        const int t = tile_of(u), j0 = first_of(u);
        if (PREP && has_new && u == t_new) {           // rows from the newest position on (those behind it are masked)
            const int from = w.pmax - j0;
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) {
                    const u32x4 nk = *(const u32x4*)&newest[ks * 32 + lg * 8];
                    if (tt * 16 + lr >= from) kr[tt][ks] = nk;
                }
            const u32x4 nv = *(const u32x4*)&newest[DP + (lane % VC) * 8];
#pragma unroll
            for (int k = 0; k < VPL; ++k)
                if (lane / VC + k * (64 / VC) >= from) vr[k] = nv;
        }
        f32x4 s[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) s[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int k = PACK ? 0 : 2; k >= 0; --k) {  // the smallest part first
                u32x4 qv = *(const u32x4*)&Qs[(PACK ? min(part_of, 2) * QR + (lr & 3) : k * 16 + lr) * QLD + ks * 32 + lg * 8];
                if (PACK && part_of == 3) qv = (u32x4){0u, 0u, 0u, 0u};
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
                    s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kr[tt][ks]), __builtin_bit_cast(bf16x8, qv), s[tt], 0, 0, 0);
            }
        if (PACK) {
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) s[tt][r] = parts_sum(s[tt][r]);
        }
        fetch_k(i + 1);
#pragma unroll
        for (int k = 0; k < VPL; ++k) *(u32x4*)&Vw[(lane / VC + k * (64 / VC)) * VLD + (lane % VC) * 8] = vr[k];
        fetch_v(i + 1);
        bf16x8 p[PACK ? 1 : 3][TT / 2];
        q.template weights<POOL>(a, w, t, j0, lg, s, p, o, part_of);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the wave's own tile is in LDS
        values<VLD>(Vw, lr, lg, p, o);
    }
    float l = q.l;
    l = rows_sum(l);
    if (lg == 0) { pm[wave][lr] = q.m; pl_[wave][lr] = l; }
    __syncthreads();                                   // every wave's value tile has been read: its place holds the sums
    float* po = (float*)smem;                          // [wave][NNT][64 lanes][4]
    if (PACK) {
#pragma unroll
        for (int n = 0; n < NNT; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[n][r] = parts_sum(o[n][r]);
    }
#pragma unroll
    for (int n = 0; n < NNT; ++n) *(f32x4*)&po[((wave * NNT + n) * 64 + lane) * 4] = o[n];
    __syncthreads();
    if (PACK && lr >= nq) return;
    float M = -INFINITY, L = 0.f, cw[DW];
#pragma unroll
    for (int k = 0; k < DW; ++k) M = fmaxf(M, pm[k][lr]);
    const float ms = M == -INFINITY ? 0.f : M;
#pragma unroll
    for (int k = 0; k < DW; ++k) { cw[k] = expf(pm[k][lr] - ms); L = fmaf(pl_[k][lr], cw[k], L); }
    const int nsplit = (int)gridDim.z;
    const size_t pr = (((size_t)blockIdx.y * a.G + g) * nsplit + blockIdx.z) * 16 + lr;
    if (nsplit > 1 && wave == 0 && lg == 0) { a.part_ml[pr * 2] = M; a.part_ml[pr * 2 + 1] = L; }
    for (int n = wave; n < NNT; n += DW) {
        const int c = n * 16 + lg * 4;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < DW; ++k) {
            const f32x4 p = *(const f32x4*)&po[((k * NNT + n) * 64 + lane) * 4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = fmaf(p[r], cw[k], v[r]);
        }
        if (c >= e) continue;
        if (nsplit > 1) {
            *(f32x4*)(a.part_o + pr * e + c) = v;      // (e and c: multiples of 16 and 4)
        } else if (q.ok) put4(a, q.row, q.head, c, v, L, ovec, head_gate);
    }
}
template <int DP, int EP, bool POOL, bool PACK, bool HALF, bool PREP>
void go_few(const LAttnArgs& a, int nsplit, bool qvec, bool ovec, hipStream_t s) {
    constexpr int DW = PACK && !HALF ? 4 : 8, QR = PACK ? 4 : 16;
    constexpr size_t lds = ((size_t)DW * (HALF ? 32 : KT) * (EP + 16) + 3 * QR * (DP + 8)) * sizeof(uint16_t);
    static_assert(lds >= (size_t)DW * (EP / 16) * 64 * 4 * sizeof(float), "the waves' sums");
    static_assert(DP / 32 <= DW, "a wave per 32 elements of the queries");
    static DevOnce attr;
    attr.run([&] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&lay_attn_few_kernel<DP, EP, POOL, PACK, HALF, PREP>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    hipLaunchKernelGGL((lay_attn_few_kernel<DP, EP, POOL, PACK, HALF, PREP>), dim3((unsigned)a.G, (unsigned)a.ntiles, (unsigned)nsplit), dim3(DW * 64), lds, s, a, qvec, ovec);
}
template <int DP, int EP, bool POOL>
void go_few(const LAttnArgs& a, int nsplit, bool qvec, bool ovec, hipStream_t s) {
    if (a.prep.on) go_few<DP, EP, false, true, true, true>(a, nsplit, qvec, ovec, s);      // (lay_attn_prep_fits)
    else if (lay_attn_packed(a) && a.ntiles == 1) go_few<DP, EP, POOL, true, true, false>(a, nsplit, qvec, ovec, s);
    else if (lay_attn_packed(a)) go_few<DP, EP, POOL, true, false, false>(a, nsplit, qvec, ovec, s);
    else go_few<DP, EP, POOL, false, false, false>(a, nsplit, qvec, ovec, s);
}
// nsplit 0: the prompt kernel
template <int DP, int EP>
void go_sizes(const LAttnArgs& a, int nsplit, bool qvec, bool ovec, hipStream_t s) {
    // one block per CU at most: two groups of waves share the key tiles (a mixed batch of 24 single tokens and 300 prompt rows on 8 heads:
    // 24 us against 27); more blocks share the CUs by themselves
    const bool two = a.done != nullptr || (long long)a.ntiles * a.G <= LAY_ATTN_TILE_BLOCKS;      // (shared tiles: this form alone)
    if (nsplit > 0) { if (a.pool > 0) go_few<DP, EP, true>(a, nsplit, qvec, ovec, s); else go_few<DP, EP, false>(a, nsplit, qvec, ovec, s); }
    else if (a.pool > 0) { if (two) go<DP, EP, true, 2>(a, qvec, ovec, s); else go<DP, EP, true, 1>(a, qvec, ovec, s); }
    else { if (two) go<DP, EP, false, 2>(a, qvec, ovec, s); else go<DP, EP, false, 1>(a, qvec, ovec, s); }
}

}  // namespace

// A walk of more than six tiles in shares of `each`, six or what fits the blocks.  A launch of few blocks leaves the chip idle while its longest walk 19 tiles in ten steps; what is left
// with shares is its start, first loads and end.  us a launch, whole / shares of 4 / 6 / 10 (more than 3, 6 and 12 tiles shared: within 3 us of those of 6, either way):
// 24 single tokens and 302 rows behind 0, 302, 605, 907 and 2000 tokens, 8 heads of 128 on 2 20.6 / 17.8 / 19.1 / 19.8, 21.9 / 19.7 / 21.5 / 21.9, 28.1 / 21.6 / 22.9 / 23.2, 32.8 / 23.3 / 23.0 /
// 26.1, 50.2 / 27.8 / 27.7 / 28.4; 64 rows alone behind 500, 1000 and 4000 21.7 / 19.2 / 19.3 / 21.6, 30.0 / 20.8 / 21.0 / 23.5, 79.3 / 31.7 / 28.8 / 29.2; 512 rows behind 1000 and 4000 38.2 / 26.2 / 26.0 /
// 27.2, 88.7 / 39.4 / 39.4 / 39.5; 4 on 1, 32 on 8 and heads of 64 (16 on 4, 16 on 16) alike.  They are looked at while the tiles as a whole fit one round of blocks: up to half of them, as
// long as it was, 60 single tokens and 128 rows behind 1000 on 2 key heads (136 blocks) took 30.8, now 23.2, 24 and 302 on 4 heads of 64 (172) behind 302, 605, 907 and 2000 16.2, 20.1,
// 23.4, 34.5, now 16.6, 18.0, 19.8, 25.5
static int lay_attn_tile_shares(int tiles, int each) { return tiles > 6 ? std::min(127, (tiles + each - 1) / each) : 1; }
int lay_attn_tile_shared(const int2* tiles, int n, const LaySegDev* segs, int nrep, int heads, long long win, int2* out) {
    if (heads <= 0 || (long long)n * heads > LAY_ATTN_TILE_BLOCKS) return 0;
    auto walk = [&](const int2& t) {                   // (of a window alone: first tokens that are kept count as if they lay in front of it)
        const LaySegDev& sg = segs[t.x];
        const long long first = sg.start_pos + t.y / nrep, newest = sg.start_pos + (std::min(t.y + LAY_ATTN_MFMA_ROWS, sg.n * nrep) - 1) / nrep;
        return (int)(newest / KT - std::max(0ll, first - win + 1) / KT + 1);
    };
    int each = 6, total;
    for (;; each += std::max(2, each / 8)) {           // (an eighth at a time where walks are thousands of tiles)
        total = 0;
        for (int i = 0; i < n; ++i) total += lay_attn_tile_shares(walk(tiles[i]), each);
        if (total * heads <= LAY_ATTN_TILE_BLOCKS) break;
    }
    if (total == n) return 0;
    for (int i = 0, at = 0; i < n; ++i)
        for (int k = 0, shares = lay_attn_tile_shares(walk(tiles[i]), each); k < shares; ++k) out[at++] = make_int2(lay_share(tiles[i].x, k, shares), tiles[i].y);
    return total;
}

bool lay_attn_tile_fits(int d, int e, bool own_v, int page) {
    return d > 0 && e > 0 && d % 16 == 0 && e % 16 == 0 && d <= 128 && e <= 128 && (own_v || e <= d) && page % KT == 0;
}

// queries of one row on their way through lay_attn_few_kernel: a wave per query head, a pair of neighbouring elements per lane, heads of unit root mean square, values in pages of their own
bool lay_attn_prep_fits(const LayerSpec& sp, int dims, int page) {
    return sp.unit_qk && !(dims > 0 && sp.rot.half) && sp.pool == 0 && lay_attn_tile_fits(sp.dim, sp.vdim, true, page) && sp.heads <= 4 * sp.kv_heads && sp.heads % sp.kv_heads == 0 &&
           dims % 2 == 0 && dims <= sp.dim && (page & (page - 1)) == 0;
}

static void launch(const LAttnArgs& a0, int nsplit, hipStream_t s) {
    LAttnArgs a = a0;
    if (!a.gbuf) { a.gbuf = a.proj + a.g_off; a.ldg = a.ldp; }
    if (a.e <= 0) a.e = a.d;
    if (a.prep.on) {
        Walk w;
        a.prep.nrep = a.H / a.G;
        w.init<false>(a, a.prep.seg, 0, a.prep.nrep, a.prep.nrep);
        a.prep.walk = w;
        a.prep.clo = w.chunk > 0 ? w.pmax / w.chunk * w.chunk : 0;
        for (a.prep.page_shift = 0; (1 << a.prep.page_shift) < a.page;) ++a.prep.page_shift;
    }
    const bool qvec = a.ldp % 4 == 0 && a.q_off % 4 == 0 && ((uintptr_t)a.proj & 15) == 0;
    const bool ovec = a.ldo % 4 == 0 && ((uintptr_t)a.out & 15) == 0;
    if (a.d <= 64) { if (a.e <= 64) go_sizes<64, 64>(a, nsplit, qvec, ovec, s); else go_sizes<64, 128>(a, nsplit, qvec, ovec, s); }
    else { if (a.e <= 64) go_sizes<128, 64>(a, nsplit, qvec, ovec, s); else go_sizes<128, 128>(a, nsplit, qvec, ovec, s); }
}

void launch_lay_attn_tile(const LAttnArgs& a, hipStream_t s) {
    if (a.ntiles > 0) launch(a, 0, s);
}

int lay_attn_few_split(long long visible, int blocks, int parts, bool packed) {
    // one key tile per wave, then more blocks and a merge: a further tile in the same wave costs about 4 us (its keys and values are two trips to
    // memory), the merge 6.  Eight tokens of four layers of width 4096, 32 heads on 8: context 3500 5.02 - 5.20 ms with one, 5.17 - 5.23 with two
    // tiles per wave; context 100 (no split) 4.96
    const int DW = packed ? 4 : 8;
    const long long tiles = (visible + KT - 1) / KT + 1;
    if (tiles <= DW) return 1;
    return (int)std::max(1ll, std::min({(tiles + DW - 1) / DW, (packed ? 512ll : 256ll) / std::max(1, blocks), (long long)parts / std::max(1, blocks)}));
}

void launch_lay_attn_few(const LAttnArgs& a, hipStream_t s, bool merge) {
    if (a.ntiles <= 0) return;
    const int nsplit = a.part_o && a.part_ml && a.nsplit > 1 ? a.nsplit : 1;
    launch(a, nsplit, s);
    if (nsplit > 1 && merge) launch_lay_attn_merge(a, nsplit, s);
}

}  // namespace cm
