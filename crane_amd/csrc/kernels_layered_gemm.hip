// Products of the layer-list decoders' mixtures of experts (bfloat16 format, more rows than the streaming row kernel takes):
// C[p] = act(A[row(p)] W_g^T) * (A[row(p)] W2_g^T) or A[row(p)] W_g^T, rows sorted by expert, one matrix (pair) per expert.
//
// A block makes BM x BN outputs with four waves (2 x 2) on v_mfma_f32_16x16x32_bf16.  Both operands are bfloat16 rows with K contiguous
// and go from memory into LDS without passing registers (global_load_lds_dwordx4: 8 rows x 128 bytes per wave instruction, k-tiles of 64
// elements = whole cache lines); the rows of A are gathered by their token there, for nothing.  The LDS image of such a load is linear in
// the lane, so the bank swizzle sits on the source: slot p of a row holds its 16-byte chunk p ^ ((row >> 1) & 7), and fragment reads undo
// it.  ST stages, one barrier per k-tile; two blocks share a CU, so one multiplies while the other waits.
//
// Which (row tile, expert) a block has follows from the group offsets in device memory: the tiles of all experts are numbered through and
// every block finds its own with one scan over the offsets (at most 64 experts: a wave's lanes), so the grid is rows / BM + experts tiles
// high whatever the router chose -- not experts x rows / BM, of which a 16-expert launch filled a quarter.  Numbered by expert, then column tile, then
// row tile, each XCD a contiguous share of the real count: an XCD's 64 blocks share their expert's gathered rows as well as weight columns (row tiles
// of all experts under one column tile: every XCD read all rows once per two column tiles, 1.6 GB a launch at the first size below, 4 TB/s;
// 402 / 264 us there, 132 for 99 with 300 tokens).  The expert of every token rides in the same launches: its tiles
// fill what the routed ones leave of the last round of blocks, and two launches less (a mixed step of 326 rows, 24 layers of width 1024: 54 us a layer
// of the four products in four launches, 37 in two).  A wave whose rows lie behind a ragged tile's end loads its share and multiplies nothing.
//
// Bound: LDS.  A wave's k-step of 64 x 64 outputs reads 8 KB of fragments for 16 products (256 cycles); four waves of two blocks ask for the
// LDS ports' full 128 bytes a cycle.  64 x 64 tiles: the latency of the weights' first touch and the L2's traffic per product.
// Measured (us per launch, gate-and-up / down; the 64 x 64 kernel without a pipeline that this replaces in brackets): 8192 rows, 16 experts of
// 2048 x 4096: 375 / 243 (2481 / 1566), 0.73 PFLOP/s; 1200 rows, 14 experts of 768 x 1024: 14.8 / 11.1 (60 / 50); before 16-byte stores.  Tiles of 128 x 256 and 256 x 256
// with eight waves: 388 and 396 at the first size (coarser shares of the last round), 70 for 75 on one matrix of 4096 x 4096; not kept.
#include <algorithm>

#include "dev_common.h"
#include "kernels.h"
#include "layered.h"
#include "layered_dev.h"

namespace cm {

namespace {

constexpr int BK = 64;
// experts: k-tiles between the starts of neighbouring column tiles (2 KB).  Few rows per expert read matrices out of memory, and blocks in step along K ask
// for the same columns of all their rows, a part of the memory channels: 40 tokens, 16 experts of 2048 x 4096: gate-and-up 126 -> 102 us (5.3 TB/s), down 70 ->
// 51; 700 tokens (175 rows each) 165 / 107 -> 165 / 98.  Not where a matrix is read by many row tiles, whose rows then come from several places: 2048 tokens, four
// layers, 4.85 -> 4.95 ms; one matrix alone 77 -> 91 us
constexpr int K_TURN = 16;

// a block's tile: sorted rows [p0, p0 + rows) of group g, column tile nt, of the launch's first product or (side) its second; false: a block behind
// the last tile.  Every XCD takes a contiguous share of either product's tiles, numbered by group, then column tile, then row tile
struct Tile { int g, p0, rows, nt; bool side; };
template <int BM>
__device__ __forceinline__ bool find_tile(const LTileArgs& a, const LTileArgs& b, int ntiles, int ntiles_b, int lane, Tile& t) {
    int o0 = 0, o1 = a.M;
    if (a.grp_off) {
        o1 = 0;
        if (lane < a.groups) { o0 = a.grp_off[lane]; o1 = a.grp_off[lane + 1]; }
    }
    const int mine = (o1 - o0 + BM - 1) / BM;
    int incl = mine;
    if (a.grp_off) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) { const int v = __shfl_up(incl, d); if (lane >= d) incl += v; }
    }
    const int total = __builtin_amdgcn_readlane(incl, 63) * ntiles, share = (total + 7) >> 3;
    const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
    t.side = slot >= share;
    if (t.side) {
        const int mb = (b.M + BM - 1) / BM, total_b = mb * ntiles_b, share_b = (total_b + 7) >> 3, at = xcd * share_b + slot - share;
        if (slot - share >= share_b || at >= total_b) return false;
        t.g = 0;
        t.nt = at / mb;
        t.p0 = (at - t.nt * mb) * BM;
        t.rows = min(BM, b.M - t.p0);
        return true;
    }
    const int at = xcd * share + slot;
    if (at >= total) return false;
    t.g = a.grp_off ? __builtin_ctzll(__ballot(at < incl * ntiles)) : 0;
    const int m = __builtin_amdgcn_readlane(mine, t.g), local = at - (__builtin_amdgcn_readlane(incl, t.g) - m) * ntiles;
    t.nt = local / m;
    t.p0 = __builtin_amdgcn_readlane(o0, t.g) + (local - t.nt * m) * BM;
    t.rows = min(BM, __builtin_amdgcn_readlane(o1, t.g) - t.p0);
    return true;
}

// field by field: a choice between the two by reference puts them into scratch memory (6 us a launch)
__device__ __forceinline__ void take(LTileArgs& a, const LTileArgs& b) {
    a.A = b.A; a.lda = b.lda; a.a_idx = nullptr; a.W = b.W; a.W2 = b.W2; a.w_stride = 0; a.C = b.C; a.ldc = b.ldc; a.c_idx = nullptr;
    a.M = b.M; a.N = b.N; a.K = b.K; a.grp_off = nullptr; a.bias = b.bias; a.act = b.act; a.act2 = b.act2; a.act_split = b.act_split; a.act_param = b.act_param;
}

// a wave's NI x NJ products to memory, rows mw .. and columns nw .. of the tile.  The weight is a product's first operand: a lane has columns 4 (lane / 16) + r of row
// lane % 16, one store of 8 or 16 bytes per product and one look at c_idx per band (a column of four rows each: 54 us for 46 and 49 for 37, gate-and-up and
// down of 1200 tokens, 14 experts of 768 x 1024; 417 and 174 for 409 and 163, 2048 tokens, 16 of 2048 x 4096 and the projections beside them).  DUAL: the upper half of the NJ
// columns belongs to W2.  The outputs' function is chosen once per block
template <int NI, int NJ, bool DUAL>
__device__ __forceinline__ void store_tile(const LTileArgs& a, f32x4 (&acc)[NI][NJ], int rows, int p0, int mw, int nw, int lane) {
    constexpr int NC = DUAL ? NJ / 2 : NJ;
    const int fr = lane & 15, lg = lane >> 4;
    const bool vec = a.ldc % 4 == 0 && ((uintptr_t)a.C & (DUAL ? 7 : 15)) == 0;
    size_t row[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int p = p0 + min(mw + i * 16 + fr, rows - 1);
        row[i] = a.c_idx ? (size_t)a.c_idx[p] : (size_t)p;
    }
    auto apply = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NC; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = f(acc[i][j][r], acc[i][j + (DUAL ? NC : 0)][r], min(nw + j * 16 + lg * 4 + r, a.N - 1));
    };
    if (DUAL) {
        if (a.act == LACT_SILU) apply([](float v, float u, int) { return lay_act(v, LACT_SILU) * u; });
        else if (a.act == LACT_CAPGLU) apply([&](float v, float u, int) { return lay_capglu(v, u, a.act_param); });
        else apply([&](float v, float u, int) { return lay_act(v, a.act) * u; });
    } else if (a.bias || a.act != LACT_NONE || a.act2 != LACT_NONE)
        apply([&](float v, float, int n) { return lay_act(a.bias ? v + a.bias[n] : v, n < a.act_split ? a.act : a.act2, a.act_param); });
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        if (mw + i * 16 + fr >= rows) continue;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int n = nw + j * 16 + lg * 4;
            const f32x4 v = acc[i][j];
            const size_t at = row[i] * a.ldc + n;
            if (vec && n + 4 <= a.N) {
                if (DUAL) *(u32x2*)((uint16_t*)a.C + at) = (u32x2){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                else *(f32x4*)((float*)a.C + at) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (n + r >= a.N) continue;
                    if (DUAL) ((uint16_t*)a.C)[at + r] = f32_to_bf16(v[r]); else ((float*)a.C)[at + r] = v[r];
                }
            }
        }
    }
}

template <int BM, int BN, int ST, bool DUAL>
__global__ __launch_bounds__(256, 2) void lay_tile_gemm_kernel(LTileArgs first, LTileArgs second, int ntiles, int ntiles_b) {
    constexpr int WM = BM / 2, WN = BN / 2, NI = WM / 16, NJ = WN / 16, APC = BM / 8, NL = (BM + BN) / 32;      // NL: loads per wave and k-tile
    constexpr int NC = DUAL ? WN / 2 : WN;                                // output columns of a wave
    constexpr int STAGE = (BM + BN) * BK;
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    Tile at;
    if (!find_tile<BM>(first, second, ntiles, ntiles_b, lane, at)) return;
    LTileArgs a = first;
    if (at.side) take(a, second);
    const int p0 = at.p0, rows = at.rows, nt = at.nt;
    const uint16_t* W = a.W + (size_t)at.g * a.w_stride;
    const uint16_t* W2 = DUAL ? a.W2 + (size_t)at.g * a.w_stride : nullptr;
    const int n0 = nt * (DUAL ? BN / 2 : BN);

    // this lane's share of the loads: piece wave + 4 i covers 8 rows of A (pieces below APC) or of the weight tile.  Rows past the end repeat
    // the last one; their outputs are not stored.  DUAL: a wave's columns of the weight tile are NC rows of W, then the same NC of W2
    const int prow = lane >> 3, pslot = lane & 7;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;                       // LDS offset of the dynamic segment (low half of the flat address)
    const uint16_t* src[NL];
    uint32_t dst[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int p = wave + 4 * i;
        const bool isA = p < APC;
        const int row = (isA ? p : p - APC) * 8 + prow;
        const int kc = (pslot ^ ((row >> 1) & 7)) << 3;
        if (isA) {
            const int r = p0 + min(row, rows - 1);
            src[i] = a.A + (size_t)(a.a_idx ? a.a_idx[r] / a.a_div : r) * a.lda + kc;
        } else {
            const int c = row / WN, q = row - c * WN;
            const bool second = DUAL && q >= NC;
            const int n = min(n0 + c * NC + (second ? q - NC : q), a.N - 1);
            src[i] = (second ? W2 : W) + (size_t)n * a.K + kc;
        }
        dst[i] = lds0 + (uint32_t)((isA ? p * 8 : BM + (p - APC) * 8) * BK) * 2u;
    }
    const int nk = a.K / BK;
    const int turn = a.grp_off && a.total < 256 * a.groups ? (nt & 3) * K_TURN % nk : 0;
    auto request = [&](int t) __attribute__((always_inline)) {            // past the end: the last tile again, into a stage nobody reads
        int tc = min(t, nk - 1) + turn;
        tc = tc < nk ? tc : tc - nk;
        const uint32_t at = (uint32_t)((t % ST) * STAGE) * 2u;
#pragma unroll
        for (int i = 0; i < NL; ++i) lds_load16(src[i] + (size_t)tc * BK, dst[i] + at);
    };
    f32x4 acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int fr = lane & 15, lg = lane >> 4, sw = (fr >> 1) & 7;
    const bool idle = wm * WM >= rows;                                    // a ragged tile's lower half: this wave loads, the matrix cores are the others'
#pragma unroll
    for (int t = 0; t < ST - 1; ++t) request(t);
    for (int t = 0; t < nk; ++t) {
        // this wave's share of tile t has landed and its reads of tile t - 1 are done; behind the barrier that holds for every wave
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * NL) : "memory");
        request(t + ST - 1);
        if (idle) continue;
        const uint16_t* As = lds + (t % ST) * STAGE + wm * WM * BK;
        const uint16_t* Bs = lds + (t % ST) * STAGE + (BM + wn * WN) * BK;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int fk = ((s * 4 + lg) ^ sw) << 3;
            bf16x8 af[NI], bf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) bf[j] = *(const bf16x8*)&Bs[(j * 16 + fr) * BK + fk];
#pragma unroll
            for (int i = 0; i < NI; ++i) af[i] = *(const bf16x8*)&As[(i * 16 + fr) * BK + fk];
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                      // the repeated loads of the tail: none may land after the block is gone
    store_tile<NI, NJ, DUAL>(a, acc, rows, p0, wm * WM, n0 + wn * NC, lane);
}

// row tiles of a launch; grouped: every expert ends in at most one ragged tile, and none has more than M rows
template <int BM>
int mtiles(const LTileArgs& a) {
    return a.grp_off ? std::min((a.total + BM - 1) / BM + a.groups, a.groups * ((a.M + BM - 1) / BM)) : (a.M + BM - 1) / BM;
}

template <int BM, int BN, int ST, bool DUAL>
void go(const LTileArgs& a, const LTileArgs& b, hipStream_t s) {
    constexpr size_t lds = (size_t)ST * (BM + BN) * BK * sizeof(uint16_t);
    static DevOnce attr;
    attr.run([&] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&lay_tile_gemm_kernel<BM, BN, ST, DUAL>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    const int cols = DUAL ? BN / 2 : BN, nt = (a.N + cols - 1) / cols, ntb = (b.N + cols - 1) / cols;
    const int share = (mtiles<BM>(a) * nt + 7) / 8 + ((b.M + BM - 1) / BM * ntb + 7) / 8;
    hipLaunchKernelGGL((lay_tile_gemm_kernel<BM, BN, ST, DUAL>), dim3((unsigned)share * 8), dim3(256), lds, s, a, b, nt, ntb);
}

}  // namespace

bool lay_tile_gemm_fits(int N, int K, int groups) { return N > 0 && K >= 2 * BK && K % BK == 0 && groups <= 64; }

void launch_lay_tile_gemm(const LTileArgs& a, hipStream_t s, const LTileArgs* beside) {
    if (a.M <= 0 || a.N <= 0) return;
    const LTileArgs b = beside ? *beside : LTileArgs();
    // 128 x 128 tiles where they still give the chip 320 blocks and a group fills half a tile of rows; measured (us, gate-and-up, 128 / 64
    // tiles): 16 experts of 2048 x 4096 -- 2048 tokens 375 / 541, 300 tokens (75 rows, 832 blocks) 99 / 138, 128 tokens (32 rows) 151 / 142;
    // 14 of 768 x 1024 -- 2048 tokens 49 / 55, 700 tokens (432 blocks) 25 / 24; one matrix pair 2048 x 4096 -- 1200 rows (320 blocks) 66 / 79,
    // 600 rows (160) 64 / 46
    const int total = a.grp_off ? a.total : a.M, groups = a.grp_off ? a.groups : 1;
    const int blocks = mtiles<128>(a) * ((a.N + (a.W2 ? 63 : 127)) / (a.W2 ? 64 : 128));
    // (the second product of 16 experts of 2048 x 4096: 100 tokens, 25 rows each, 54 / 66 -- twice the columns per block count there)
    const bool wide = blocks >= LAY_TILE_WIDE_BLOCKS && (total >= 64 * groups || (a.grp_off && !a.W2));
    if (a.W2) { if (wide) go<128, 128, 2, true>(a, b, s); else go<64, 64, 3, true>(a, b, s); }
    else { if (wide) go<128, 128, 2, false>(a, b, s); else go<64, 64, 3, false>(a, b, s); }
}

// rows of f32, gathered and scaled -> bfloat16: out[p] = x[idx[p] / div] * scale[idx[p]]
__global__ __launch_bounds__(256) void lay_round_scaled_kernel(const float* __restrict__ x, int ldx, const int32_t* __restrict__ idx, int div,
                                                               const float* __restrict__ scale, uint16_t* __restrict__ out, int K) {
    const int p = blockIdx.x, at = idx[p];
    const float* xr = x + (size_t)(at / div) * ldx;
    const float sc = scale[at];
    for (int k = threadIdx.x * 2; k < K; k += 512) {                      // K is even (a multiple of the k-tile)
        *(uint32_t*)(out + (size_t)p * K + k) = pack_bf16x2(xr[k] * sc, xr[k + 1] * sc);
    }
}
void launch_lay_round_scaled(const float* x, int ldx, const int32_t* idx, int div, const float* scale, uint16_t* out, int P, int K, hipStream_t s) {
    if (P <= 0) return;
    hipLaunchKernelGGL(lay_round_scaled_kernel, dim3((unsigned)P), dim3(256), 0, s, x, ldx, idx, div, scale, out, K);
}

}  // namespace cm
