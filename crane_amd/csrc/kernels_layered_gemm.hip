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
// 2048 x 4096: 375 / 243 (2481 / 1566), 0.73 PFLOP/s; 1200 rows, 14 experts of 768 x 1024: 14.8 / 11.1 (60 / 50); before 16-byte stores.  Larger tiles read fewer
// fragments per product: 192 x 128 and 128 x 192 on the same kernel (two blocks still share a CU: 160 KB of LDS), 256 x 256 with eight waves in two phases
// (lay_tall_gemm_kernel; with this kernel's one barrier per k-tile it was no faster); lay_tile_shape says which a product takes, with the figures.
#include <algorithm>
#include <cmath>
#include <type_traits>

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
struct Tile { int g, p0, rows, nt, shift; bool side; };      // shift: from a sorted row to its place among the indices
template <int BM>
__device__ __forceinline__ bool find_tile(const LTileArgs& a, const LTileArgs& b, int ntiles, int ntiles_b, int lane, Tile& t) {
    int o0 = 0, n = a.M;
    auto running = [&](int v) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) { const int u = __shfl_up(v, d); if (lane >= d) v += u; }
        return v;
    };
    if (a.grp_off) {
        n = 0;
        if (a.bucket > 0) {
            if (lane < a.groups) n = a.grp_off[lane * LAY_COUNT_STRIDE];
            o0 = running(n) - n;
        } else if (lane < a.groups) { o0 = a.grp_off[lane]; n = a.grp_off[lane + 1] - o0; }
    }
    const int mine = (n + BM - 1) / BM, incl = a.grp_off ? running(mine) : mine;
    const int total = __builtin_amdgcn_readlane(incl, 63) * ntiles, share = (total + 7) >> 3;
    const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
    t.side = slot >= share;
    if (t.side) {
        const int mb = (b.M + BM - 1) / BM, total_b = mb * ntiles_b, share_b = (total_b + 7) >> 3, at = xcd * share_b + slot - share;
        if (slot - share >= share_b || at >= total_b) return false;
        t.g = 0; t.shift = 0;
        t.nt = at / mb;
        t.p0 = (at - t.nt * mb) * BM;
        t.rows = min(BM, b.M - t.p0);
        return true;
    }
    const int at = xcd * share + slot;
    if (at >= total) return false;
    t.g = a.grp_off ? __builtin_ctzll(__ballot(at < incl * ntiles)) : 0;
    const int m = __builtin_amdgcn_readlane(mine, t.g), local = at - (__builtin_amdgcn_readlane(incl, t.g) - m) * ntiles;
    const int first = __builtin_amdgcn_readlane(o0, t.g), row = (local - (t.nt = local / m) * m) * BM;
    t.p0 = first + row;
    t.rows = min(BM, __builtin_amdgcn_readlane(n, t.g) - row);
    t.shift = a.bucket > 0 ? t.g * a.bucket - first : 0;
    return true;
}

// field by field: a choice between the two by reference puts them into scratch memory (6 us a launch)
__device__ __forceinline__ void take(LTileArgs& a, const LTileArgs& b) {
    a.A = b.A; a.lda = b.lda; a.a_idx = nullptr; a.W = b.W; a.W2 = b.W2; a.w_stride = 0; a.C = b.C; a.ldc = b.ldc; a.c_idx = nullptr;
    a.M = b.M; a.N = b.N; a.K = b.K; a.grp_off = nullptr; a.bucket = 0; a.bias = b.bias; a.act = b.act; a.act2 = b.act2; a.act_split = b.act_split; a.act_param = b.act_param;
}

// a wave's NI x NJ products to memory, rows mw .. and columns nw .. of the tile.  The weight is a product's first operand: a lane has columns 4 (lane / 16) + r of row
// lane % 16, one store of 8 or 16 bytes per product and one look at c_idx per band (a column of four rows each: 54 us for 46 and 49 for 37, gate-and-up and
// down of 1200 tokens, 14 experts of 768 x 1024; 417 and 174 for 409 and 163, 2048 tokens, 16 of 2048 x 4096 and the projections beside them).  DUAL: the upper half of the NJ
// columns belongs to W2.  The outputs' function is chosen once per block
template <int NI, int NJ, bool DUAL, bool FN = true>
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
    } else if (FN && (a.bias || (nw < a.act_split && a.act != LACT_NONE) || (nw + NC * 16 > a.act_split && a.act2 != LACT_NONE))) {
        // (columns that have a function; a sigmoid behind the rest by itself, lay_act for every element is 10 KB of code and more: the projection of 326 rows of 1024
        // 13.3 us, 8.2 here)
        if (!a.bias && a.act == LACT_NONE && a.act2 == LACT_SIGMOID) apply([&](float v, float, int n) { const float g = lay_act(v, LACT_SIGMOID); return n < a.act_split ? v : g; });
        else apply([&](float v, float, int n) { return lay_act(a.bias ? v + a.bias[n] : v, n < a.act_split ? a.act : a.act2, a.act_param); });
    }
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

template <int BM, int BN, int ST, bool DUAL, bool FN>
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
    if (a.a_idx) a.a_idx += at.shift;
    if (a.c_idx) a.c_idx += at.shift;
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
    store_tile<NI, NJ, DUAL, FN>(a, acc, rows, p0, wm * WM, n0 + wn * NC, lane);
}

// 256 x 256 tiles, eight waves as 2 x 4, a wave 128 x 64 outputs: 24 KB of fragments for 64 products a k-tile, three quarters of what the 64 x 64 of the
// kernel above ask the LDS for per product.  The two wave rows run half a tile apart: in one slot a row fetches its fragments of a tile, in the next it multiplies, the other row the other way
// round.  The first slot of tile t asks for the rows of tile t + 1, the second for the weights of tile t + 2 (three stages of those: 160 KB), a request between two bands of products: 32 requests
// of 16 cycles each per slot of 1024 (both for t + 1 in the first slot, which they filled: 8192 rows, 16 experts of 2048 x 4096 and one of every token, gate-and-up / down 350 / 212 us, here 337 / 202).  A band of 16 rows
// behind a ragged tile's end multiplies nothing.  8192 rows, 4096 columns, K 4096: 359 us on 128 x 128 tiles, 228 - 305 here by what the clock allows (183 with
// operands of zeros: 1.5 PFLOP/s)
//
// 128 x 256 and 128 x 384 are two tiles of 128 x 128 or 128 x 192 side by side, of one matrix: the same schedule over half the rows, which the two tiles read once.  A block of 128 x 128 asks for
// 32 KB per k-tile of 512 MFMA cycles, which is all that the address path takes in that time; two together 48 KB per 1024.  384 columns leave LDS for two stages of weights and three of rows:
// there the weights are the near operand.  Bound by the LDS: 16 fragments per 32 products of a wave and the 48 KB that come in are 1400 cycles of its port per 1024 of the matrix cores.  2048 rows, K 4096,
// single tiles / in pairs: 4096 columns 79 / 69 us, 6144 109 / 100; a prompt of four layers 3.70 -> 3.64 ms, 1200 tokens 2.88 -> 2.84, 650 2.25 -> 2.22; width 1024 equal.
template <bool DUAL, int BM, int BN>
__global__ __launch_bounds__(512) void lay_tall_gemm_kernel(LTileArgs first, LTileArgs second, int ntiles, int ntiles_b) {
    constexpr int WM = BM / 2, WN = BN / 4, NI = WM / 16, NJ = WN / 16, NA = BM / 64, NW = BN / 64, NC = DUAL ? WN / 2 : WN;
    constexpr bool WFAR = BN == 256;                                      // the operand with three stages, asked for two tiles ahead: weights, or rows
    constexpr int AST = WFAR ? 2 : 3, WST = WFAR ? 3 : 2, ASTAGE = BM * BK, WSTAGE = BN * BK, WBASE = AST * ASTAGE, NEAR = WFAR ? NA : NW, FAR = WFAR ? NW : NA;
    static_assert(!DUAL || BN == 256, "a wave's pieces are all of W or all of W2");
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    Tile at;
    if (!find_tile<BM>(first, second, ntiles, ntiles_b, lane, at)) return;
    LTileArgs a = first;
    if (at.side) take(a, second);
    if (a.a_idx) a.a_idx += at.shift;
    if (a.c_idx) a.c_idx += at.shift;
    const int p0 = at.p0, rows = at.rows;
    const int n0 = at.nt * (DUAL ? BN / 2 : BN);

    // loads as above: piece wave + 8 i covers 8 rows of A, and as many of the weight tile, a wave's all in W or all in W2.  32-bit offsets from bases in scalar registers: 16
    // vector registers for pointers are 8 too many (launch_lay_tile_gemm: the rows of A are within reach)
    const int r0 = wave * 8 + (lane >> 3), slot = lane & 7;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    const char* const A0 = (const char*)a.A;
    const char* const W0 = (const char*)((DUAL && (wave & 4) ? a.W2 : a.W) + (size_t)at.g * a.w_stride + (size_t)n0 * a.K);
    uint32_t aoff[NA], woff[NW];
    const uint32_t kc = (uint32_t)(slot ^ ((r0 >> 1) & 7)) << 4;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int r = p0 + min(i * 64 + r0, rows - 1);
        aoff[i] = (uint32_t)(a.a_idx ? a.a_idx[r] / a.a_div : r) * (uint32_t)(a.lda * 2) + kc;
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) woff[i] = (uint32_t)min(DUAL ? i * NC + (r0 & 31) : i * 64 + r0, a.N - 1 - n0) * (uint32_t)(a.K * 2) + kc;
    const int nk = a.K / BK;
    // (past the end: the last tile again, into a stage nobody reads)
    auto ask_a = [&](int i, int t) __attribute__((always_inline)) { lds_load16_at(A0 + (size_t)min(t, nk - 1) * (BK * 2), aoff[i], lds0 + (uint32_t)(t % AST * ASTAGE + (wave + 8 * i) * 8 * BK) * 2u); };
    auto ask_w = [&](int i, int t) __attribute__((always_inline)) { lds_load16_at(W0 + (size_t)min(t, nk - 1) * (BK * 2), woff[i], lds0 + (uint32_t)(WBASE + t % WST * WSTAGE + (wave + 8 * i) * 8 * BK) * 2u); };
    auto ask_near = [&](int i, int t) __attribute__((always_inline)) { if (i < NEAR) { if (WFAR) ask_a(i, t); else ask_w(i, t); } };
    auto ask_far = [&](int i, int t) __attribute__((always_inline)) { if (i < FAR) { if (WFAR) ask_w(i, t); else ask_a(i, t); } };
    f32x4 acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int fr = lane & 15, lg = lane >> 4, sw = (fr >> 1) & 7;
    const int bands = min(NI, (rows - wm * WM + 15) >> 4);                // bands of this wave that have rows (none: 0 or less)
    bf16x8 af[2][NI], bf[2][NJ];
    auto fetch = [&](int t) __attribute__((always_inline)) {
        const uint16_t* As = lds + t % AST * ASTAGE + wm * WM * BK;
        const uint16_t* Bs = lds + WBASE + t % WST * WSTAGE + wn * WN * BK;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int fk = ((s * 4 + lg) ^ sw) << 3;
#pragma unroll
            for (int j = 0; j < NJ; ++j) bf[s][j] = *(const bf16x8*)&Bs[(j * 16 + fr) * BK + fk];
#pragma unroll
            for (int i = 0; i < NI; ++i) af[s][i] = *(const bf16x8*)&As[(i * 16 + fr) * BK + fk];
        }
    };
    auto band = [&](int s, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[s][j], af[s][i], acc[i][j], 0, 0, 0);
    };
    // a slot's products with its requests between the bands
    constexpr int PER = (std::max(NEAR, FAR) + NI - 1) / NI;
    auto multiply = [&](auto ask) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (i < bands) { band(0, i); band(1, i); }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < PER; ++k) ask(i * PER + k);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // every wave runs 2 nk + 2 barriers.  What is asked for in the second slot of a tile, the newest FAR requests, may stay in flight at its end
#pragma unroll
    for (int i = 0; i < std::max(NEAR, FAR); ++i) { ask_near(i, 0); ask_far(i, 0); }
#pragma unroll
    for (int i = 0; i < FAR; ++i) ask_far(i, 1);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(FAR) : "memory");
    if (wm == 0) {
        for (int t = 0; t < nk; ++t) {
#pragma unroll
            for (int i = 0; i < NEAR; ++i) ask_near(i, t + 1);
            fetch(t);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            multiply([&](int i) __attribute__((always_inline)) { ask_far(i, t + 2); });
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(FAR) : "memory");
        }
        asm volatile("s_barrier" ::: "memory");
    } else {
#pragma unroll
        for (int i = 0; i < NEAR; ++i) ask_near(i, 1);                    // in the slot in which row 0 fetches tile 0
        asm volatile("s_barrier" ::: "memory");
        for (int t = 0; t < nk; ++t) {
#pragma unroll
            for (int i = 0; i < FAR; ++i) ask_far(i, t + 2);
            fetch(t);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(FAR) : "memory");
            multiply([&](int i) __attribute__((always_inline)) { ask_near(i, t + 2); });
            asm volatile("s_barrier" ::: "memory");
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                      // the repeated loads of the tail
    store_tile<NI, NJ, DUAL, DUAL>(a, acc, rows, p0, wm * WM, n0 + wn * NC, lane);
}

// row tiles of a launch; grouped: every expert ends in at most one ragged tile, and none has more than M rows
template <int BM>
int mtiles(const LTileArgs& a) {
    return a.grp_off ? std::min((a.total + BM - 1) / BM + a.groups, a.groups * ((a.M + BM - 1) / BM)) : (a.M + BM - 1) / BM;
}

template <int BM, int BN, int ST, bool DUAL, bool FN = true>
void go(const LTileArgs& a, const LTileArgs& b, hipStream_t s) {
    constexpr size_t lds = (size_t)ST * (BM + BN) * BK * sizeof(uint16_t);
    static DevOnce attr;
    attr.run([&] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&lay_tile_gemm_kernel<BM, BN, ST, DUAL, FN>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    const int cols = DUAL ? BN / 2 : BN, nt = (a.N + cols - 1) / cols, ntb = (b.N + cols - 1) / cols;
    const int share = (mtiles<BM>(a) * nt + 7) / 8 + ((b.M + BM - 1) / BM * ntb + 7) / 8;
    hipLaunchKernelGGL((lay_tile_gemm_kernel<BM, BN, ST, DUAL, FN>), dim3((unsigned)share * 8), dim3(256), lds, s, a, b, nt, ntb);
}
template <bool DUAL, int BM = 256, int BN = 256>
void go_tall(const LTileArgs& a, const LTileArgs& b, hipStream_t s) {
    constexpr size_t lds = (size_t)(BN == 256 ? 2 * BM + 3 * BN : 3 * BM + 2 * BN) * BK * sizeof(uint16_t);
    static DevOnce attr;
    attr.run([&] { (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&lay_tall_gemm_kernel<DUAL, BM, BN>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
    const int cols = DUAL ? BN / 2 : BN, nt = (a.N + cols - 1) / cols, ntb = (b.N + cols - 1) / cols;
    const int share = (mtiles<BM>(a) * nt + 7) / 8 + ((b.M + BM - 1) / BM * ntb + 7) / 8;
    hipLaunchKernelGGL((lay_tall_gemm_kernel<DUAL, BM, BN>), dim3((unsigned)share * 8), dim3(512), lds, s, a, b, nt, ntb);
}

// The last columns of one matrix, [n0, N), at most 64 of them: 16 rows per block, the k-tiles dealt to its eight waves, operands from memory straight into fragments.
// What it saves: 32 gate columns behind 4096 others were a column tile of their own, 16 blocks behind the 512 that fill the chip (2048 rows, K 4096: 116 us in
// the place of 76; here 76 + 14; four tiles requested together 13, but 7 for 5 at K 1024)
template <int NJ>
__global__ __launch_bounds__(512) void lay_few_cols_kernel(LTileArgs a, int n0) {
    constexpr int NW = 8;
    __shared__ __attribute__((aligned(16))) float part[NW][NJ][64][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 15, lg = lane >> 4, m0 = (int)blockIdx.x * 16;
    const uint16_t* A = a.A + (size_t)min(m0 + fr, a.M - 1) * a.lda + lg * 8;
    const uint16_t* W[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) W[j] = a.W + (size_t)min(n0 + j * 16 + fr, a.N - 1) * a.K + lg * 8;
    f32x4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // (a row's stride is a multiple of the memory channels' turn where K is a power of two: blocks start at different tiles, or all ask the same channels at once: 16 us)
    const int cnt = (a.K / BK - wave + NW - 1) / NW;
    const int first = cnt > 0 ? (int)blockIdx.x % cnt : 0;
    for (int i = 0; i < cnt; ++i) {
        const int k = ((i + first < cnt ? i + first : i + first - cnt) * NW + wave) * BK;
        bf16x8 x[2], w[2][NJ];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            x[h] = *(const bf16x8*)(A + k + h * 32);
#pragma unroll
            for (int j = 0; j < NJ; ++j) w[h][j] = *(const bf16x8*)(W[j] + k + h * 32);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h][j], x[h], acc[j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) *(f32x4*)part[wave][j][lane] = acc[j];
    __syncthreads();
    for (int i = threadIdx.x; i < NJ * 256; i += 512) {                   // element i: fragment i / 256, row i / 16 % 16, column i % 16
        const int j = i >> 8, m = (i >> 4) & 15, c = i & 15, l = (c >> 2) * 16 + m, n = n0 + j * 16 + c;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += part[w][j][l][c & 3];
        if (m0 + m < a.M && n < a.N) ((float*)a.C)[(size_t)(m0 + m) * a.ldc + n] = lay_act(a.bias ? v + a.bias[n] : v, n < a.act_split ? a.act : a.act2, a.act_param);
    }
}
void go_few_cols(const LTileArgs& a, int n0, hipStream_t s) {
    const dim3 grid((unsigned)((a.M + 15) / 16));
    if (a.N - n0 <= 16) hipLaunchKernelGGL(lay_few_cols_kernel<1>, grid, dim3(512), 0, s, a, n0);
    else if (a.N - n0 <= 32) hipLaunchKernelGGL(lay_few_cols_kernel<2>, grid, dim3(512), 0, s, a, n0);
    else hipLaunchKernelGGL(lay_few_cols_kernel<4>, grid, dim3(512), 0, s, a, n0);
}

// row tiles that a launch will have: of n rows an expert has on average, spread by their root
float row_tiles(const LTileArgs& a, int bm) {
    if (!a.grp_off) return (float)((a.M + bm - 1) / bm);
    const float avg = (float)a.total / a.groups, sd = std::sqrt(avg) + 1e-3f;
    float t = 1.f;
    for (int k = 1; k * bm < a.M; ++k) t += std::min(1.f, std::max(0.f, 0.5f + (avg - (float)(k * bm)) / (3.f * sd)));
    return t * a.groups;
}
// every row of A within lay_tall_gemm_kernel's 32-bit offsets
bool lay_near(const LTileArgs& x) { return (uint64_t)std::max(x.total, x.M) * x.lda * 2 + (uint64_t)x.K * 2 < 1ull << 32; }
bool plain_out(const LTileArgs& a) { return !a.bias && (a.act == LACT_NONE || a.act_split <= 0) && (a.act2 == LACT_NONE || a.act_split >= a.N); }

}  // namespace

bool lay_tile_gemm_fits(int N, int K, int groups) { return N > 0 && K >= 2 * BK && K % BK == 0 && groups <= 64; }

// 128 x 128 tiles where they still give the chip 320 blocks and a group fills half a tile of rows.  us a launch, 128 / 64 tiles: 16 experts of 2048 x 4096, 4 per token, and one
// of every token beside them, gate-and-up and down: 40 tokens 153 / 110, 75 / 59, 100 155 / 115, 77 / 61, 128 157 / 120, 78 / 63, 200 159 / 143, 82 / 74, 300 (75 rows each)
// 164 / 166, 82 / 87, 2048 375 / 541 and more; one matrix pair 2048 x 4096: 1200 rows (320 blocks) 66 / 79, 600 rows (160) 64 / 46.  The second product of experts alone in their
// launch has half the blocks of the first for the same columns, and all of them long: 128 tiles from the first row on (a layer of the same experts and none of every
// token, 20 / 100 / 200 tokens: 276 / 284 us, 297 / 304, 331 / 343; with it beside them 306 / 290, 327 / 309, 373 / 365; 32 experts of 1024 x 2048 and one of 512
// beside, 100 tokens, 271 / 267)
bool lay_tile_wide(const LTileArgs& a, bool beside) {
    const int total = a.grp_off ? a.total : a.M, groups = a.grp_off ? a.groups : 1;
    const int blocks = mtiles<128>(a) * ((a.N + (a.W2 ? 63 : 127)) / (a.W2 ? 64 : 128));
    return blocks >= LAY_TILE_WIDE_BLOCKS && (total >= 64 * groups || (a.grp_off && !a.W2 && !beside));
}

// Larger tiles than those two have fewer blocks, and a launch takes as many rounds of blocks as do not fit the chip at once (512 of four waves, 256 of eight): the shape
// whose rounds take the least.  A round in quarters of one of 128 x 128 tiles, measured: 192 x 128 5, 128 x 192 5.4, 256 x 256 6.2; 64 x 64 tiles, three blocks on a CU and
// short ones, 2.6 and half a round for the ends.  us a launch, the two above / the shape taken, experts of 2048 x 4096 as above, weights out of memory:
// gate-and-up 2048 tokens 465 / 397 (256 x 256), 1200 310 / 289 (192 x 128), 700 231 / 198 (192 x 128), 450 185 / 130 (128 x 192), 300 177 / 119, 200 126 / 113, 100 115 / 115 (64);
// down 250 / 219, 167 / 156, 124 / 110, 92 / 83, 87 / 73, 69 / 62, 62 / 62.  14 experts of 768 x 1024, one of 512: 2048 tokens 47, 38 / 30 (192 x 128), 1300 43 / 33, 22, 500 24, 15.
// One matrix, K 4096: 2048 rows, 6144 columns 136 / 100 (128 x 192; 256 x 256 109, 192 x 128 140), 8192 columns 155 / 114 (256 x 256; 192 x 128 149, 128 x 192 154), 4096 columns 79 (128; the others 89 to
// 102); 1536 rows, 8192 columns 128 / 98 (192 x 128; 256 x 256 107)
static LayTileShape lay_tile_least(const LTileArgs& a, const LTileArgs& b, float& least) {
    struct { LayTileShape shape; int bm, bn, slots; float round; } const all[] = {
        {LTILE_128, 128, 128, 512, 4.f}, {LTILE_192_128, 192, 128, 512, 5.f}, {LTILE_128_192, 128, 192, 512, 5.4f}, {LTILE_256, 256, 256, 256, 6.2f}};
    auto blocks = [&](int bm, int bn) {
        const int cols = a.W2 ? bn / 2 : bn;
        return row_tiles(a, bm) * (float)((a.N + cols - 1) / cols) + (b.M > 0 ? row_tiles(b, bm) * (float)((b.N + cols - 1) / cols) : 0.f);
    };
    const bool wide = lay_tile_wide(a, b.M > 0);
    LayTileShape best = wide ? LTILE_128 : LTILE_64;
    least = wide ? 4.f * std::ceil(blocks(128, 128) / 512.f) : 2.6f * (blocks(64, 64) / 768.f + 0.5f);
    if (!a.W2 && !(plain_out(a) && (b.M <= 0 || plain_out(b)))) return best;      // (the large tiles' stores know no bias and no function)
    for (const auto& c : all) {
        if (c.shape == LTILE_256 && !(lay_near(a) && lay_near(b))) continue;
        const float t = c.round * std::ceil(blocks(c.bm, c.bn) / (float)c.slots);
        if (t < least) { least = t; best = c.shape; }
    }
    return best;
}

LayTileShape lay_tile_shape(const LTileArgs& a, const LTileArgs& b) { float t; return lay_tile_least(a, b, t); }

// One matrix whose last 1 .. 64 columns reach into a further column tile: a launch of their own (5 us at K 1024, 14 at 4096) where it saves more rounds' time than that, a quarter of a round of 128 x 128
// tiles being about 5 us per 1024 of K.  2048 rows, K 4096: 4128 columns 116 us in one launch, 76 + 14 in two; 6176 145, 109 + 14; K 1024, 1032 columns: 14 in one, 11 + 5
bool lay_tile_tail(const LTileArgs& a, bool beside) {
    const int rest = a.N % 128;
    if (a.grp_off || a.W2 || a.a_idx || a.c_idx || beside || rest == 0 || rest > 64 || a.N < 256) return false;
    LTileArgs m = a;
    m.N -= rest;
    float all, main;
    lay_tile_least(a, LTileArgs(), all);
    lay_tile_least(m, LTileArgs(), main);
    return (all - main) * (float)a.K > 4096.f * 0.8f;
}

void launch_lay_tile_gemm(const LTileArgs& a0, hipStream_t s, const LTileArgs* beside) {
    if (a0.M <= 0 || a0.N <= 0) return;
    LTileArgs a = a0;
    const LTileArgs b = beside ? *beside : LTileArgs();
    const int rest = a.N % 128;
    if (lay_tile_tail(a, b.M > 0)) {                                      // the last columns in a launch of their own
        go_few_cols(a, a.N - rest, s);
        a.N -= rest;
    }
    // (one matrix: the tiles of a shape in pairs, rows by rows, where their number is even)
    auto pairs = [&](int bn) { return !a.grp_off && !a.W2 && b.M <= 0 && plain_out(a) && lay_near(a) && a.N % (2 * bn) == 0; };
    auto launch = [&](auto dual) {
        constexpr bool DUAL = decltype(dual)::value;
        const LayTileShape shape = lay_tile_shape(a, b);
        if constexpr (!DUAL) {
            if (shape == LTILE_128 && pairs(128)) return go_tall<false, 128, 256>(a, b, s);
            if (shape == LTILE_128_192 && pairs(192)) return go_tall<false, 128, 384>(a, b, s);
        }
        switch (shape) {
            case LTILE_64: go<64, 64, 3, DUAL>(a, b, s); break;
            case LTILE_128: go<128, 128, 2, DUAL>(a, b, s); break;
            case LTILE_192_128: go<192, 128, 2, DUAL, DUAL>(a, b, s); break;
            case LTILE_128_192: go<128, 192, 2, DUAL, DUAL>(a, b, s); break;
            case LTILE_256: go_tall<DUAL>(a, b, s); break;
        }
    };
    if (a.W2) launch(std::true_type()); else launch(std::false_type());
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
