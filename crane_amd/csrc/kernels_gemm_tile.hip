// Prompt products of more than 128 rows with bf16 hi + lo activations: C[M, N] (+)= A[M, K] . W[N, K]^T, two MFMAs per product, f32 accumulate; per accumulator the MFMAs
// of gemm_bf16_kernel in its order (k ascending, hi then lo inside 32 of them).
//
// What bounds it: with real operands the card's power -- a loop of these MFMAs on registers alone runs at 2.1 GHz, the tiles here at 1.7 .. 1.9 -- so that every byte through
// the LDS counts twice, once for its time and once for the clock.  The 128 x 256 tiles of gemm256_kernel that were here before read 24 fragments from the LDS per
// 64 MFMAs and asked for a whole k-tile in one of its two slots, 64 requests that take the address path 16 cycles each: 1024 of that slot's 1024 cycles, and the matrix cores were busy
// 65 .. 73 % of the cycles (with the requests taken out of that loop 96 %, with the fragment reads taken out instead no more than before).  Here
//   * a tile is 256 x 256 or 128 x 384 where that fills the chip: 20 or 19 fragments per 64 MFMAs, 48 or 55 KB into the LDS per 2048 MFMA cycles in the place of 64;
//   * the walk is in slots of 32 elements of K, and the requests for a later tile are spread over two or three of the four slots that a tile of activations lasts;
//   * a request's address is a scalar base, advanced with K, and one 32-bit offset per lane and row band: no 64-bit pointers in vector registers (256 x 256: 230 of 256 registers).
// Measured (us a launch, real operands back to back, before / here): 24576 x 4096 at 2048 rows 674 / 560, at 452 180 / 145, at 300 158 / 123; 6144 x 4096 at 2048 193 / 162;
// 4096 x 12288 at 2048 330 / 288 (one round of 128 x 256 either way); 12288 x 2048 at 2048 196 / 171; 4096 x 1024 with gelu at 3172 72 / 60.  (Gate and up in these with a SiLU of
// fewer roundings than silu_mul's, which takes 1 .. 2 % more: 24576 x 4096 at 2048 rows 545 / 556, at 452 147.7 / 149.)
//
// LDS: two stages of activations, 64 deep (an operand row is one whole 128-byte line per stage), and two of weights, 64 deep, or 32 where 256 rows of activations leave 32 KB
// for them (their lines are fetched twice, which the L1's fill path has room for: 64 KB of lines per 2048 cycles of MFMA at 64 bytes a cycle).  Slot p of a row holds its 16-byte
// chunk p ^ turn(row), so that the 16 lanes of a fragment read fall on 16 different slots of the 256-byte bank row.
#include <algorithm>

#include "dev_common.h"
#include "kernels.h"

namespace cm {

namespace {

// silu(g) u with the roundings of the other kernels' epilogues, so that a row has the same bits beside any number of rows (exp2(-1.4427 g) and a bare reciprocal round the exponent:
// 1.8e-6 of the value at g above -30 where this is 1.4e-7 off; the product is rounded before its planes are taken)
__device__ __forceinline__ float silu_mul(float g, float u) {
#pragma clang fp contract(off)
    return g / (1.0f + expf(-g)) * u;
}
template <int NW>
__device__ __forceinline__ void put_words(uint16_t* p, const uint32_t* w) {
    if constexpr (NW == 4) *(u32x4*)p = (u32x4){w[0], w[1], w[2], w[3]};
    else *(u32x2*)p = (u32x2){w[0], w[1]};
}

// Slots: the waves 0-3 and 4-7 (each SIMD hosts one of either) are half a step apart.  A step is 32 elements of K: in one slot a wave fetches all its fragments, in the next
// it multiplies, while the other half does the opposite; the workgroup barrier closes every slot.  A tile of 64 is four slots.  The stage of tile t is free
// once waves 4-7 have fetched its second step, in its fourth slot: from the first slot of tile t + 1 on, tile t + 2 is asked for into it, and it has landed, by every wave's own count, at
// the end of that tile's fourth.  32-deep weights: the stage of step u is asked for in the slot in which waves 0-3 fetch step u - 1 and has landed one slot later.
template <int EPI, int BM, int BN>
__global__ __launch_bounds__(512) void gemm_tile_kernel(GemmArgs a) {
    constexpr int GM = BN == 192 ? 4 : 2, GN = 8 / GM, WM = BM / GM, WN = BN / GN, NI = WM / 16, NJ = WN / 16;      // waves GM x GN, NI x NJ tiles of 16 x 16 each
    constexpr int WD = BM == 256 ? 32 : 64;                               // depth of a weight stage
    constexpr int SPREAD = BM == 256 ? 2 : 3;                             // slots over which a tile's requests are spread (three for the former: 560 -> 585 us; two for the latter: 312 -> 320)
    // A 16-bit output has a lane's columns C fragments wide next to each other, 16 bytes (8 at 96 columns a wave) per store: row 4 g + r of weight fragment j is
    // column 16 C (j / C) + 4 C g + 4 (j % C) + r of the wave's
    constexpr int C = EPI == GEPI_ACT_SPLIT ? 2 : EPI == GEPI_SILUMUL ? (NJ % 4 == 0 ? 4 : 2) : 1;
    constexpr bool SWAP = EPI != GEPI_PARTIAL;                            // the weight first: a lane has four columns of one row
    static_assert(NJ % C == 0 && WN % (16 * C) == 0, "column groups");
    constexpr int PLANE = BM * 64, ASTAGE = 2 * PLANE, WSTAGE = BN * WD, WBASE = 2 * ASTAGE;      // elements
    constexpr int NA = BM / 64;                                           // requests of a wave per activation plane and tile (8 rows x 128 bytes each)
    constexpr int WPC = BN * WD / 512, NW = (WPC + 7) / 8;                // requests per weight stage, of a wave (8 rows x 128 bytes, 16 x 64)
    constexpr int NP = 2 * NA + (WD == 64 ? NW : 0);                      // requests of a wave per tile, and those of 32-deep weights apart
    constexpr int NS = WD == 32 ? NW : 0, NMAX = (NP + SPREAD - 1) / SPREAD + NS;
    extern __shared__ __attribute__((aligned(16))) uint16_t ldst[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % GM, wn = wave / GM;
    const int tiles_m = (a.M + BM - 1) / BM, nb = tiles_m * (a.N / BN);
    const int ks = (int)blockIdx.x / nb, bid = xcd_neighbours((int)blockIdx.x - ks * nb, nb);
    // The tiles of an XCD are a patch of four row tiles and the columns beside them, which its L2 fetches once for all: a whole column of 16 row tiles and the next one was the
    // activations of every row, 8 times over the chip.  us, columns first / patches (of eight rows in brackets): 4096 x 12288 at 2048 rows 304 / 288 (291), at 1400 245 / 237 (245), at 1000
    // 165 / 160 (165); 4096 x 4096 at 2048 110 / 103 (104); 2048 x 6144 at 2048 89.4 / 86.0 (87.0); products of one or two row patches as before
    const int tiles_n = a.N / BN, patches = (tiles_m + 3) / 4, high = (tiles_m + patches - 1) / patches, patch = bid / (high * tiles_n), in = bid - patch * high * tiles_n;
    const int rows = min(high, tiles_m - patch * high), tn = in / rows, m0 = (patch * high + in - tn * rows) * BM, n0 = tn * BN;
    const int K = a.K, nt = K / 64 / a.ksplit;                            // tiles of 64 of this block, from ks * nt on

    f32x4 acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // ---- requests: activation piece i holds the rows 64 i + 8 wave .. + 7 of the tile (rows past M: the last one again, their products are dropped) ----
    const uint32_t lds0 = (uint32_t)(uintptr_t)ldst, ldsw = lds0 + (uint32_t)wave * 1024u;
    uint32_t aoff[NA], woff[NW];
    {
        const int r = wave * 8 + (lane >> 3);
#pragma unroll
        for (int i = 0; i < NA; ++i) aoff[i] = (uint32_t)min(64 * i + r, a.M - 1 - m0) * (uint32_t)(K * 2) + ((uint32_t)((lane & 7) ^ ((r >> 1) & 7)) << 4);
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int p = wave + 8 * i < WPC ? wave + 8 * i : wave;       // (no piece left: the first one again, so that every wave counts the same)
            const int row = WD == 64 ? p * 8 + (lane >> 3) : p * 16 + (lane >> 2), g = row / (4 * C) & 3;
            const int slot = WD == 64 ? (lane & 7) ^ (g * 2 + ((row >> 1) & 1)) : (lane & 3) ^ g;
            woff[i] = (uint32_t)row * (uint32_t)(K * 2) + ((uint32_t)slot << 4);
        }
    }
    const size_t kbeg = (size_t)ks * nt * 128;
    const char* const hi0 = (const char*)(a.A_hi + (size_t)m0 * K) + kbeg;
    const char* const lo0 = (const char*)(a.A_lo + (size_t)m0 * K) + kbeg;
    const char* const w0 = (const char*)(a.W + (size_t)n0 * K) + kbeg;
    // (past the end: the last tile or step again, into a stage that nobody reads any more)
    auto ask_a = [&](int i, int t) __attribute__((always_inline)) {
        const int p = i < NA ? i : i - NA;
        lds_load16_at((i < NA ? hi0 : lo0) + (size_t)min(t, nt - 1) * 128, aoff[p], ldsw + (uint32_t)((t & 1) * ASTAGE + (i < NA ? 0 : PLANE)) * 2u + (uint32_t)p * 8192u);
    };
    auto ask_w = [&](int i, int u) __attribute__((always_inline)) {       // u: tile (64 deep) or step (32 deep)
        const int p = wave + 8 * i < WPC ? wave + 8 * i : wave;
        lds_load16_at(w0 + (size_t)min(u, nt * 64 / WD - 1) * (WD * 2), woff[i], lds0 + (uint32_t)(WBASE + (u & 1) * WSTAGE) * 2u + (uint32_t)p * 1024u);
    };
    // the g-th request of slot q of tile t
    auto ask = [&](int g, int q, int t) __attribute__((always_inline)) {
        if (NS > 0 && (q & 1) == 0) {
            if (g < NS) { ask_w(g, 2 * t + q / 2 + 1); return; }
            g -= NS;
        }
        const int b = q * NP / SPREAD, i = b + g;
        if (q >= SPREAD || i >= (q + 1) * NP / SPREAD) return;
        if (WD == 64 && i < NW) ask_w(i, t + 1);
        else ask_a(WD == 64 ? i - NW : i, t + 1);
    };
    auto ask_all = [&](int q, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < NMAX; ++g) ask(g, q, t);
    };

    const int fr = lane & 15, fq = lane >> 4, sw = fr >> 1;
    const int arow = (wm * WM + fr) * 64, wrow = wn * WN + (fr >> 2) * 4 * C + (fr & 3);
    bf16x8 ah[NI], al[NI], bw[NJ];
    auto fetch = [&](int u) __attribute__((always_inline)) {
        const int t = u >> 1, c64 = (((u & 1) * 4 + fq) ^ sw) << 3, c32 = (fq ^ (fr >> 2)) << 3;
        const uint16_t* A = ldst + (t & 1) * ASTAGE + arow + c64;
        const uint16_t* B = ldst + WBASE + (WD == 64 ? (t & 1) * WSTAGE + c64 : (u & 1) * WSTAGE + c32);
#pragma unroll
        for (int j = 0; j < NJ; ++j) bw[j] = *(const bf16x8*)&B[(wrow + j / C * 16 * C + j % C * 4) * WD];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            ah[i] = *(const bf16x8*)&A[i * 16 * 64];
            al[i] = *(const bf16x8*)&A[PLANE + i * 16 * 64];
        }
    };
    auto product = [](const bf16x8& x, const bf16x8& w, const f32x4& c) __attribute__((always_inline)) {
        return SWAP ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w, c, 0, 0, 0);
    };
    // a step's products, the requests of slot q between them (pinned: left alone the scheduler moves every MFMA in front of them)
    auto multiply = [&](int q, int t) __attribute__((always_inline)) {
        constexpr int PER = (NMAX + NI - 1) / NI;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = product(ah[i], bw[j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < PER; ++p) ask(i * PER + p, q, t);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = product(al[i], bw[j], acc[i][j]);
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // what a wave may leave in flight at the end of slot 1: the activations asked for behind the weights of slot 0
    constexpr int LATE = 2 * NP / SPREAD;

#pragma unroll
    for (int i = 0; i < NW; ++i) ask_w(i, 0);
#pragma unroll
    for (int i = 0; i < 2 * NA; ++i) ask_a(i, 0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if (wave < 4) {
        for (int t = 0; t < nt; ++t) {
            ask_all(0, t);
            fetch(2 * t);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            multiply(1, t);
            if constexpr (WD == 32) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LATE) : "memory");
            else asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            ask_all(2, t);
            fetch(2 * t + 1);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            multiply(3, t);
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_barrier" ::: "memory");                           // (every wave passes the same number of barriers)
    } else {
        ask_all(0, 0);
        asm volatile("s_barrier" ::: "memory");                           // one slot behind
        for (int t = 0; t < nt; ++t) {
            ask_all(1, t);
            fetch(2 * t);
            if constexpr (WD == 32) asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(LATE) : "memory");
            else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            multiply(2, t);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            ask_all(3, t);
            fetch(2 * t + 1);
            asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            multiply(0, t + 1);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                      // the requests past the end: none of this wave's may land after it is gone

    const int mw = m0 + wm * WM, nw = n0 + wn * WN;
    if constexpr (EPI == GEPI_PARTIAL) {                                  // D row = 4 (lane >> 4) + r: m, column = lane & 15: n
        float* P = a.ws + (size_t)ks * a.M * a.N;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = mw + i * 16 + fq * 4 + r;
                    if (m < a.M) P[(size_t)m * a.N + nw + j * 16 + fr] = acc[i][j][r];
                }
        return;
    }
    f32x4 bv[NJ];                                                         // the lane's columns: nw + 16 C (j / C) + 4 C fq + 4 (j % C) ..
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        bv[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (a.bias != nullptr) bv[j] = *(const f32x4*)(a.bias + nw + j / C * 16 * C + fq * 4 * C + j % C * 4);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int m = mw + i * 16 + fr;
        if (m >= a.M) continue;
        if constexpr (C == 1) {
            float* c = a.C + (size_t)m * a.ldc + nw + fq * 4;
            f32x4 old[NJ];
            if (EPI == GEPI_RESADD) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) old[j] = *(const f32x4*)(c + j * 16);
            }
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                f32x4 v = acc[i][j];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (a.bias != nullptr) v[r] += bv[j][r];
                    if (EPI == GEPI_RESADD) v[r] = old[j][r] + v[r];
                }
                *(f32x4*)(c + j * 16) = v;
            }
        } else {
#pragma unroll
            for (int q = 0; q < NJ / C; ++q) {
                const int n = nw + q * 16 * C + fq * 4 * C;
                uint32_t hi[2 * C], lo[2 * C];
#pragma unroll
                for (int j = 0; j < C; ++j) {
                    f32x4 v = acc[i][q * C + j];
                    if (a.bias != nullptr) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] += bv[q * C + j][r];
                    }
                    if constexpr (EPI == GEPI_ACT_SPLIT) {
                        // 0.5 v (1 + tanh u) = v / (1 + e^-2u).  Against 64 bits, normal v: 4.7e-8 of the row, with tanhf 3.8e-8 -- under the planes' 2^-17, whose rows are
                        // as far off either way
                        if (a.act == 1) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const float x = v[r], u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
                                v[r] = x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.8853900817779268f * u));
                            }
                        } else if (a.act == 2) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) v[r] = 0.5f * v[r] * (1.0f + erff(v[r] * 0.7071067811865476f));
                        }
#pragma unroll
                        for (int r = 0; r < 4; r += 2) {
                            const uint32_t h = pack_bf16x2(v[r], v[r + 1]);
                            hi[j * 2 + r / 2] = h;
                            lo[j * 2 + r / 2] = pack_bf16x2(v[r] - bf16_lo(h), v[r + 1] - bf16_hi(h));
                        }
                    } else {                                              // even column = gate, odd column = up
                        const float x = silu_mul(v[0], v[1]), y = silu_mul(v[2], v[3]);
                        hi[j] = pack_bf16x2(x, y);
                        lo[j] = pack_bf16x2(x - bf16_lo(hi[j]), y - bf16_hi(hi[j]));
                    }
                }
                const size_t at = EPI == GEPI_ACT_SPLIT ? (size_t)m * a.N + n : (size_t)m * (a.N / 2) + (n >> 1);
                constexpr int WORDS = EPI == GEPI_ACT_SPLIT ? 2 * C : C;
                put_words<WORDS>(a.H_hi + at, hi);
                put_words<WORDS>(a.H_lo + at, lo);
            }
        }
    }
}

template <int EPI, int BM, int BN>
void launch_one(const GemmArgs& a, hipStream_t s) {
    static DevOnce attr;
    const size_t lds = ((size_t)4 * BM * 64 + (size_t)2 * BN * (BM == 256 ? 32 : 64)) * 2;
    attr.run([&] { (void)hipFuncSetAttribute((const void*)gemm_tile_kernel<EPI, BM, BN>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
    const int blocks = (a.M + BM - 1) / BM * (a.N / BN) * a.ksplit;
    hipLaunchKernelGGL((gemm_tile_kernel<EPI, BM, BN>), dim3(blocks), dim3(512), lds, s, a);
}
template <int BM, int BN>
void launch_shape(const GemmArgs& a, int epi, hipStream_t s) {
    if (a.ksplit > 1) launch_one<GEPI_PARTIAL, BM, BN>(a, s);
    else if (epi == GEPI_STORE) launch_one<GEPI_STORE, BM, BN>(a, s);
    else if (epi == GEPI_RESADD) launch_one<GEPI_RESADD, BM, BN>(a, s);
    else if (epi == GEPI_ACT_SPLIT) launch_one<GEPI_ACT_SPLIT, BM, BN>(a, s);
    else launch_one<GEPI_SILUMUL, BM, BN>(a, s);
}

}  // namespace

// What M rows take on tiles of bm x bn with K in ks slices, in seconds (norm: a norm of the rows behind the product, in the reduction where K is split, else a launch): `step`
// per 64 of K and `around` for a round of 256 blocks; a round that is not full takes less for each, the clock rises from 1.8 to 2.4 GHz; the reduction's bytes beyond 60 MB come from the
// memory. A fit to 1700 launches of 130 .. 3200 rows over the widths of the 0.6B, 2B and 8B models and of a vision tower, 8 % off in the mean square; the shape it picks is 0.7 % slower
// than the best on average.  (72 launches of 3328 .. 4224 rows, which the passes of one prompt reach: 5 %.)
double gemm_tile_seconds(int M, int N, int K, int bm, int bn, int ks, bool norm) {
    const double step = bm == 256 ? 2.62e-6 : bn == 384 ? 1.97e-6 : bn == 256 ? 1.40e-6 : 1.13e-6;
    const double walk = K / 64 / ks * step, around = 4.5e-6 + 4e-6 * bm * bn / 65536.0, bytes = (double)(2 * ks + 1) * M * N * 4.0;
    const int blocks = (M + bm - 1) / bm * (N / bn) * ks, full = blocks / 256, rest = blocks % 256;
    double t = full * (walk + around);
    if (rest) t += walk * std::max(0.78, 0.56 + 0.44 * rest / 256) + around;
    if (ks > 1) t += bytes / 28e12 + std::max(0.0, bytes - 60e6) / 3e12 + 5e-6;
    else if (norm) t += (double)M * N * 8.0 / 4e12 + 2.5e-6;
    return t;
}
// The tile and the K slices of M > 128 rows that take least by that.  false: no tile divides the width, or fewer than 64 blocks, where the 128-column kernel's smaller tiles
// are as fast (1024 x 2048, norm behind, tiles here / there: 32 blocks 16.1 / 14.4 us, 48 18.6 / 18.4, 64 23.2 / 23.1 of 1024 x 3072, 80 20.0 / 26.4), and up to 256 rows, where
// the memory's latency counts and its smaller tiles have more requests in flight, than 128 (layers of width 1024, 200 rows: 2680 / 2740 us a prompt with 64)
bool gemm_tile_plan(int M, int N, int K, size_t ws_floats, bool norm, int* bm_out, int* bn_out, int* ks_out, double* seconds) {
    if (M <= 128 || K % 64 != 0) return false;
    static constexpr int shapes[4][2] = {{256, 256}, {128, 384}, {128, 256}, {128, 192}};
    const int nk = K / 64;
    double best = 1e30;
    int blocks = 0;
    for (const auto& sh : shapes) {
        const int bm = sh[0], bn = sh[1];
        if (N % bn != 0) continue;
        for (int ks = 1; ks <= 8; ks *= 2) {
            if (nk % ks != 0 || nk / ks < 8 || (ks > 1 && (size_t)ks * M * N > ws_floats)) break;
            const double t = gemm_tile_seconds(M, N, K, bm, bn, ks, norm);
            if (t < best) { best = t; *bm_out = bm; *bn_out = bn; *ks_out = ks; blocks = (M + bm - 1) / bm * (N / bn) * ks; }
        }
    }
    if (seconds != nullptr) *seconds = best;
    return blocks >= (M <= 256 ? 128 : 64);
}
// a.ksplit set; more than one slice: partial tiles in a.ws
bool launch_gemm_tile(const GemmArgs& a, int epi, int bm, int bn, hipStream_t s) {
    if (a.A_lo == nullptr || a.N % bn != 0 || a.K % 64 != 0 || (a.K / 64) % a.ksplit != 0) return false;
    const bool planes = epi == GEPI_ACT_SPLIT || epi == GEPI_SILUMUL;
    if (a.ksplit == 1 && (planes ? a.H_lo == nullptr || (((uintptr_t)a.H_hi | (uintptr_t)a.H_lo) & 15) != 0 : ((uintptr_t)a.C & 15) != 0 || a.ldc % 4 != 0)) return false;      // (16 bytes at a time)
    if (a.bias != nullptr && ((uintptr_t)a.bias & 15) != 0) return false;
    if (bm == 256 && bn == 256) launch_shape<256, 256>(a, epi, s);
    else if (bm == 128 && bn == 384) launch_shape<128, 384>(a, epi, s);
    else if (bm == 128 && bn == 256) launch_shape<128, 256>(a, epi, s);
    else if (bm == 128 && bn == 192) launch_shape<128, 192>(a, epi, s);
    else return false;
    return true;
}

}  // namespace cm
