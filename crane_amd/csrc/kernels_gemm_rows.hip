// Products of 9 .. 128 rows, decode groups and short prompts (from 65 rows on projections of up to 128 column tiles): C[M, N] (+)= A[M, K] . W[N, K]^T with the
// activations as bf16 hi + lo planes, two MFMAs per product -- gemm256_kernel's arithmetic and epilogues on tiles made for a launch that waits
// for its weights.
//
// What bounds it: the weight stream, and from 64 rows on what every column tile reads of the activations out of the L2 (128 rows, gate_up of width
// 4096: 32 KB of them next to 12 KB of weights per tile and k-tile, 11 TB/s in all).  gemm256_kernel's tiles are 192 or 256 columns wide: 96 ..
// 128 workgroups for a 24576-column projection, on half of the chip.  Here a workgroup owns 128 columns, or 96 where that fills the chip better,
// one workgroup on each CU, with two (at 32 rows: three) weight tiles in flight under the one it multiplies.  Tiles go from memory into LDS
// without passing registers (8 rows x 128 bytes per wave instruction, the bank swizzle on the source address: slot p of a row holds its 16-byte
// chunk p ^ ((row >> 1) & 7)), ST stages, one barrier per k-tile.  Narrow projections split K and leave f32 partial tiles for the fixed-order
// reduction kernels.  Measured (us per launch with its reduction, 32 rows, gemm256_kernel / gemm_bf16_kernel -> here):
//   width 4096:  gate_up (24576 x 4096) 50.3 -> 38.0 (5.3 TB/s; 45.0 with all workgroups in step along K), down (4096 x 12288) 34.4 -> 24.4, qkv (6144 x
//                4096) 17.5 -> 14.1, o 15.0 -> 11.6
//   width 2048 (I 6144): layer 58 -> 45;  width 1024 (I 3072): 40 -> 30;  lm_head (151936 x 4096) 385 -> 226 (5.5 TB/s; 275 in step)
// Tiles of 64 columns, weight loads that bypass the caches, two workgroups per CU with fewer stages and two k-tiles per barrier were all no faster.
#include "dev_common.h"
#include "kernels.h"

namespace cm {

namespace {

constexpr int RBK = 64;
// k-tiles between the starts of neighbouring workgroups of an XCD.  In step, all workgroups ask for the same columns of all rows, and those reach a part
// of the memory channels.  Rows of 8 KB read by 256 workgroups as here: 42 us for 201 MB (36.5 for the 8 matrices of 36 that happen to lie well), 36.0 with
// four starts 2 KB apart, 37 .. 39 with as many as there are workgroups, 43 with two
constexpr int K_TURN = 16;

template <int BM, int RBN, int ST, int EPI, int NW>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void gemm_rows_kernel(GemmArgs a) {
    constexpr int GM = RBN == 96 ? NW / 2 : NW == 8 ? (BM == 128 ? 4 : 2) : BM == 32 ? 1 : 2, GN = NW / GM, WM = BM / GM, WN = RBN / GN, NI = WM / 16, NJ = WN / 16;      // NW waves GM x GN, WM x WN outputs each
    constexpr int PLANE = BM * RBK, STAGE = 2 * PLANE + RBN * RBK;
    constexpr int APC = BM / 8, NP = 2 * APC + RBN / 8, NL = (NP + NW - 1) / NW;                          // pieces per plane / requests per wave and k-tile
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / GN, wn = wave % GN;
    const int tiles = a.N / RBN, ks = (int)blockIdx.x / tiles, n0 = ((int)blockIdx.x - ks * tiles) * RBN;
    const int K = a.K, kpb = K / RBK / a.ksplit, kbeg = ks * kpb;

    const int prow = lane >> 3, pslot = lane & 7;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    const uint16_t* src[NL];
    uint32_t dst[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int p = min(wave + NW * i, NP - 1), plane = p / APC;                                   // 0: hi, 1: lo, 2 and up: weights
        const int r0 = (plane < 2 ? p - plane * APC : p - 2 * APC) * 8, row = r0 + prow;
        const size_t kc = (size_t)kbeg * RBK + (size_t)((pslot ^ ((row >> 1) & 7)) << 3);
        const bool isw = plane >= 2;
        src[i] = isw ? a.W + (size_t)(n0 + row) * K + kc : (plane ? a.A_lo : a.A_hi) + (size_t)min(row, a.M - 1) * K + kc;
        dst[i] = lds0 + (uint32_t)((isw ? 2 * PLANE : plane * PLANE) + r0 * RBK) * 2u;
    }
    // (slices of K start apart by themselves: 16.0 / 16.3 us with a turn on top; so do the 128-row tiles, which all have slices)
    const int turn = EPI != GEPI_PARTIAL && BM < 128 ? ((int)blockIdx.x >> 3 & 3) * K_TURN % kpb : 0;
    auto request = [&](int t) __attribute__((always_inline)) {                          // past the end: the last tile again, into a stage nobody reads
        const int k = min(t, kpb - 1) + turn;
        const size_t at = (size_t)(k < kpb ? k : k - kpb) * RBK;
        const uint32_t stage = (uint32_t)((t % ST) * STAGE) * 2u;
#pragma unroll
        for (int i = 0; i < NL; ++i) lds_load16(src[i] + at, dst[i] + stage);
    };
    f32x4 acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int fr = lane & 15, lg = lane >> 4, sw = (fr >> 1) & 7;
#pragma unroll
    for (int t = 0; t < ST - 1; ++t) request(t);
    for (int t = 0; t < kpb; ++t) {
        // this wave's share of tile t has landed and its reads of tile t - 1 are done; behind the barrier that holds for every wave
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * NL) : "memory");
        request(t + ST - 1);
        const uint16_t* S = lds + (t % ST) * STAGE;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int fk = ((s * 4 + lg) ^ sw) << 3;
            bf16x8 ah[NI], al[NI], bf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) bf[j] = *(const bf16x8*)&S[2 * PLANE + (wn * WN + j * 16 + fr) * RBK + fk];
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                ah[i] = *(const bf16x8*)&S[(wm * WM + i * 16 + fr) * RBK + fk];
                al[i] = *(const bf16x8*)&S[PLANE + (wm * WM + i * 16 + fr) * RBK + fk];
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bf[j], acc[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bf[j], acc[i][j], 0, 0, 0);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                    // no request of the tail may land after the block is gone
    // D of a product: column = lane % 16, rows 4 (lane / 16) + r
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = wm * WM + i * 16 + lg * 4 + r;
            const bool ok = m < a.M;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int n = n0 + wn * WN + j * 16 + fr;
                float v = acc[i][j][r];
                if (EPI == GEPI_PARTIAL) {
                    if (ok) a.ws[((size_t)ks * a.M + m) * a.N + n] = v;
                    continue;
                }
                if (a.bias != nullptr) v += a.bias[n];
                if (EPI == GEPI_STORE) {
                    if (ok) a.C[(size_t)m * a.ldc + n] = v;
                } else if (EPI == GEPI_RESADD) {
                    if (ok) a.C[(size_t)m * a.ldc + n] += v;
                } else {                                                                // GEPI_SILUMUL: even column = gate_j, odd column = up_j
                    const float up = dpp_mov<0xB1>(v);                                  // lane ^ 1
                    if (((lane & 1) == 0) && ok) {
                        const float h = (v / (1.0f + expf(-v))) * up;
                        const size_t off = (size_t)m * (a.N / 2) + (n >> 1);
                        const uint16_t hh = f32_to_bf16(h);
                        a.H_hi[off] = hh;
                        if (a.H_lo) a.H_lo[off] = f32_to_bf16(h - bf16_to_f32(hh));
                    }
                }
            }
        }
}

template <int BM, int RBN, int ST, int EPI, int NW>
void go(const GemmArgs& a, hipStream_t s) {
    constexpr size_t lds = (size_t)ST * (2 * BM + RBN) * RBK * sizeof(uint16_t);
    static DevOnce attr;
    attr.run([&] { (void)hipFuncSetAttribute((const void*)gemm_rows_kernel<BM, RBN, ST, EPI, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
    hipLaunchKernelGGL((gemm_rows_kernel<BM, RBN, ST, EPI, NW>), dim3((unsigned)(a.N / RBN * a.ksplit)), dim3(64 * NW), lds, s, a);
}
template <int BM, int RBN, int ST, int NW>
void go_epi(const GemmArgs& a, int epi, hipStream_t s) {
    if (a.ksplit > 1) go<BM, RBN, ST, GEPI_PARTIAL, NW>(a, s);
    else if (epi == GEPI_STORE) go<BM, RBN, ST, GEPI_STORE, NW>(a, s);
    else if (epi == GEPI_RESADD) go<BM, RBN, ST, GEPI_RESADD, NW>(a, s);
    else go<BM, RBN, ST, GEPI_SILUMUL, NW>(a, s);
}

}  // namespace

// Where the lines lie (both sides measured, old kernels / these, us): more than one round of workgroups pays only while the last round is well
// filled -- 272 tiles (34816 x 5120, 64 rows) 98 / 124, 1187 tiles 391 / 290; above 64 rows a launch is bound by its activations as much as by the
// weights, and wide projections stay with the wider tiles -- 192 tiles at 128 rows 62 / 78, 1187 tiles 405 / 405, while 32 .. 48 tiles split 4
// ways 46 / 38 and 28 / 24.  A slice of K keeps at least four k-tiles: the pipeline's fill costs two or three.  96 columns where they fill more of
// the last round (24576 columns: 256 workgroups for 192, 46.5 -> 44.6 at 32 rows, 53.5 -> 49.2 at 64; 6144: 4 x 64 for 4 x 48, 14.7 -> 14.1).
static int rows_split(int M, int N, int K, int bn, size_t ws_floats) {
    const int tiles = N / bn, nk = K / RBK;
    int ks = 1;
    while (ks < 8 && 2 * ks * tiles <= 256 && nk % (2 * ks) == 0 && nk / (2 * ks) >= 4 && (size_t)2 * ks * M * N <= ws_floats) ks *= 2;
    return ks;
}
bool gemm_rows_plan(int M, int N, int K, size_t ws_floats, int* bn, int* ks) {
    if (M < 9 || M > 128 || K % RBK != 0) return false;
    double best = 0.0;
    for (int b : {128, 96}) {
        if (N % b != 0) continue;
        const int tiles = N / b, s = rows_split(M, N, K, b, ws_floats), rounds = (tiles * s + 255) / 256;
        const double fill = (double)tiles * s / (rounds * 256);
        if (tiles > 256 && fill < 0.9) continue;
        if (M > 64 && tiles > 128) continue;
        if (fill > best + 0.05) { best = fill; *bn = b; *ks = s; }
    }
    return best > 0.0;
}

// a.ksplit set by the caller (1: epilogue `epi`; > 1: partial tiles, the caller runs the reduction)
bool launch_gemm_rows(const GemmArgs& a, int epi, int bn, hipStream_t s) {
    if (a.M > 128 || a.A_lo == nullptr || a.N % bn != 0 || a.K % (RBK * a.ksplit) != 0 || epi == GEPI_ACT_SPLIT) return false;
    // (eight waves against four: 128 rows 153 -> 147 us for the layer of width 4096, 32 rows 98 -> 96; the 96-column tiles of up to 64 rows have no
    // use for them: 17.9 / 16.8 us for the qkv of 64 rows)
    if (bn == 96) {
        if (a.M <= 32) go_epi<32, 96, 4, 4>(a, epi, s);
        else if (a.M <= 64) go_epi<64, 96, 3, 4>(a, epi, s);
        else go_epi<128, 96, 3, 8>(a, epi, s);
    }
    else if (a.M <= 32) go_epi<32, 128, 4, 8>(a, epi, s);
    else if (a.M <= 64) go_epi<64, 128, 3, 8>(a, epi, s);
    else go_epi<128, 128, 3, 8>(a, epi, s);
    return true;
}

}  // namespace cm
