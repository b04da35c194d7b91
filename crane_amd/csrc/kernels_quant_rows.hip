// Decode groups of up to 64 rows over Q8_0-layout weights on the int8 matrix cores: gemm_q8_i8_kernel's products, scales and sums (one
// v_mfma_i32_32x32x32_i8 per 32-block and 32 x 32 outputs, acc = fma(dw * dx, dot, acc) over the blocks in order, the same K slices: bit for bit
// the same outputs) around a pipeline made for a launch that waits for its weights.
//
// What bounds it: the weight stream, its start, and the scaling of the dots on the vector units (48 instructions per 32 x 32 outputs and block).  A
// slice of a Qwen3-8B projection is 2 .. 16 groups of 128 codes per row; with one group on its way per workgroup, through registers, a launch was
// mostly waiting.  Here a group (16 KB of weight codes, 4 KB of activation codes per 32 rows, their scales) goes from memory into one of two
// stages of LDS while the other is multiplied, 45 KB per workgroup: three on every CU.  Rows of a group are 128 bytes in LDS, 16-byte chunks moved
// by an XOR of the row (on the source address) so that 16 rows of a fragment read do not meet in a bank; the weight scales stay f16 and are widened
// by the multiplication that uses them.  Measured (us per launch, 20 rows, gemm_q8_i8_kernel -> here): gate_up (24576 x 4096, two slices) 32.7 ->
// 25.5, down (4096 x 12288, sixteen) 19.3 -> 15.4, qkv (6144 x 4096, eight) 14.2 -> 10.3, o 10.8 -> 7.7; a layer pair of width 1024 and the head
// at 16 rows 210 -> 191.  Three and more stages were no faster (12.6 / 17.4 against 11.6 for o and down): workgroups on a CU count for more.
#include <algorithm>
#include "dev_common.h"
#include "kernels.h"

namespace cm {

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

// f32 product of one half of a register and x: the widening and the multiplication in one instruction, rounded once like (float)half * x
template <int HI>
__device__ __forceinline__ float half_times(uint32_t w, float x) {
    float r;
    if constexpr (HI) asm("v_fma_mix_f32 %0, %1, %2, neg(0) op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(x));
    else asm("v_fma_mix_f32 %0, %1, %2, neg(0) op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(x));
    return r;
}
__device__ __forceinline__ float f16r(float v) { return (float)(_Float16)v; }

constexpr int QG = 4, GB = QG * 32, ST = 2;                    // blocks and bytes of a row per group, stages

// weight codes and scales, activation codes and scales of a stage
template <int NW, int MT> constexpr int stage_bytes() { return NW * 32 * (GB + QG * 2) + MT * 32 * (GB + QG * 4) + (NW == 4 && MT == 1 ? 512 : 0); }

// workgroup: 32 NW weight rows (wave w: rows 32 w ..) x 32 MT activation rows x one K slice
template <int NW, int MT>
__global__ __launch_bounds__(64 * NW, 2) void gemm_q8_rows_kernel(QGemmArgs a) {
    constexpr int STAGE = stage_bytes<NW, MT>(), TN = 32 * NW, NT = 64 * NW, PR = 32 * MT, WB = TN * GB, SB = TN * QG * 2;
    constexpr int AI = 4 * MT / NW, XI = NW == 4 && MT == 1 ? 1 : 2 * MT / NW;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int K = a.w.K, N = a.w.N, nkb = K >> 5, G = nkb / QG, tiles = N / TN;
    const int ks = (int)blockIdx.x / tiles, tn = (int)blockIdx.x - ks * tiles;
    const int g0 = ks * G / a.ksplit, n = (ks + 1) * G / a.ksplit - g0;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    const int prow = lane >> 3, pslot = lane & 7;
    const uint8_t* wsrc[4];
    const signed char* xsrc[AI];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = wave * 32 + 8 * i + prow;
        wsrc[i] = a.w.p0 + (size_t)(tn * TN + row) * K + (size_t)g0 * GB + ((pslot ^ ((row >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < AI; ++i) {
        const int row = (wave * AI + i) * 8 + prow;            // (rows past M: the last one again, dropped at the store)
        xsrc[i] = a.xq + (size_t)min(row, a.M - 1) * K + (size_t)g0 * GB + ((pslot ^ ((row >> 1) & 7)) << 4);
    }
    const uint8_t* ssrc = (const uint8_t*)a.w.p1 + ((size_t)(tn * TN + wave * 32 + (lane >> 1)) * nkb + (size_t)g0 * QG) * 2 + (lane & 1) * 4;
    // activation scales [block][row] of the group: 128 MT floats (four waves, MT = 1: two of them bring the same again, into space nobody reads)
    const float* dsrc[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int e = ((wave * XI + i) * 64 + lane) % (QG * PR);
        dsrc[i] = a.xd + ((size_t)g0 * QG + e / PR) * a.xs + e % PR;
    }
    auto request = [&](int g) __attribute__((always_inline)) {
        const uint32_t st = lds0 + (uint32_t)((g % ST) * STAGE);
#pragma unroll
        for (int i = 0; i < 4; ++i) lds_load16(wsrc[i] + (size_t)g * GB, st + (uint32_t)((wave * 4 + i) * 1024));
#pragma unroll
        for (int i = 0; i < AI; ++i) lds_load16(xsrc[i] + (size_t)g * GB, st + (uint32_t)(WB + (wave * AI + i) * 1024));
        lds_load4(ssrc + (size_t)g * (QG * 2), st + (uint32_t)(WB + PR * GB + wave * 256));
#pragma unroll
        for (int i = 0; i < XI; ++i) lds_load4(dsrc[i] + (size_t)g * QG * a.xs, st + (uint32_t)(WB + PR * GB + SB + (wave * XI + i) * 256));
    };
    float acc[MT][16];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;
    const int sw = (r >> 1) & 7;
    request(0);
    for (int g = 0; g < n; ++g) {
        // this wave's share of group g has landed and its reads of group g - 1 are done; behind the barrier that holds for every wave
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (g + 1 < n) request(g + 1);
        const unsigned char* S = lds + (g % ST) * STAGE;
        const float* dx = (const float*)(S + WB + PR * GB + SB);
        u32x4 sc[4][2];                                         // scales of weight rows 8 q + 4 h + 2 p, + 1: four f16 each
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int p = 0; p < 2; ++p) sc[q][p] = *(const u32x4*)(S + WB + PR * GB + wave * 256 + (8 * q + 4 * h + 2 * p) * 8);
#pragma unroll
        for (int j = 0; j < QG; ++j) {
            const int at = ((2 * j + h) ^ sw) << 4;
            const i32x4 wf = *(const i32x4*)(S + (wave * 32 + r) * GB + at);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const i32x4 xf = *(const i32x4*)(S + WB + (mt * 32 + r) * GB + at);
                const i32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                const i32x16 c = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf, xf, zero, 0, 0, 0);
                const float d = dx[j * PR + mt * 32 + r];
                // c[i] of lane (r, h): weight row 8 (i / 4) + 4 h + i % 4 of the strip, activation row r
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t w = sc[i >> 2][(i >> 1) & 1][(i & 1) * 2 + (j >> 1)];
                    acc[mt][i] = fmaf(j & 1 ? half_times<1>(w, d) : half_times<0>(w, d), (float)c[i], acc[mt][i]);
                }
            }
        }
    }
    float* P = a.ws + (size_t)ks * a.slice;
    if (!a.silu) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 32 + r;
            if (m >= a.M) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *(f32x4*)(P + (size_t)m * a.ldp + tn * TN + wave * 32 + 4 * h + 8 * q) = (f32x4){acc[mt][4 * q], acc[mt][4 * q + 1], acc[mt][4 * q + 2], acc[mt][4 * q + 3]};
        }
        return;
    }
    // unsplit gate|up: columns (2 k, 2 k + 1) = (gate_k, up_k) sit in one lane.  The 64 outputs of a row through LDS: whole 256-byte runs to
    // memory, and two Q8_0 blocks of the down projection's input (quant_rows_q8_kernel's arithmetic) where the caller asks for them
    constexpr int TS = TN / 2 + 4;
    float* T = (float*)lds;
    __syncthreads();                                            // every wave's reads of the last stages are done
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float gate = acc[mt][2 * i], up = acc[mt][2 * i + 1];
            T[(mt * 32 + r) * TS + wave * 16 + 2 * h + 4 * (i >> 1) + (i & 1)] = (gate / (1.0f + expf(-gate))) * up;
        }
    __syncthreads();
    for (int it = tid; it < PR * (TN / 8); it += NT) {
        const int row = it / (TN / 8), c4 = it % (TN / 8);
        if (row < a.M) *(f32x4*)(P + (size_t)row * a.ldp + tn * (TN / 2) + 4 * c4) = *(const f32x4*)(T + row * TS + 4 * c4);
    }
    if (a.nxq == nullptr) return;
    const int nout = N >> 1, l8 = tid & 7;
    for (int it = tid >> 3; it < PR * (NW / 2); it += NT / 8) {
        const int row = it / (NW / 2), b = it % (NW / 2);
        const f32x4 v = *(const f32x4*)(T + row * TS + b * 32 + 4 * l8);
        float am = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
        am = fmaxf(am, __shfl_xor(am, 1)); am = fmaxf(am, __shfl_xor(am, 2)); am = fmaxf(am, __shfl_xor(am, 4));
        const float d = am / 127.0f;
        const float id = d != 0.f ? 1.0f / d : 0.f;
        uint32_t pk = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) pk |= ((uint32_t)(int)roundf(v[e] * id) & 0xFFu) << (8 * e);
        if (row < a.M) {
            ((uint32_t*)(a.nxq + (size_t)row * nout))[(tn * (NW / 2) + b) * 8 + l8] = pk;
            if (l8 == 0) a.nxd[(size_t)(tn * (NW / 2) + b) * a.xs + row] = f16r(d);
        }
    }
}

template <int NW, int MT>
void go(const QGemmArgs& a, hipStream_t s) {
    constexpr size_t lds = std::max(ST * (size_t)stage_bytes<NW, MT>(), (size_t)32 * MT * (16 * NW + 4) * 4);
    static DevOnce attr;
    attr.run([&] { (void)hipFuncSetAttribute((const void*)gemm_q8_rows_kernel<NW, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
    hipLaunchKernelGGL((gemm_q8_rows_kernel<NW, MT>), dim3((unsigned)(a.w.N / (32 * NW) * a.ksplit)), dim3(64 * NW), lds, s, a);
}

}  // namespace

void launch_gemm_q8_rows(const QGemmArgs& a, int num_cu, hipStream_t s) {
    // 64 weight rows per workgroup while 128 would leave CUs with one workgroup where others have two and the slices are long (gate_up of width
    // 4096: 384 workgroups of 16 groups 29.7 -> 25.5 us; qkv, 4 groups, 10.9 -> 10.3); slices of one or two groups lose by it (width 1024, a layer
    // pair of 16 rows 193 -> 205 us), and so do 33 rows and more (464 -> 513)
    const bool narrow = a.M <= 32 && a.w.N / 128 * a.ksplit < 2 * num_cu && (a.w.K >> 5) / QG >= 4 * a.ksplit;
    if (narrow) go<2, 1>(a, s);
    else if (a.M <= 32) go<4, 1>(a, s);
    else go<4, 2>(a, s);
}

}  // namespace cm
