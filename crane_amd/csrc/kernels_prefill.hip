// Prefill (S > 1) kernels for gfx950: MFMA-bound.
//
// Replaces the S>1 branch of Qwen3Model::decode (reference qwen3/modeling.rs:984-1036): candle
// GEMMs + an O(S*L) materialised score matrix with an additive -1e9 mask (modeling.rs:493-532,
// 1000-1017), or the CPU flash_attn path (modeling.rs:422-456).  Here:
//   * every projection is one bf16 MFMA GEMM  C[M,N] = A[M,K] . W[N,K]^T  with f32 accumulate;
//     the ACTIVATION operand is carried as a 2-term bf16 split (hi = bf16(x), lo = bf16(x-hi)),
//     so activations keep ~16 mantissa bits and logits stay within the 1e-3 parity bar
//     against the f32 CPU reference (plain bf16 activations measure 1.7e-3 on 12 layers);
//     cm_opts.prefill_split = 1 selects plain bf16 (half the MFMA work);
//   * attention is a causal flash kernel over the paged KV cache: S^T = K.Q^T
//     (mfma 16x16x32), online softmax with lane-local row statistics, O^T = V^T.P^T
//     (mfma 16x16x16, V fragments through ds_read_b64_tr_b16), nothing O(S*L) in HBM.
#include <cstdlib>

#include <type_traits>

#include "dev_common.h"
#include "kernels.h"

namespace cm {

// ---------------------------------------------------------------------------------------------
// small row kernels
// ---------------------------------------------------------------------------------------------
__global__ void embed_rows_kernel(const uint16_t* __restrict__ emb, const uint32_t* __restrict__ ids,
                                  float* __restrict__ x, int H, int V) {
    const int row = blockIdx.x;
    uint32_t tok = ids[row];
    if (tok >= (uint32_t)V) tok = 0;
    for (int i = threadIdx.x * 4; i < H; i += blockDim.x * 4) {
        const u32x2 p = *(const u32x2*)(emb + (size_t)tok * H + i);
        *(f32x4*)(x + (size_t)row * H + i) = (f32x4){bf16_lo(p[0]), bf16_hi(p[0]), bf16_lo(p[1]), bf16_hi(p[1])};
    }
}


// one block per token row: out = x * w / sqrt(mean(x^2)+eps) -> bf16 hi (+ lo)
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                                           int H, float eps) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float* xr = x + (size_t)row * H;
    float ss = 0.f;
    for (int i = tid * 4; i < H; i += 1024) {
        const f32x4 v = *(const f32x4*)(xr + i);
        ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    const float r = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)H + eps);
    for (int i = tid * 4; i < H; i += 1024) {
        const f32x4 v = *(const f32x4*)(xr + i);
        const f32x4 ww = *(const f32x4*)(w + i);
        const float o[4] = {v[0] * r * ww[0], v[1] * r * ww[1], v[2] * r * ww[2], v[3] * r * ww[3]};
        split_store4(hi, lo, (size_t)row * H + i, o);
    }
}

// grid (S, Hq + 2 Hkv), block 64: per-head RMSNorm(q,k) BEFORE RoPE (qwen3/modeling.rs:341-359,
// qwen3_5/modeling.rs:464-468), rotate-half over the first rot_dim dims, q scaled by 1/sqrt(D)
// -> bf16 hi/lo [S, Hq, D]; k, v -> paged cache at position start+s.
template <int D, int KVT>
__global__ __launch_bounds__(64) void qknorm_rope_kv_kernel(QkRopeArgs a_in) {
    QkRopeArgs a = a_in;
    if (a.segs != nullptr) {          // a pass over several sequences: this row's sequence gives position, page table and rope offset
        const PrefillSegDev sg = a.segs[a.rowseg[blockIdx.x]];
        a.start_pos = sg.start_pos - sg.row0;          // (position = start_pos + row of the pass)
        a.block_table += sg.bt_off;
        a.rope_delta = sg.rope_delta;
    }
    constexpr int EPL = D / 64;
    constexpr bool KVF32 = KVT == 1;
    __shared__ float tmp[D];
    const int s = blockIdx.x, item = blockIdx.y, lane = threadIdx.x;
    const int Hq = a.Hq, Hkv = a.Hkv;
    const int pos = a.start_pos + s;
    const bool is_q = item < Hq, is_k = !is_q && item < Hq + Hkv;
    const int kvh = is_k ? item - Hq : item - Hq - Hkv;
    const float* src = a.qkv + (size_t)s * a.row_stride +
                       (is_q ? a.q_off + item * D : (is_k ? a.k_off + kvh * D : a.v_off + kvh * D));
    float xv[EPL];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < EPL; ++j) { xv[j] = src[lane + 64 * j]; ss += xv[j] * xv[j]; }
    if (is_q || is_k) {
        const float* nw = is_q ? a.qnw : a.knw;
        if (nw) {
            ss = wave_sum(ss);
            const float r = 1.0f / sqrtf(ss / (float)D + a.eps);
#pragma unroll
            for (int j = 0; j < EPL; ++j) xv[j] = xv[j] * r * nw[lane + 64 * j];
        }
        const int rot = a.rot_dim, hrot = rot >> 1;
#pragma unroll
        for (int j = 0; j < EPL; ++j) tmp[lane + 64 * j] = xv[j];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            const int d = lane + 64 * j;
            if (d < rot) {
                const int i = d < hrot ? d : d - hrot;
                int rp = pos + a.rope_delta;
                if (a.pos3 != nullptr) {   // index-interleaved MRoPE (qwen3_5/modeling.rs:156-245): column i -> axis i % 3
                    const int ax = (i % 3 == 1 && i < 3 * a.sec_h) ? 1 : ((i % 3 == 2 && i < 3 * a.sec_w) ? 2 : 0);
                    rp = a.pos3[ax * a.pos3_stride + s];
                }
                const float c = a.cos[(size_t)rp * hrot + i], sn = a.sin[(size_t)rp * hrot + i];
                const float lo = tmp[i], hi = tmp[i + hrot];
                xv[j] = d < hrot ? lo * c - hi * sn : lo * sn + hi * c;
            }
        }
    }
    if (is_q) {
        const size_t off = ((size_t)s * Hq + item) * D;
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            // (f16 pages: the flash kernel multiplies cached halves with q on the f16 matrix-core path, so q is split into f16 hi + lo)
            const float x = xv[j] * a.scale;
            const uint16_t h = kv16_from_f32<KVT>(x);
            a.q_hi[off + lane + 64 * j] = h;
            a.q_lo[off + lane + 64 * j] = kv16_from_f32<KVT>(x - kv16_to_f32<KVT>(h));
        }
    } else if (KVT == KV_INT8 || KVT == KV_INT4) {
        // quantize_per_token (qwen3_5/kv_cache.rs:253-268), same arithmetic as the decode kernel's append
        constexpr float QMAX = KVT == 2 ? 127.f : 7.f, OFFS = KVT == 2 ? 128.f : 8.f;
        constexpr int ROWB = KVT == 2 ? D : D / 2;
        float amax = 0.f;
#pragma unroll
        for (int j = 0; j < EPL; ++j) amax = fmaxf(amax, fabsf(xv[j]));
        amax = wave_max(amax);
        const float scale = __fadd_rn(__fmul_rn(amax, (float)(1.0 / (double)QMAX)), 1e-8f);
        uint8_t* pb = (uint8_t*)(is_k ? a.kpool : a.vpool);
        float* sh = is_k ? a.kshadow : a.vshadow;
        const int page = a.block_table[pos / a.page];
        const size_t roff = (size_t)page * a.page_bytes + (size_t)(kvh * a.page + (pos % a.page)) * ROWB;
        const size_t soff = (size_t)page * a.page_bytes + (size_t)Hkv * a.page * ROWB + (size_t)(kvh * a.page + (pos % a.page)) * 4;
        const size_t hoff = ((size_t)((pos / a.page) * Hkv + kvh) * a.page + (pos % a.page)) * D;       // shadow: identity pages
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            const int d = lane + 64 * j;
            const float code = roundf(__fdiv_rn(xv[j], scale)) + OFFS;
            sh[hoff + d] = __fmul_rn(code - OFFS, scale);
            const uint32_t ci = (uint32_t)(int)code;
            if (KVT == 2) pb[roff + d] = (uint8_t)ci;
            else {
                const uint32_t hi = (uint32_t)__shfl_down((int)ci, 1);
                if (!(lane & 1)) pb[roff + (d >> 1)] = (uint8_t)(ci | (hi << 4));
            }
        }
        if (lane == 0) *(float*)(pb + soff) = scale;
    } else {
        void* pool = is_k ? a.kpool : a.vpool;
        const int page = a.block_table[pos / a.page];
        const size_t off = ((size_t)(page * Hkv + kvh) * a.page + (pos % a.page)) * D;
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            if (KVF32) ((float*)pool)[off + lane + 64 * j] = xv[j];
            else ((uint16_t*)pool)[off + lane + 64 * j] = kv16_from_f32<KVT>(xv[j]);
        }
    }
}

// The same for the common dense case -- head_dim 128, rotation over the whole head, one rotary position per token, bf16 / f16 / f32
// pages -- four elements per thread: the kernel above is (S, Hq + 2 Hkv) workgroups of ONE wave with 4-byte loads and
// 2-byte stores (49 152 workgroups and 27 us per layer for a 1024-token prompt of Qwen3-8B: every wave is a chain of dependent
// loads).  Here 32 lanes own a head (4 consecutive d each; the rotate-half partner is 16 lanes away, the per-head sum of squares an
// xor tree over the 32 lanes) and a 256-thread block takes 8 heads of a token.  Per element the same expressions; the sum of squares
// is associated differently (last-ulp differences of the norm's scale).
template <int KVT>
__global__ __launch_bounds__(256) void qknorm_rope_kv4_kernel(QkRopeArgs a_in) {
    constexpr int D = 128;
    constexpr bool KVF32 = KVT == 1;
    QkRopeArgs a = a_in;
    if (a.segs != nullptr) {
        const PrefillSegDev sg = a.segs[a.rowseg[blockIdx.x]];
        a.start_pos = sg.start_pos - sg.row0;
        a.block_table += sg.bt_off;
        a.rope_delta = sg.rope_delta;
    }
    const int s = blockIdx.x, item = (int)blockIdx.y * 8 + ((int)threadIdx.x >> 5), l32 = threadIdx.x & 31, d0 = l32 * 4;
    const int Hq = a.Hq, Hkv = a.Hkv;
    if (item >= Hq + 2 * Hkv) return;                          // (whole heads: 32 lanes leave together)
    const int pos = a.start_pos + s;
    const bool is_q = item < Hq, is_k = !is_q && item < Hq + Hkv;
    const int kvh = is_k ? item - Hq : item - Hq - Hkv;
    const float* src = a.qkv + (size_t)s * a.row_stride + (is_q ? a.q_off + item * D : (is_k ? a.k_off + kvh * D : a.v_off + kvh * D));
    f32x4 xv = *(const f32x4*)(src + d0);
    // a split projection's slices, as gemm_splitk_epilogue_kernel adds them (its launch in front of this one: 5.4 + 5.2 us for 117 rows of 6144 columns in four slices, 5.3 here alone;
    // 117 tokens of the 8B model 5.98 -> 5.89 ms, of the 0.6B model 2.03 -> 1.95)
    for (int k = 1; k < a.parts; ++k) {
        const f32x4 p = *(const f32x4*)(src + (size_t)k * a.part + d0);
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[e] += p[e];
    }
    if (is_q || is_k) {
        const float* nw = is_q ? a.qnw : a.knw;
        if (nw) {
            float ss = xv[0] * xv[0] + xv[1] * xv[1] + xv[2] * xv[2] + xv[3] * xv[3];
            ss += lane_xor<1>(ss); ss += lane_xor<2>(ss); ss += lane_xor<4>(ss); ss += lane_xor<8>(ss); ss += lane_xor<16>(ss);
            const float r = 1.0f / sqrtf(ss / (float)D + a.eps);
            const f32x4 w4 = *(const f32x4*)(nw + d0);
#pragma unroll
            for (int e = 0; e < 4; ++e) xv[e] = xv[e] * r * w4[e];
        }
        const int rp = pos + a.rope_delta, i0 = d0 & 63;
        const f32x4 c4 = *(const f32x4*)(a.cos + (size_t)rp * 64 + i0), s4 = *(const f32x4*)(a.sin + (size_t)rp * 64 + i0);
        // x c -+ other s: elements 0 and 1 of four with one rounding at the end, 2 and 3 with one more.  Written out, so that pages, and the codes made of rows that have read them, stay
        // what they are however the compiler would contract these
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
            const float other = lane_xor<16>(xv[e]), p = other * s4[e], y = d0 < 64 ? -p : p;         // other: d < 64: x[d + 64], else x[d - 64]
            xv[e] = e < 2 ? __builtin_fmaf(xv[e], c4[e], y) : xv[e] * c4[e] + y;
        }
    }
    auto pack4 = [&](const float (&v)[4], u32x2& o) {
        o[0] = (uint32_t)kv16_from_f32<KVT>(v[0]) | ((uint32_t)kv16_from_f32<KVT>(v[1]) << 16);
        o[1] = (uint32_t)kv16_from_f32<KVT>(v[2]) | ((uint32_t)kv16_from_f32<KVT>(v[3]) << 16);
    };
    if (is_q) {
        const size_t off = ((size_t)s * Hq + item) * D + d0;
        float x[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[e] = xv[e] * a.scale; lo[e] = x[e] - kv16_to_f32<KVT>(kv16_from_f32<KVT>(x[e])); }
        u32x2 ph, pl;
        pack4(x, ph); pack4(lo, pl);
        *(u32x2*)(a.q_hi + off) = ph;
        *(u32x2*)(a.q_lo + off) = pl;
    } else {
        void* pool = is_k ? a.kpool : a.vpool;
        const int page = a.block_table[pos / a.page];
        const size_t off = ((size_t)(page * Hkv + kvh) * a.page + (pos % a.page)) * D + d0;
        if (KVF32) *(f32x4*)((float*)pool + off) = xv;
        else {
            const float v[4] = {xv[0], xv[1], xv[2], xv[3]};
            u32x2 pk;
            pack4(v, pk);
            *(u32x2*)((uint16_t*)pool + off) = pk;
        }
    }
}

// chunked prefill over a quantised cache: the tokens already cached are dequantised into the f32 shadow first
// grid (tokens, 2 * Hkv), one wave per (token, K|V, kv head)
template <int D, int KVT>
__global__ __launch_bounds__(64) void kvq_dequant_prefix_kernel(const uint8_t* __restrict__ kpool, const uint8_t* __restrict__ vpool,
                                                                const int32_t* __restrict__ block_table, float* __restrict__ kshadow,
                                                                float* __restrict__ vshadow, int Hkv, int page, size_t page_bytes) {
    constexpr int ROWB = KVT == 2 ? D : D / 2;
    constexpr float OFFS = KVT == 2 ? 128.f : 8.f;
    const int t = blockIdx.x, kvh = blockIdx.y % Hkv, lane = threadIdx.x;
    const bool is_k = (int)blockIdx.y < Hkv;
    const uint8_t* pb = is_k ? kpool : vpool;
    float* sh = is_k ? kshadow : vshadow;
    const int pg = block_table[t / page];
    const size_t roff = (size_t)pg * page_bytes + (size_t)(kvh * page + (t % page)) * ROWB;
    const float scale = *(const float*)(pb + (size_t)pg * page_bytes + (size_t)Hkv * page * ROWB + (size_t)(kvh * page + (t % page)) * 4);
    const size_t hoff = ((size_t)((t / page) * Hkv + kvh) * page + (t % page)) * D;
    for (int d = lane; d < D; d += 64) {
        float code;
        if (KVT == 2) code = (float)pb[roff + d];
        else { const uint8_t b = pb[roff + (d >> 1)]; code = (float)((d & 1) ? (b >> 4) : (b & 0xF)); }
        sh[hoff + d] = __fmul_rn(code - OFFS, scale);
    }
}

// f32 rows -> bf16 hi (+lo) rows (A operand of the next GEMM)
__global__ void split_rows_kernel(const float* __restrict__ x, uint16_t* __restrict__ hi, uint16_t* __restrict__ lo, size_t n4) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
        const f32x4 v = ((const f32x4*)x)[i];
        const float o[4] = {v[0], v[1], v[2], v[3]};
        split_store4(hi, lo, i * 4, o);
    }
}

// the same for `rows` rows of `cols` columns that sit ldx floats apart (batched decode: the attention / GDN output rows)
__global__ void split_rows2d_kernel(const float* __restrict__ x, int ldx, uint16_t* __restrict__ hi, uint16_t* __restrict__ lo, int cols) {
    const float* xr = x + (size_t)blockIdx.x * ldx;
    for (int c = threadIdx.x * 4; c < cols; c += blockDim.x * 4) {
        const f32x4 v = *(const f32x4*)(xr + c);
        const float o[4] = {v[0], v[1], v[2], v[3]};
        split_store4(hi, lo, (size_t)blockIdx.x * cols + c, o);
    }
}

__global__ void add_rows_kernel(float* __restrict__ x, const float* __restrict__ y, size_t n4) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
        f32x4 a = ((const f32x4*)x)[i];
        const f32x4 b = ((const f32x4*)y)[i];
        a[0] += b[0]; a[1] += b[1]; a[2] += b[2]; a[3] += b[3];
        ((f32x4*)x)[i] = a;
    }
}

// ---------------------------------------------------------------------------------------------
// bf16 MFMA GEMM, 128x128x32 tiles, 4 waves (2x2), each wave 64x64 = 4x4 mfma_f32_16x16x32_bf16.
//   A: activation hi (+lo) [Mpad, K] row-major; W: [N, K] row-major (both K-contiguous, so both
//   MFMA operands are plain 16-byte row segments); f32 accumulate.
//   Double-buffered LDS (row stride 40 elements = 80 B: the 16 rows of a fragment read fall on 16 distinct
//   16-B bank slots) fed from PD = 4 register stages of k-tile loads.
// ---------------------------------------------------------------------------------------------
constexpr int GBM = 128, GBK = 32, GLD = 32;
// register stages of the 256-wide kernel (164 VGPRs at 4 stages leave room at 2 waves per SIMD): 4 -> 33.3 ms, 6 -> 32.5 ms,
// 8 -> 32.8 ms per 1024-token Qwen3-8B prompt
#ifndef PD_WIDE
#define PD_WIDE 6
#endif
// LDS tile rows are 64 B = four 16-byte k-chunks, unpadded; chunk c of row r sits at position c ^ gemm_swz(r).  A wave's
// ds_read_b128 / ds_write_b128 is served in four groups of 16 lanes -- {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same
// + 32 (MI355X_MICROARCH.md, LDS) -- and with this permutation the 16 lanes of every group of a fragment read (lane = 16 fk +
// row) and of a staging write (lane = 4 row + chunk) fall on 16 different 16-byte bank slots.  The 80-byte padded rows
// used before were conflict-free only for 16 CONSECUTIVE lanes: SQ_LDS_BANK_CONFLICT was 50 % of SQ_LDS_IDX_ACTIVE.
__device__ __forceinline__ int gemm_swz(int row) { return (4 - ((row >> 2) & 3)) & 3; }

// BN = 128: 4 waves (2 x 2), two blocks per CU.  BN = 256: 8 waves (2 x 4), one block per CU -- the same 8 waves per CU, but
// the activation tile (hi + lo: twice the bytes of a weight tile) is fetched and written to LDS once for 256 output columns
// instead of once per 128: a third less L2 -> CU traffic per flop (the waves of the 128-wide kernel spend ~39 % of their
// cycles waiting for global loads).
// BM = 64 (BN = 128 only; launch_gemm: M <= 64 -- the rows of a large decode batch, very short prompts): the two wave rows
// take 32 rows each, half the activation tile and half the MFMAs of a tile whose upper 64 rows would be padding.
template <int SPLIT, int EPI, int BN, int BM = 128>
__global__ __launch_bounds__(BN * 2) void gemm_bf16_kernel(GemmArgs a) {
    constexpr int WM = BM / 2, NI = WM / 16;                            // rows per wave row, 16-row MFMA tiles of them
    constexpr int GBN = BN, NT = BN * 2, NWC = BN / 64;                 // threads, wave columns
    constexpr int LA = (BM * 4) / NT, LB = (GBN * 4) / NT;             // 16-byte loads per thread, k-tile and operand
    __shared__ __attribute__((aligned(16))) uint16_t As[2][SPLIT][BM * GLD];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][GBN * GLD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / NWC, wc = wave % NWC;
    const int tiles_m = (a.M + BM - 1) / BM;
    // XCD-aware order: blocks that share a weight tile (same n-tile, different m-tile) get
    // consecutive logical ids AND the same XCD (hardware places block b on XCD b % 8)
    // split-K (a.ksplit > 1; short prompts: one or two m-tiles leave most CUs idle and every block walks all of K as one
    // serial chain of k-tiles): blockIdx = ks * tiles + tile, block ks multiplies k-tiles [ks, ks + 1) * nk / ksplit and
    // stores its raw partial tile (EPI == GEPI_PARTIAL); gemm_splitk_epilogue_kernel adds the partials in a fixed order
    const int nb = tiles_m * (a.N / GBN);
    const int ks = (int)blockIdx.x / nb;
    int bid = (int)blockIdx.x % nb;
    if (nb % 8 == 0) bid = (bid % 8) * (nb / 8) + bid / 8;
    const int tn = bid / tiles_m, tm = bid % tiles_m;
    const int m0 = tm * BM, n0 = tn * GBN;
    const int K = a.K;

    f32x4 acc[NI][4];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // staging map: chunk c = tid + 256*i (i<2): row = c >> 2, 16-byte k-chunk = c & 3.
    // PD register stages: the global loads of k-tile i + PD are requested while tile i is multiplied, so a block's chain
    // is K/32 x (latency / PD) instead of K/32 x latency -- a 128-token prompt has ONE m-tile and 32..192 blocks, nothing
    // else hides the latency (24 ms per 128-token prefill on Qwen3-8B with a single stage).  Loads are unconditional
    // (tile index clamped) and the stages are statically named (loop unrolled by PD).
    constexpr int PD = (BN == 256 && PD_WIDE > 0) ? PD_WIDE : 4;
    const int nk_all = K / GBK, kpb = nk_all / a.ksplit;      // k-tiles per block (launch_gemm: ksplit divides nk_all)
    const int kbeg = ks * kpb, nk = kbeg + kpb;                // this block's k-tiles [kbeg, nk)
    u32x4 ra[PD][SPLIT][LA], rb[PD][LB];
    auto g_load = [&](u32x4 (&qa)[SPLIT][LA], u32x4 (&qb)[LB], int tile) {
        const int k0 = min(tile, nk - 1) * GBK;
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int c = tid + NT * i, row = c >> 2, kc = (c & 3) * 8;
            qa[0][i] = ld16(a.A_hi + (size_t)(m0 + row) * K + k0 + kc);
            if (SPLIT == 2) qa[SPLIT - 1][i] = ld16(a.A_lo + (size_t)(m0 + row) * K + k0 + kc);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int c = tid + NT * i, row = c >> 2, kc = (c & 3) * 8;
            qb[i] = ld16(a.W + (size_t)(n0 + row) * K + k0 + kc);   // cacheable: other m-tiles of this XCD reuse the weight tile from L2
        }
    };
    auto s_store = [&](const u32x4 (&qa)[SPLIT][LA], const u32x4 (&qb)[LB], int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int c = tid + NT * i, row = c >> 2;
            const int so = row * GLD + ((((c & 3) ^ gemm_swz(row))) << 3);
            *(u32x4*)&As[buf][0][so] = qa[0][i];
            if (SPLIT == 2) *(u32x4*)&As[buf][SPLIT - 1][so] = qa[SPLIT - 1][i];
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int c = tid + NT * i, row = c >> 2;
            *(u32x4*)&Bs[buf][row * GLD + ((((c & 3) ^ gemm_swz(row))) << 3)] = qb[i];
        }
    };
    const int fr = lane & 15, fk = (((lane >> 4) ^ gemm_swz(fr)) << 3);      // (tile row offsets are multiples of 16: swz(row) = swz(fr))
    auto compute = [&](int buf) {
        bf16x8 bfrag[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) bfrag[j] = *(const bf16x8*)&Bs[buf][(wc * 64 + j * 16 + fr) * GLD + fk];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const bf16x8 ah = *(const bf16x8*)&As[buf][0][(wr * WM + i * 16 + fr) * GLD + fk];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bfrag[j], acc[i][j], 0, 0, 0);
            if (SPLIT == 2) {
                const bf16x8 al = *(const bf16x8*)&As[buf][SPLIT - 1][(wr * WM + i * 16 + fr) * GLD + fk];
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bfrag[j], acc[i][j], 0, 0, 0);
            }
        }
    };

#pragma unroll
    for (int d = 0; d < PD; ++d) g_load(ra[d], rb[d], kbeg + d);   // tiles 0 .. PD-1 -> stages 0 .. PD-1
    s_store(ra[0], rb[0], 0);
    __syncthreads();
    for (int kt = kbeg; kt < nk; kt += PD) {
#pragma unroll
        for (int d = 0; d < PD; ++d) {
            const int i = kt + d;                                   // tile in LDS buffer d & 1 (kt - kbeg is a multiple of PD)
            if (i >= nk) break;
            g_load(ra[d], rb[d], i + PD);                           // stage d was parked in LDS one step ago: refill it
            compute(d & 1);
            s_store(ra[(d + 1) % PD], rb[(d + 1) % PD], (d + 1) & 1);   // unconditional: past the end a clamped tile nobody reads
            __syncthreads();
        }
    }

    // epilogue: C layout of mfma 16x16: col = lane & 15 (n), row = (lane >> 4) * 4 + reg (m)
    if (EPI == GEPI_PARTIAL) {
        float* P = a.ws + (size_t)ks * a.M * a.N;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + wr * WM + i * 16 + (lane >> 4) * 4 + r;
                    if (m < a.M) P[(size_t)m * a.N + n0 + wc * 64 + j * 16 + (lane & 15)] = acc[i][j][r];
                }
        return;
    }
    float bv[4] = {0.f, 0.f, 0.f, 0.f};                      // a lane's 4 columns: the bias is loaded once, not per element
    if (a.bias != nullptr) {
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[j] = a.bias[n0 + wc * 64 + j * 16 + (lane & 15)];
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        // residual add: the 16 old values of this row band are requested in ONE batch from clamped (always valid)
        // addresses -- a load under the `m < M` guard is followed by vmcnt(0), i.e. 64 serial round trips per lane
        float cold[4][4];
        if (EPI == GEPI_RESADD) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = min(m0 + wr * WM + i * 16 + (lane >> 4) * 4 + r, a.M - 1);
                    cold[j][r] = a.C[(size_t)m * a.ldc + n0 + wc * 64 + j * 16 + (lane & 15)];
                }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + wc * 64 + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wr * WM + i * 16 + (lane >> 4) * 4 + r;
                float v = acc[i][j][r];
                if (a.bias != nullptr) v += bv[j];
                if (EPI == GEPI_STORE) {
                    if (m < a.M) a.C[(size_t)m * a.ldc + n] = v;
                } else if (EPI == GEPI_RESADD) {
                    if (m < a.M) a.C[(size_t)m * a.ldc + n] = cold[j][r] + v;
                } else if (EPI == GEPI_ACT_SPLIT) {   // H[m, n] = act(v) as bf16 hi (+lo): A operand of the next GEMM
                    if (m < a.M) {
                        float h = v;
                        if (a.act == 1) h = 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
                        else if (a.act == 2) h = 0.5f * v * (1.0f + erff(v * 0.7071067811865476f));
                        const size_t off = (size_t)m * a.N + n;
                        const uint16_t hh = f32_to_bf16(h);
                        a.H_hi[off] = hh;
                        if (a.H_lo) a.H_lo[off] = f32_to_bf16(h - bf16_to_f32(hh));
                    }
                } else {   // GEPI_SILUMUL: even column = gate_j, odd column = up_j
                    const float up = dpp_mov<0xB1>(v);          // lane ^ 1
                    if (((lane & 1) == 0) && m < a.M) {
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
}

// ---------------------------------------------------------------------------------------------
// causal flash attention over the paged cache.  grid (Hq, query tiles of 64 rows), 4 waves x 16 query rows.
// ---------------------------------------------------------------------------------------------
// V tile row stride in LDS = D + 16 elements: the 4 key rows of a tr-read group land on disjoint banks
// KVT: KV_BF16 pages (K rows / V^T fragments feed the bf16 MFMAs as cached), KV_F16 pages (the same on the f16 MFMAs; q_hi / q_lo
// and P are then f16 hi + lo), KV_F32 (f32 rows split into bf16 hi + lo on load: f32 pages, the int8 / int4 shadow)
// e^x for x <= 0 (softmax numerators after the running max): v_exp_f32 (2^x, 1 ulp) on x * log2(e) -- two instructions where
// expf()'s range reduction and polynomial are ~20; 17 of them per lane and key tile were a quarter of the tile's VALU work
__device__ __forceinline__ float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

template <int D, int KVT>
__global__ __launch_bounds__(256) void attn_prefill_kernel(AttnPreArgs a_in) {
    AttnPreArgs a = a_in;
    int qt_seg = -1;
    if (a.tiles != nullptr) {         // causal pass over several sequences: this workgroup's (sequence, query tile), longest first
        const int2 tq = a.tiles[gridDim.y - 1 - blockIdx.y];
        const PrefillSegDev sg = a.segs[tq.x];
        const size_t r0 = (size_t)sg.row0 * a.Hq * D;
        a.S = sg.S; a.start_pos = sg.start_pos; a.block_table += sg.bt_off;
        a.q_hi += r0; a.out_hi += r0;
        if (a.q_lo != nullptr) a.q_lo += r0;
        if (a.out_lo != nullptr) a.out_lo += r0;
        if (a.out_f32 != nullptr) a.out_f32 += r0;
        if (a.gate != nullptr) a.gate += (size_t)sg.row0 * a.gate_stride;
        qt_seg = tq.y;
    }
    constexpr bool THREE = KVT == KV_F32;
    constexpr int KT = 64, VLD = D + 16, NKS = D / 32, NNT = D / 16;
    __shared__ __attribute__((aligned(16))) uint16_t Vs[THREE ? 2 : 1][KT * VLD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sub = lane & 15, g = lane >> 4;
    // grid (Hq, query tiles) walked LONGEST TILE FIRST (a query tile of index i attends i + 1 key tiles): at 2048 rows the
    // 1024 workgroups do not fit at once, and in ascending order the last ones dispatched are the longest -- the launch ended
    // with a tail of up to 32 tile times; descending, a slot that finishes a long tile picks up a short one (LPT).
    const int h = blockIdx.x, kvh = h / a.nrep;
    const int qb = (qt_seg >= 0 ? qt_seg : (int)(gridDim.y - 1 - blockIdx.y)) * 64;      // first query row of this block
    const int qrow = qb + wave * 16 + sub;          // this lane's query row (as Q^T column / stats owner)
    const int qrow_c = qrow < a.S ? qrow : a.S - 1; // clamp for loads
    const int qpos = a.start_pos + qrow;

    // Q^T fragments: B operand of S^T = K.Q^T : lane holds Q[q = sub][dims g*8 + 32*ks ..+8]
    bf16x8 qh[NKS], ql[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const size_t off = ((size_t)qrow_c * a.Hq + h) * D + ks * 32 + g * 8;
        qh[ks] = *(const bf16x8*)(a.q_hi + off);
        ql[ks] = *(const bf16x8*)(a.q_lo + off);
    }
    f32x4 o[NNT];
#pragma unroll
    for (int nt = 0; nt < NNT; ++nt) o[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    const int last_q = min(qb + 63, a.S - 1);
    const int kv_end = a.start_pos + last_q + 1;    // tokens [0, start_pos + last_q]
    for (int t0 = 0; t0 < kv_end; t0 += KT) {
        __syncthreads();                                   // previous tile's V fully consumed
        // ---- stage V tile (64 tokens x D dims) into LDS, shared by the 4 waves ----
#pragma unroll
        for (int i = 0; i < (KT * D / 8) / 256; ++i) {
            const int c = tid + 256 * i, tok = c / (D / 8), d8 = (c % (D / 8)) * 8;
            const int t = min(t0 + tok, kv_end - 1);
            const int page = a.block_table[t / a.page];
            const size_t off = ((size_t)(page * a.Hkv + kvh) * a.page + (t % a.page)) * D + d8;
            if (THREE) {
                const f32x4 v0 = *(const f32x4*)((const float*)a.vpool + off);
                const f32x4 v1 = *(const f32x4*)((const float*)a.vpool + off + 4);
                const float vv[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint16_t h0 = f32_to_bf16(vv[2 * e]), h1 = f32_to_bf16(vv[2 * e + 1]);
                    hi[e] = (uint32_t)h0 | ((uint32_t)h1 << 16);
                    lo[e] = pack_bf16x2(vv[2 * e] - bf16_to_f32(h0), vv[2 * e + 1] - bf16_to_f32(h1));
                }
                *(u32x4*)&Vs[0][tok * VLD + d8] = (u32x4){hi[0], hi[1], hi[2], hi[3]};
                *(u32x4*)&Vs[THREE ? 1 : 0][tok * VLD + d8] = (u32x4){lo[0], lo[1], lo[2], lo[3]};
            } else {
                *(u32x4*)&Vs[0][tok * VLD + d8] = ld16((const uint16_t*)a.vpool + off);
            }
        }
        // ---- S^T = K . Q^T for 4 sub-tiles of 16 tokens: rows = tokens, cols = queries ----
        f32x4 s[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            s[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
            const int t = min(t0 + tt * 16 + sub, kv_end - 1);          // this lane's K row (A operand row)
            const int page = a.block_table[t / a.page];
            const size_t kb = ((size_t)(page * a.Hkv + kvh) * a.page + (t % a.page)) * D + g * 8;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                bf16x8 kh, kl;
                if (THREE) {
                    const f32x4 k0 = *(const f32x4*)((const float*)a.kpool + kb + ks * 32);
                    const f32x4 k1 = *(const f32x4*)((const float*)a.kpool + kb + ks * 32 + 4);
                    const float kk[8] = {k0[0], k0[1], k0[2], k0[3], k1[0], k1[1], k1[2], k1[3]};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint16_t hh = f32_to_bf16(kk[e]);
                        kh[e] = (short)hh;
                        kl[e] = (short)f32_to_bf16(kk[e] - bf16_to_f32(hh));
                    }
                } else {
                    kh = *(const bf16x8*)((const uint16_t*)a.kpool + kb + ks * 32);
                }
                s[tt] = mma_k32<KVT>(kh, qh[ks], s[tt]);
                s[tt] = mma_k32<KVT>(kh, ql[ks], s[tt]);
                if (THREE) s[tt] = mma_k32<KVT>(kl, qh[ks], s[tt]);
            }
        }
        // ---- causal mask + online softmax (row statistics live in the lanes with the same `sub`) ----
        float mt = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = t0 + tt * 16 + g * 4 + r;
                if (t > qpos) s[tt][r] = -INFINITY;
                mt = fmaxf(mt, s[tt][r]);
            }
        mt = rows_max(mt);
        const float m_new = fmaxf(m_run, mt);               // finite: token 0 is visible to every query
        const float alpha = fast_exp(m_run - m_new);
        float psum = 0.f;
        bf16x4 ph[4], pl[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = fast_exp(s[tt][r] - m_new);  // exp(-inf) = 0 for masked tokens
                psum += p;
                const uint16_t hh = kv16_from_f32<KVT>(p);
                ph[tt][r] = (short)hh;
                pl[tt][r] = (short)kv16_from_f32<KVT>(p - kv16_to_f32<KVT>(hh));
            }
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int nt = 0; nt < NNT; ++nt) { o[nt][0] *= alpha; o[nt][1] *= alpha; o[nt][2] *= alpha; o[nt][3] *= alpha; }
        __syncthreads();                                   // V tile visible
        // ---- O^T += V^T . P^T : A = V^T fragment (tr-read), B = P^T fragment (registers) ----
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
#pragma unroll
            for (int nt = 0; nt < NNT; ++nt) {
                const uint16_t* vp = &Vs[0][(tt * 16 + g * 4 + (sub >> 2)) * VLD + nt * 16 + (sub & 3) * 4];
                const bf16x4 vh = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
                o[nt] = mma_k16<KVT>(vh, ph[tt], o[nt]);
                o[nt] = mma_k16<KVT>(vh, pl[tt], o[nt]);
                if (THREE) {
                    const uint16_t* vq = &Vs[THREE ? 1 : 0][(tt * 16 + g * 4 + (sub >> 2)) * VLD + nt * 16 + (sub & 3) * 4];
                    const bf16x4 vl = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vq);
                    o[nt] = mma_k16<KVT>(vl, ph[tt], o[nt]);
                }
            }
        }
    }
    // ---- finalize: l over the 4 lane groups; O^T rows = dims nt*16 + g*4 + r, col = query `sub` ----
    l_run = rows_sum(l_run);
    const float inv = 1.0f / l_run;
    if (qrow < a.S) {
#pragma unroll
        for (int nt = 0; nt < NNT; ++nt) {
            float v[4] = {o[nt][0] * inv, o[nt][1] * inv, o[nt][2] * inv, o[nt][3] * inv};
            if (a.gate != nullptr) {        // Qwen3.5: y * sigmoid(gate) (qwen3_5/modeling.rs:556-561)
                const f32x4 gv = *(const f32x4*)(a.gate + (size_t)qrow * a.gate_stride + h * D + nt * 16 + g * 4);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= 1.0f / (1.0f + expf(-gv[r]));
            }
            // (f32 rows: the input of the int8 o_proj GEMM's quantiser -- prompts over Q8_0-layout weights)
            if (a.out_f32 != nullptr) *(f32x4*)(a.out_f32 + ((size_t)qrow * a.Hq + h) * D + nt * 16 + g * 4) = (f32x4){v[0], v[1], v[2], v[3]};
            else
            split_store4(a.out_hi, a.out_lo, ((size_t)qrow * a.Hq + h) * D + nt * 16 + g * 4, v);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Fast path of the causal prompt attention: head_dim 128, 2-byte pages (f16 / bf16), page size a multiple of the
// 64-token key tile, no output gate -- the dense family's prompt pass.  Same tiling, fragments and arithmetic as
// attn_prefill_kernel above (S^T = K Q^T with q as hi + lo, online softmax per query column, O^T += V^T P^T with P as hi + lo);
// what changed is everything AROUND the 96 MFMAs of a key tile, which the ISA of the general kernel shows at ~870 VALU
// instructions per tile and wave (3500 cycles against 1024 of matrix-core issue):
//   * a key tile lies inside ONE page (tile start and page size are multiples of 64): one scalar page-table lookup per tile,
//     K rows and V rows at compile-time offsets from one base -- no per-row division, clamp and 64-bit address chain;
//   * only the tiles that touch the diagonal (or the end of the context) are masked and clamped: two loop bodies;
//   * the softmax runs in the exp2 domain (one FMA + v_exp_f32 per score), P is split with packed conversions;
//   * K AND V go through LDS once per workgroup, double-buffered (comment at kv_fetch): one workgroup barrier per tile;
//   * the products of a tile are all 32 keys deep (126 -> 109 us for 2048 tokens of 32 heads, 78 -> 66 for 452 behind them, when the second product
//     took 16 at a time).
// A launch of few query tiles behind many keys leaves the chip idle and walks the keys one after the other: there several blocks share a query tile's keys and
// attn_prefill_merge_kernel adds the shares (452 queries behind 2048 keys, 32 heads: 66 -> 55 us and 7).
// ---------------------------------------------------------------------------------------------
// workgroup barrier for LDS hand-offs only: waits for this wave's LDS operations, not for its outstanding global loads
// (__syncthreads() drains vmcnt as well and would retire the two-tiles-ahead requests at every tile)
__device__ __forceinline__ void lds_wg_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// (69 KB of LDS per workgroup: two on a CU)
template <int KVT>
__global__ __launch_bounds__(256) void attn_prefill_fast_kernel(AttnPreArgs a_in) {
    constexpr int D = 128, KT = 64, VLD = D + 16, NKS = D / 32, NNT = D / 16, NTT = KT / 16, CPR = D / 8, RPP = 256 / CPR;      // chunks per row, rows per staging pass
    static_assert(KT * CPR == 4 * 256, "four 16-byte chunks per thread and tile");
    constexpr float L2E = 1.4426950408889634f;
    AttnPreArgs a = a_in;
    int qt_seg = -1;
    if (a.tiles != nullptr) {         // causal pass over several sequences: this workgroup's (sequence, query tile), longest first
        const int2 tq = a.tiles[gridDim.y - 1 - blockIdx.y];
        const PrefillSegDev sg = a.segs[tq.x];
        const size_t r0 = (size_t)sg.row0 * a.Hq * D;
        a.S = sg.S; a.start_pos = sg.start_pos; a.block_table += sg.bt_off;
        a.q_hi += r0; a.out_hi += r0;
        if (a.q_lo != nullptr) a.q_lo += r0;
        if (a.out_lo != nullptr) a.out_lo += r0;
        if (a.out_f32 != nullptr) a.out_f32 += r0;
        qt_seg = tq.y;
    }
    __shared__ __attribute__((aligned(16))) uint16_t Vs[2][KT * VLD];
    __shared__ __attribute__((aligned(16))) uint16_t Ks[2][KT * (D + 8)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sub = lane & 15, g = lane >> 4;
    const int h = blockIdx.x, kvh = h / a.nrep;
    // query tile of this workgroup: the first half of the grid takes the LONG tiles in descending order, the second half the SHORT ones
    // in ascending order -- with two workgroups resident per CU (dispatch order, observed: workgroup i and i + 256 share a CU at
    // 1024 tokens x 32 heads) a 16-tile workgroup is then paired with a 1-tile one instead of an 8-tile one and runs most of its
    // life alone on its SIMDs.  Placement only affects speed.
    const int ny = (int)gridDim.y, yy = (int)blockIdx.y, nlong = (ny + 1) / 2;
    const int qb = (qt_seg >= 0 ? qt_seg : (yy < nlong ? ny - 1 - yy : yy - nlong)) * 64;
    const int qrow = qb + wave * 16 + sub;
    const int qrow_c = qrow < a.S ? qrow : a.S - 1;
    const int qpos = a.start_pos + qrow;
    bf16x8 qh[NKS], ql[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const size_t off = ((size_t)qrow_c * a.Hq + h) * D + ks * 32 + g * 8;
        qh[ks] = *(const bf16x8*)(a.q_hi + off);
        ql[ks] = *(const bf16x8*)(a.q_lo + off);
    }
    f32x4 o[NNT];
#pragma unroll
    for (int nt = 0; nt < NNT; ++nt) o[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    const int last_q = min(qb + 63, a.S - 1);
    const int kv_end = a.start_pos + last_q + 1;
    const int ntile = (kv_end + KT - 1) / KT;
    const int nfull = (a.start_pos + qb + 1) / KT;          // tiles every query of the block sees completely (and that end before kv_end)
    const int tps = a.nsplit > 1 ? ((ntile + a.nsplit - 1) / a.nsplit + 1) / 2 * 2 : ntile;        // tiles of a share (even: the buffers alternate)
    const int tbeg = (int)blockIdx.z * tps, tend = min(ntile, tbeg + tps);
    const uint16_t* kpool = (const uint16_t*)a.kpool;
    const uint16_t* vpool = (const uint16_t*)a.vpool;
    // element offset of the first row of key tile t inside the pool (one page per tile).  The page ids of 64 consecutive tiles sit
    // in one VGPR (lane i: tile 64 grp + i) and are picked with v_readlane: a scalar load of the table entry per tile and use
    // was ~1 us of exposed latency twice per tile -- the first version of this kernel ran 82 us against the general kernel's 73
    const int tpp = a.page / KT;                            // key tiles per page
    const int npg = (kv_end + a.page - 1) / a.page;         // pages of the context
    int pgs_grp = 0;
    int pgs = a.block_table[min(lane / tpp, npg - 1)];
    auto tile_base = [&](int t) __attribute__((always_inline)) -> size_t {
        if ((t >> 6) != pgs_grp) {                           // (uniform; every 64 tiles)
            pgs_grp = t >> 6;
            pgs = a.block_table[min((pgs_grp * 64 + lane) / tpp, npg - 1)];
        }
        const int pg = __builtin_amdgcn_readlane(pgs, t & 63);
        return ((size_t)(pg * a.Hkv + kvh) * a.page + ((t * KT) % a.page)) * D;
    };
    // K and V rows of a tile go through LDS ONCE per workgroup: thread c = tid + 256 i covers token c / 16, dims (c % 16) * 8 .. + 8
    // (whole 256-byte rows, coalesced).  The general kernel's waves each fetch the K tile themselves as MFMA A fragments -- 16
    // wave-loads of 16 rows x 64 bytes, the same 16 KB four times per workgroup: ablated (no K loads in the loop) this kernel ran
    // 41 us instead of 73, with the K rows prefetched into registers still 69.  K rows in LDS are 272 bytes apart (the 16 rows of a
    // fragment read start 4 banks apart); both tiles are double-buffered: the next tile's rows are requested before this tile's
    // products and parked after them -- one workgroup barrier per tile.
    constexpr int KLD = D + 8;
    const int vtok = tid / CPR, vd8 = (tid % CPR) * 8;
    struct KvRegs { u32x4 k[4], v[4]; };
    auto kv_fetch = [&](int t, KvRegs& rg) __attribute__((always_inline)) {
        const int tc = min(t, ntile - 1);                   // (past the end: the last tile again, parked into buffers nobody reads)
        const size_t b = tile_base(tc);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tok = min(vtok + RPP * i, kv_end - 1 - tc * KT);
            rg.k[i] = ld16(kpool + b + (size_t)tok * D + vd8);
            rg.v[i] = ld16(vpool + b + (size_t)tok * D + vd8);
        }
    };
    auto kv_park = [&](int buf, const KvRegs& rg) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *(u32x4*)&Ks[buf][(vtok + RPP * i) * KLD + vd8] = rg.k[i];
            *(u32x4*)&Vs[buf][(vtok + RPP * i) * VLD + vd8] = rg.v[i];
        }
    };
    // rows are requested TWO tiles ahead (two alternating register sets: a tile's rows are requested at the top of tile t - 2 and
    // parked at the bottom of tile t - 1): the workgroup barrier at the bottom of a tile drains the wave's loads, so with one tile
    // of distance a tile lasted as long as an L2 / HBM round trip (~2.4 us against ~1 us of work)
    auto tile = [&](int t, auto masked_c, KvRegs& rg_new, const KvRegs& rg_next) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked_c)::value;
        const int t0 = t * KT;
        kv_fetch(t + 2, rg_new);
        // ---- S^T = K . Q^T for 4 sub-tiles of 16 tokens (A fragments: this lane's K row, 16 bytes per k-step, from LDS) ----
        const uint16_t* Kb = Ks[t & 1];
        f32x4 s[NTT];
#pragma unroll
        for (int tt = 0; tt < NTT; ++tt) {
            s[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const bf16x8 kh = *(const bf16x8*)&Kb[(tt * 16 + sub) * KLD + ks * 32 + g * 8];
                s[tt] = mma_k32<KVT>(kh, qh[ks], s[tt]);
                s[tt] = mma_k32<KVT>(kh, ql[ks], s[tt]);
            }
        }
        // ---- (mask +) online softmax in the exp2 domain ----
        float mt = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (MASKED) { if (t0 + tt * 16 + g * 4 + r > qpos) s[tt][r] = -INFINITY; }
                mt = fmaxf(mt, s[tt][r]);
            }
        mt = rows_max(mt);
        const float m_new = fmaxf(m_run, mt);               // finite: token 0 is visible to every query (the first share; in others nothing may be so far)
        const float m_use = MASKED && m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * L2E);
        const float nm = -m_use * L2E;
        float psum = 0.f;
        bf16x4 ph[NTT], pl[NTT];
#pragma unroll
        for (int tt = 0; tt < NTT; ++tt) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) { p[r] = __builtin_amdgcn_exp2f(fmaf(s[tt][r], L2E, nm)); psum += p[r]; }
            p_split4<KVT>(p, ph[tt], pl[tt]);
        }
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int nt = 0; nt < NNT; ++nt) { o[nt][0] *= alpha; o[nt][1] *= alpha; o[nt][2] *= alpha; o[nt][3] *= alpha; }
        // ---- O^T += V^T . P^T : A = V^T fragment (tr-read from this tile's LDS buffer), B = P^T fragment.  The 32 keys of a product are two score tiles side
        // by side (the k index of a product is any order its operands agree on): a 16-deep product takes the matrix unit as long ----
        const uint16_t* Vb = Vs[t & 1];
#pragma unroll
        for (int tt = 0; tt < NTT; tt += 2) {
            const bf16x8 p8h = __builtin_shufflevector(ph[tt], ph[tt + 1], 0, 1, 2, 3, 4, 5, 6, 7);
            const bf16x8 p8l = __builtin_shufflevector(pl[tt], pl[tt + 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int nt = 0; nt < NNT; ++nt) {
                bf16x4 v2[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint16_t* vp = &Vb[((tt + k) * 16 + g * 4 + (sub >> 2)) * VLD + nt * 16 + (sub & 3) * 4];
                    v2[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)vp);
                }
                const bf16x8 vh = __builtin_shufflevector(v2[0], v2[1], 0, 1, 2, 3, 4, 5, 6, 7);
                o[nt] = mma_k32<KVT>(vh, p8h, o[nt]);
                o[nt] = mma_k32<KVT>(vh, p8l, o[nt]);
            }
        }
        kv_park((t + 1) & 1, rg_next);                      // the other buffers: last read one iteration ago, behind that iteration's barrier
        lds_wg_barrier();
    };
    KvRegs rA, rB;
    kv_fetch(tbeg, rA);
    kv_fetch(tbeg + 1, rB);
    kv_park(0, rA);
    __syncthreads();
    // (a tile is "full" when every query of the block sees all of it; the diagonal / ragged tiles are masked)
    for (int t = tbeg; t < tend; t += 2) {
        if (t < nfull) tile(t, std::false_type{}, rA, rB); else tile(t, std::true_type{}, rA, rB);
        if (t + 1 < tend) { if (t + 1 < nfull) tile(t + 1, std::false_type{}, rB, rA); else tile(t + 1, std::true_type{}, rB, rA); }
    }
    // ---- finalize: l over the 4 lane groups; O^T rows = dims nt*16 + g*4 + r, col = query `sub` ----
    l_run = rows_sum(l_run);
    if (a.nsplit > 1) {                                     // attn_prefill_merge_kernel takes it from here
        if (qrow >= a.S) return;
        const size_t at = ((size_t)blockIdx.z * a.S + qrow) * a.Hq + h;
#pragma unroll
        for (int nt = 0; nt < NNT; ++nt) *(f32x4*)(a.ws + at * D + nt * 16 + g * 4) = o[nt];
        float* ml = a.ws + (size_t)a.nsplit * a.S * a.Hq * D + at * 2;
        if (g == 0) { ml[0] = m_run; ml[1] = l_run; }
        return;
    }
    const float inv = 1.0f / l_run;
    if (qrow < a.S) {
#pragma unroll
        for (int nt = 0; nt < NNT; ++nt) {
            const float v[4] = {o[nt][0] * inv, o[nt][1] * inv, o[nt][2] * inv, o[nt][3] * inv};
            // (f32 rows: the input of the int8 o_proj GEMM's quantiser -- prompts over Q8_0-layout weights)
            if (a.out_f32 != nullptr) *(f32x4*)(a.out_f32 + ((size_t)qrow * a.Hq + h) * D + nt * 16 + g * 4) = (f32x4){v[0], v[1], v[2], v[3]};
            else
            split_store4(a.out_hi, a.out_lo, ((size_t)qrow * a.Hq + h) * D + nt * 16 + g * 4, v);
        }
    }
}

// the shares of attn_prefill_fast_kernel's and attn_prompt_wide_kernel's keys merged, four columns per thread
template <int D>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(AttnPreArgs a) {
    constexpr float L2E = 1.4426950408889634f;
    const size_t n = (size_t)a.S * a.Hq, i = (size_t)blockIdx.x * (1024 / D) + threadIdx.x / (D / 4);      // (row, head)
    if (i >= n) return;
    const int c = (int)(threadIdx.x % (D / 4)) * 4, row = (int)(i / a.Hq), h = (int)(i % a.Hq);
    const float* ml = a.ws + (size_t)a.nsplit * n * D;
    float M = -INFINITY, L = 0.f;
#pragma unroll 4
    for (int z = 0; z < a.nsplit; ++z) M = fmaxf(M, ml[((size_t)z * n + i) * 2]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < a.nsplit; ++z) {
        const float2 p = *(const float2*)(ml + ((size_t)z * n + i) * 2);
        const f32x4 v = *(const f32x4*)(a.ws + ((size_t)z * n + i) * D + c);
        const float w = __builtin_amdgcn_exp2f((p.x - M) * L2E);          // (the first share sees token 0: M is finite; a share that saw nothing: 0)
        L = fmaf(p.y, w, L);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = fmaf(v[r], w, o[r]);
    }
    const float inv = 1.0f / L;
    float v[4] = {o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
    if (a.gate != nullptr) {
        const f32x4 gv = *(const f32x4*)(a.gate + (size_t)row * a.gate_stride + h * D + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= 1.0f / (1.0f + expf(-gv[r]));
    }
    if (a.out_f32 != nullptr) *(f32x4*)(a.out_f32 + i * D + c) = (f32x4){v[0], v[1], v[2], v[3]};
    else split_store4(a.out_hi, a.out_lo, i * D + c, v);
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
void launch_embed_rows(const uint16_t* emb, const uint32_t* ids, float* x, int S, int H, int V, hipStream_t s) {
    hipLaunchKernelGGL(embed_rows_kernel, dim3(S), dim3(256), 0, s, emb, ids, x, H, V);
}
void launch_rmsnorm_rows(const float* x, const float* w, uint16_t* hi, uint16_t* lo, int S, int H, float eps,
                         hipStream_t s) {
    hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3(S), dim3(256), 0, s, x, w, hi, lo, H, eps);
}
bool qknorm_rope_adds_slices(const QkRopeArgs& a, int D, int kv_mode) {
    static const int v4 = getenv("CM_ROPE_KV4") ? atoi(getenv("CM_ROPE_KV4")) : 1;          // 0: always the one-wave-per-head kernel (A/B)
    return v4 && D == 128 && a.rot_dim == 128 && a.pos3 == nullptr && (kv_mode == 0 || kv_mode == 1 || kv_mode == KV_F16) &&
           a.q_off % 4 == 0 && a.k_off % 4 == 0 && a.v_off % 4 == 0 && a.row_stride % 4 == 0;
}
void launch_qknorm_rope_kv(const QkRopeArgs& a, int D, int S, int kv_mode, hipStream_t s) {
    if (qknorm_rope_adds_slices(a, D, kv_mode)) {
        dim3 g4(S, (a.Hq + 2 * a.Hkv + 7) / 8);
        if (kv_mode == 1) hipLaunchKernelGGL((qknorm_rope_kv4_kernel<1>), g4, dim3(256), 0, s, a);
        else if (kv_mode == KV_F16) hipLaunchKernelGGL((qknorm_rope_kv4_kernel<KV_F16>), g4, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((qknorm_rope_kv4_kernel<0>), g4, dim3(256), 0, s, a);
        return;
    }
    dim3 grid(S, a.Hq + 2 * a.Hkv);
#define CM_QK(DD) \
    if (kv_mode == 1) hipLaunchKernelGGL((qknorm_rope_kv_kernel<DD, 1>), grid, dim3(64), 0, s, a); \
    else if (kv_mode == 2) hipLaunchKernelGGL((qknorm_rope_kv_kernel<DD, 2>), grid, dim3(64), 0, s, a); \
    else if (kv_mode == 3) hipLaunchKernelGGL((qknorm_rope_kv_kernel<DD, 3>), grid, dim3(64), 0, s, a); \
    else if (kv_mode == KV_F16) hipLaunchKernelGGL((qknorm_rope_kv_kernel<DD, KV_F16>), grid, dim3(64), 0, s, a); \
    else hipLaunchKernelGGL((qknorm_rope_kv_kernel<DD, 0>), grid, dim3(64), 0, s, a);
    if (D == 128) { CM_QK(128) } else { CM_QK(256) }
#undef CM_QK
}
void launch_kvq_dequant_prefix(const void* kpool, const void* vpool, const int32_t* block_table, float* kshadow, float* vshadow,
                               int tokens, int Hkv, int page, int D, int kv_mode, size_t page_bytes, hipStream_t s) {
    if (tokens <= 0) return;
    dim3 grid(tokens, 2 * Hkv);
    const uint8_t *kp = (const uint8_t*)kpool, *vp = (const uint8_t*)vpool;
    if (D == 128) {
        if (kv_mode == 2) hipLaunchKernelGGL((kvq_dequant_prefix_kernel<128, 2>), grid, dim3(64), 0, s, kp, vp, block_table, kshadow, vshadow, Hkv, page, page_bytes);
        else hipLaunchKernelGGL((kvq_dequant_prefix_kernel<128, 3>), grid, dim3(64), 0, s, kp, vp, block_table, kshadow, vshadow, Hkv, page, page_bytes);
    } else {
        if (kv_mode == 2) hipLaunchKernelGGL((kvq_dequant_prefix_kernel<256, 2>), grid, dim3(64), 0, s, kp, vp, block_table, kshadow, vshadow, Hkv, page, page_bytes);
        else hipLaunchKernelGGL((kvq_dequant_prefix_kernel<256, 3>), grid, dim3(64), 0, s, kp, vp, block_table, kshadow, vshadow, Hkv, page, page_bytes);
    }
}
void launch_split_rows(const float* x, uint16_t* hi, uint16_t* lo, size_t n, hipStream_t s) {
    const size_t n4 = n / 4;
    int blocks = (int)std::min<size_t>((n4 + 255) / 256, 4096);
    hipLaunchKernelGGL(split_rows_kernel, dim3(blocks < 1 ? 1 : blocks), dim3(256), 0, s, x, hi, lo, n4);
}
void launch_split_rows2d(const float* x, int ldx, uint16_t* hi, uint16_t* lo, int rows, int cols, hipStream_t s) {
    hipLaunchKernelGGL(split_rows2d_kernel, dim3(rows), dim3(256), 0, s, x, ldx, hi, lo, cols);
}
void launch_add_rows(float* x, const float* y, size_t n, hipStream_t s) {
    const size_t n4 = n / 4;
    int blocks = (int)std::min<size_t>((n4 + 255) / 256, 4096);
    hipLaunchKernelGGL(add_rows_kernel, dim3(blocks < 1 ? 1 : blocks), dim3(256), 0, s, x, y, n4);
}
// second half of a split-K GEMM: thread = 4 consecutive columns of one row; partials added in the order ks = 0, 1, ...
// KS = the split when it is 2, 4 or 8 (the KS slices of an element are then independent requests; as a run-time loop every slice
// is one L2 round trip behind the other), 0: any
template <int EPI, int KS>
__global__ __launch_bounds__(256) void gemm_splitk_epilogue_kernel(GemmArgs a) {
    const size_t n4 = (size_t)a.N / 4, total = (size_t)a.M * n4;
    const size_t slice = (size_t)a.M * a.N;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (size_t)gridDim.x * 256) {
        const int m = (int)(t / n4), n = (int)(t % n4) * 4;
        const float* p0 = a.ws + (size_t)m * a.N + n;
        f32x4 v;
        if (KS > 0) {
            f32x4 p[KS > 0 ? KS : 1];
#pragma unroll
            for (int k = 0; k < KS; ++k) p[k] = *(const f32x4*)(p0 + (size_t)k * slice);
            v = p[0];
#pragma unroll
            for (int k = 1; k < KS; ++k) { v[0] += p[k][0]; v[1] += p[k][1]; v[2] += p[k][2]; v[3] += p[k][3]; }
        } else {
            v = *(const f32x4*)p0;
            for (int k = 1; k < a.ksplit; ++k) {
                const f32x4 p = *(const f32x4*)(p0 + (size_t)k * slice);
                v[0] += p[0]; v[1] += p[1]; v[2] += p[2]; v[3] += p[3];
            }
        }
        if (a.bias != nullptr) {
            const f32x4 b = *(const f32x4*)(a.bias + n);
            v[0] += b[0]; v[1] += b[1]; v[2] += b[2]; v[3] += b[3];
        }
        if (EPI == GEPI_STORE) {
            *(f32x4*)(a.C + (size_t)m * a.ldc + n) = v;
        } else if (EPI == GEPI_RESADD) {
            f32x4 c = *(const f32x4*)(a.C + (size_t)m * a.ldc + n);
            c[0] += v[0]; c[1] += v[1]; c[2] += v[2]; c[3] += v[3];
            *(f32x4*)(a.C + (size_t)m * a.ldc + n) = c;
        } else if (EPI == GEPI_ACT_SPLIT) {
            float h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = v[i];
                h[i] = a.act == 1 ? 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)))
                     : a.act == 2 ? 0.5f * x * (1.0f + erff(x * 0.7071067811865476f)) : x;
            }
            split_store4(a.H_hi, a.H_lo, (size_t)m * a.N + n, h);
        } else {   // GEPI_SILUMUL: columns (gate_j, up_j) interleaved -> two outputs per thread
            const float h0 = (v[0] / (1.0f + expf(-v[0]))) * v[1], h1 = (v[2] / (1.0f + expf(-v[2]))) * v[3];
            const size_t off = (size_t)m * (a.N / 2) + (n >> 1);
            const uint16_t a0 = f32_to_bf16(h0), a1 = f32_to_bf16(h1);
            *(uint32_t*)(a.H_hi + off) = (uint32_t)a0 | ((uint32_t)a1 << 16);
            if (a.H_lo) *(uint32_t*)(a.H_lo + off) = (uint32_t)f32_to_bf16(h0 - bf16_to_f32(a0)) | ((uint32_t)f32_to_bf16(h1 - bf16_to_f32(a1)) << 16);
        }
    }
}

// gemm_splitk_epilogue_kernel<GEPI_RESADD> + rmsnorm_rows_kernel in one launch (GemmArgs::norm_w): one block per row, the thread ->
// column map and the order of every sum are those of the two kernels it replaces, so the row of C and the planes are bit-equal.
// KS = the split (2, 4, 8; 0: any, a run-time loop): the KS partial loads of a chunk are independent requests -- as a run-time loop
// the first version paid one L2 round trip per slice (12 us per launch, as much as the two launches it replaced).
template <int KS, bool LN, int NT = 256>
__global__ __launch_bounds__(NT) void gemm_splitk_resadd_norm_kernel(GemmArgs a) {
    static_assert(!LN || NT == 256, "");
    __shared__ float red[NT / 64 > 8 ? NT / 64 : 8];
    const int m = blockIdx.x, tid = threadIdx.x;
    float* __restrict__ cr = a.C + (size_t)m * a.ldc;            // (the partial slices and the row of C never overlap: the loads of the next
    const float* __restrict__ wsr = a.ws + (size_t)m * a.N;      //  chunks may pass this chunk's store)
    const size_t slice = (size_t)a.M * a.N;
    constexpr int NC = 1024 / NT, ST = 4 * NT;
    float ss = 0.f, ls = 0.f;
    // NT = 1024: decode groups and short prompts, a row of up to 4096 columns is one chunk per thread and stays in registers up to the norm
    const bool held = NT == 1024 && a.N <= 4 * NT;
    f32x4 mine = {0.f, 0.f, 0.f, 0.f}, mw = mine;
    if (held && tid * 4 < a.N) mw = *(const f32x4*)(a.norm_w + tid * 4);
    // All partial / residual loads of NC chunks of the row go out before the first of them is consumed (one block per row: at 64 rows a
    // quarter of the chip runs this kernel, so it is the round trips per thread that take the time, not the bytes); the sums keep their order
    for (int n0 = tid * 4; n0 < a.N; n0 += ST * NC) {
        f32x4 p[NC][KS > 0 ? KS : 1], c[NC], bv[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int n = n0 + ST * i < a.N ? n0 + ST * i : n0;      // (a chunk past the row re-reads the first one: unconditional loads)
            const float* __restrict__ p0 = wsr + n;
            if (KS > 0) {
#pragma unroll
                for (int k = 0; k < KS; ++k) p[i][k] = *(const f32x4*)(p0 + (size_t)k * slice);
            } else {
                p[i][0] = *(const f32x4*)p0;
            }
            c[i] = *(const f32x4*)(cr + n);
            bv[i] = a.bias != nullptr ? *(const f32x4*)(a.bias + n) : (f32x4){0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int n = n0 + ST * i;
            if (n >= a.N) break;
            f32x4 v = p[i][0];
            if (KS > 0) {
#pragma unroll
                for (int k = 1; k < KS; ++k) { v[0] += p[i][k][0]; v[1] += p[i][k][1]; v[2] += p[i][k][2]; v[3] += p[i][k][3]; }
            } else {
                for (int k = 1; k < a.ksplit; ++k) {
                    const f32x4 q = *(const f32x4*)(wsr + n + (size_t)k * slice);
                    v[0] += q[0]; v[1] += q[1]; v[2] += q[2]; v[3] += q[3];
                }
            }
            if (a.bias != nullptr) { v[0] += bv[i][0]; v[1] += bv[i][1]; v[2] += bv[i][2]; v[3] += bv[i][3]; }
            f32x4 cc = c[i];
            cc[0] += v[0]; cc[1] += v[1]; cc[2] += v[2]; cc[3] += v[3];
            *(f32x4*)(cr + n) = cc;
            if (held) mine = cc;
            if (LN) ls += cc[0] + cc[1] + cc[2] + cc[3];
            else ss += cc[0] * cc[0] + cc[1] * cc[1] + cc[2] * cc[2] + cc[3] * cc[3];
        }
    }
    if (LN) {                                                    // LayerNorm with bias: layernorm_rows_kernel's three passes
        ls = wave_sum(ls);
        if ((tid & 63) == 0) red[tid >> 6] = ls;
        __syncthreads();
        const float mu = ((red[0] + red[1]) + (red[2] + red[3])) / (float)a.N;
        float q = 0.f;
        for (int n = tid * 4; n < a.N; n += 1024) {
            const f32x4 c = *(const f32x4*)(cr + n);              // (this thread's own stores)
            q += (c[0] - mu) * (c[0] - mu) + (c[1] - mu) * (c[1] - mu) + (c[2] - mu) * (c[2] - mu) + (c[3] - mu) * (c[3] - mu);
        }
        q = wave_sum(q);
        if ((tid & 63) == 0) red[4 + (tid >> 6)] = q;
        __syncthreads();
        const float r = 1.0f / sqrtf(((red[4] + red[5]) + (red[6] + red[7])) / (float)a.N + a.norm_eps);
        for (int n = tid * 4; n < a.N; n += 1024) {
            const f32x4 c = *(const f32x4*)(cr + n);
            const f32x4 ww = *(const f32x4*)(a.norm_w + n), bb = *(const f32x4*)(a.norm_b + n);
            const float o[4] = {(c[0] - mu) * r * ww[0] + bb[0], (c[1] - mu) * r * ww[1] + bb[1],
                                (c[2] - mu) * r * ww[2] + bb[2], (c[3] - mu) * r * ww[3] + bb[3]};
            split_store4(a.norm_hi, a.norm_lo, (size_t)m * a.N + n, o);
        }
        return;
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    float all = (red[0] + red[1]) + (red[2] + red[3]);
#pragma unroll
    for (int w = 4; w < NT / 64; w += 4) all += (red[w] + red[w + 1]) + (red[w + 2] + red[w + 3]);
    const float r = 1.0f / sqrtf(all / (float)a.N + a.norm_eps);
    if (held) {
        const float o[4] = {mine[0] * r * mw[0], mine[1] * r * mw[1], mine[2] * r * mw[2], mine[3] * r * mw[3]};
        if (tid * 4 < a.N) split_store4(a.norm_hi, a.norm_lo, (size_t)m * a.N + tid * 4, o);
        return;
    }
#pragma unroll 2
    for (int n = tid * 4; n < a.N; n += ST) {
        const f32x4 c = *(const f32x4*)(cr + n);                  // (this thread's own stores)
        const f32x4 ww = *(const f32x4*)(a.norm_w + n);
        const float o[4] = {c[0] * r * ww[0], c[1] * r * ww[1], c[2] * r * ww[2], c[3] * r * ww[3]};
        split_store4(a.norm_hi, a.norm_lo, (size_t)m * a.N + n, o);
    }
}
static void launch_splitk_resadd_norm(const GemmArgs& a, hipStream_t s) {
#define CM_RN(LN) do { \
    if (a.ksplit == 2) hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<2, LN>), dim3(a.M), dim3(256), 0, s, a); \
    else if (a.ksplit == 4) hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<4, LN>), dim3(a.M), dim3(256), 0, s, a); \
    else if (a.ksplit == 8) hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<8, LN>), dim3(a.M), dim3(256), 0, s, a); \
    else hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<0, LN>), dim3(a.M), dim3(256), 0, s, a); } while (0)
    // up to 128 rows of more than 1024 columns: four times the threads per row (one workgroup per row leaves half of the chip idle either way).
    // Rows of 4096, eight slices: 32 rows 5.8 -> 4.9, 117 rows 6.9 -> 5.9 us.  Product and reduction together, 256 / 1024 threads, 9 and 128 rows:
    // 1152 columns, two slices 7.7 / 7.3 and 13.4 / 13.0; 1536, eight 8.7 / 8.0 and 15.5 / 14.6; 2048, eight 7.4 / 6.7 and 14.1 / 13.4; 5120, four
    // 15.9 / 14.6 and 27.4 / 26.2
    if (a.norm_b == nullptr && a.M <= 128 && a.N > 1024 && (a.ksplit == 2 || a.ksplit == 4 || a.ksplit == 8)) {
        if (a.ksplit == 2) hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<2, false, 1024>), dim3(a.M), dim3(1024), 0, s, a);
        else if (a.ksplit == 4) hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<4, false, 1024>), dim3(a.M), dim3(1024), 0, s, a);
        else hipLaunchKernelGGL((gemm_splitk_resadd_norm_kernel<8, false, 1024>), dim3(a.M), dim3(1024), 0, s, a);
        return;
    }
    if (a.norm_b != nullptr) CM_RN(true); else CM_RN(false);
#undef CM_RN
}

// split factor for a GEMM of `tiles` output tiles and nk k-tiles: only when the tiles alone leave the chip mostly idle
static int gemm_ksplit(int M, int N, int tiles, int nk, size_t ws_floats, int cap_arg) {
    static const int cap_env = getenv("CM_KSPLIT_CAP") ? atoi(getenv("CM_KSPLIT_CAP")) : 0;   // (0 = unset)      // blocks (tuning)
    const int ksplit_cap = cap_env > 0 ? cap_env : (cap_arg > 0 ? cap_arg : 768);
    if (ws_floats == 0) return 1;      // (any M: a GEMM of <= 256 tiles leaves half of the 2-blocks-per-CU slots empty)
    int S = 1;
    while (S < 8 && tiles * (S * 2) <= ksplit_cap && nk % (S * 2 * 4) == 0 && nk / (S * 2) >= 8 && (size_t)(S * 2) * M * N <= ws_floats) S *= 2;
    return S;
}

template <int EPI>
static void launch_splitk_epilogue(const GemmArgs& a, int eb, hipStream_t s) {
    if (a.ksplit == 2) hipLaunchKernelGGL((gemm_splitk_epilogue_kernel<EPI, 2>), dim3(eb), dim3(256), 0, s, a);
    else if (a.ksplit == 4) hipLaunchKernelGGL((gemm_splitk_epilogue_kernel<EPI, 4>), dim3(eb), dim3(256), 0, s, a);
    else if (a.ksplit == 8) hipLaunchKernelGGL((gemm_splitk_epilogue_kernel<EPI, 8>), dim3(eb), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((gemm_splitk_epilogue_kernel<EPI, 0>), dim3(eb), dim3(256), 0, s, a);
}

// GemmArgs::norm_w can ride on the split-K reduction launch (CM_GEMM_NORM_FUSED = 0: always the separate rmsnorm_rows launch, A/B)
static bool norm_fused(const GemmArgs& a) {
    static const int env = getenv("CM_GEMM_NORM_FUSED") ? atoi(getenv("CM_GEMM_NORM_FUSED")) : 1;
    return env != 0 && a.norm_w != nullptr && a.ldc == a.N && a.N % 4 == 0;
}

// the reduction behind a launch that left partial tiles of a.ksplit K slices
static void launch_splitk(GemmArgs& a, int epi, hipStream_t s) {
    const int eb = (int)std::min<size_t>(((size_t)a.M * (a.N / 4) + 255) / 256, 2048);
    if (epi == GEPI_STORE) launch_splitk_epilogue<GEPI_STORE>(a, eb, s);
    else if (epi == GEPI_RESADD && norm_fused(a)) { launch_splitk_resadd_norm(a, s); a.norm_w = nullptr; }
    else if (epi == GEPI_RESADD) launch_splitk_epilogue<GEPI_RESADD>(a, eb, s);
    else if (epi == GEPI_ACT_SPLIT) launch_splitk_epilogue<GEPI_ACT_SPLIT>(a, eb, s);
    else launch_splitk_epilogue<GEPI_SILUMUL>(a, eb, s);
}

// ... or left to a consumer that adds the slices itself
static void leave_slices(GemmArgs& a, int epi, hipStream_t s) {
    if (a.defer_ks != nullptr && epi == GEPI_STORE && a.bias == nullptr) *a.defer_ks = a.ksplit;
    else launch_splitk(a, epi, s);
}

// The LDS-DMA kernel on full cache lines (kernels_gemm256.hip; one tile of up to 128 rows with hi + lo activations, 256-row tiles with plain bf16 from 512 rows on)
// where one of its tile widths fills the chip in whole rounds -- (width, k-slices) by a small cost model: rounds of 256 CUs x one block's MFMA time + the f32 partial-tile traffic of a split.  Returns false when the
// register-staged kernel should run.
// the column tile and the K slices of such a product; false: not for that kernel.  (The environment's BN, KS and MIN_BLOCKS steer these launches alone, not those of kernels_gemm_tile.hip.)
static bool gemm256_plan(int M, int N, int K, bool lo, size_t ws_floats, bool w4, int* bn_out, int* ks_out) {
    static const int force_bn = getenv("CM_GEMM256_BN") ? atoi(getenv("CM_GEMM256_BN")) : 0;     // tuning
    static const int force_ks = getenv("CM_GEMM256_KS") ? atoi(getenv("CM_GEMM256_KS")) : 0;
    static const int min_blocks = getenv("CM_GEMM256_MIN_BLOCKS") ? atoi(getenv("CM_GEMM256_MIN_BLOCKS")) : 128;
    const int bm = w4 ? gemmw4_rows(lo) : gemm256_rows(lo, M);
    const int tiles_m = (M + bm - 1) / bm, nk = K / 64;
    const double terms = lo ? 2.0 : 1.0;
    double best = 1e30;
    int best_bn = 0, best_ks = 1;
    for (int bn : {256, 192}) {
        if (N % bn != 0 || (force_bn && bn != force_bn)) continue;
        const int tiles = tiles_m * (N / bn);
        for (int ks = 1; ks <= 8; ks *= 2) {
            if (force_ks && ks != force_ks) continue;
            if (nk % ks != 0 || nk / ks < 8) break;
            if (ks > 1 && (size_t)ks * M * N > ws_floats) break;
            const int blocks = tiles * ks, rounds = (blocks + 255) / 256;
            const double t_blk = (double)bm * bn * (double)(K / ks) * 2.0 * terms / 6.0e12;                   // ~60 % of a CU's MFMA peak
            const double t_split = ks > 1 ? ((double)(2 * ks + 1) * M * N * 4.0) / 3.0e12 + 6e-6 : 0.0;   // partial tiles out and back + a launch
            const double t = rounds * t_blk + t_split;
            if (t < best) { best = t; best_bn = bn; best_ks = ks; }
        }
    }
    if (best_bn == 0) return false;
    // the chip must be reasonably full: otherwise the 128-row kernel's own split-K heuristics do better
    const int blocks = tiles_m * (N / best_bn) * best_ks;
    // (64-row tiles, measured at 48 / 64 rows: gate||up 60 -> 51 us, QKV 25 -> 22, but o_proj 16.3 -> 17.7 and down_proj equal -- the
    // projections of fewer than 24 column tiles stay on the 128-wide kernel)
    if (bm == 64 && tiles_m * (N / best_bn) < 24 && !force_bn) return false;
    if (blocks < (M >= 512 ? 192 : min_blocks) && !force_bn) return false;
    *bn_out = best_bn; *ks_out = best_ks;
    return true;
}
static bool try_gemm256(GemmArgs& a, int epi, hipStream_t s) {
    static const int env = getenv("CM_GEMM256") ? atoi(getenv("CM_GEMM256")) : 1;
    // hi + lo: 128-row tiles, 64-row tiles up to 64 rows.  From 9 rows on (not 33): a decode round of 16 / 32 sequences 5.87 / 6.25 ->
    // 5.41 / 5.82 ms against the 128-wide kernel + split-K (profiles/r06_small_group_gemm_ab.log); a 32-row tile variant measured no faster
    // than the 64-row one (the launch is not bound by its MFMAs), 8 rows run on the batched GEMVs
    static const int min_m2 = getenv("CM_GEMM256_MIN_M") ? atoi(getenv("CM_GEMM256_MIN_M")) : 9;
    if (!env || !a.wide256 || a.wide256 == 4 || a.M < (a.A_lo ? min_m2 : 512) || a.K % 64 != 0) return false;
    // the one-wave-per-SIMD kernel (kernels_gemmw4.hip) -- built, bit-compatible, measured 0 .. 4 % SLOWER than the ping-pong kernel
    // on every prompt shape, so it is opt-in: CM_GEMMW4 = 1 from `w4_min` rows on, GemmArgs::wide256 = 2 (cm_debug_set "gemm256" = 2) always
    static const int w4_env = getenv("CM_GEMMW4") ? atoi(getenv("CM_GEMMW4")) : 0;
    static const int w4_min = getenv("CM_GEMMW4_MIN_M") ? atoi(getenv("CM_GEMMW4_MIN_M")) : 65;
    const bool w4 = a.wide256 == 2 || (a.wide256 == 1 && w4_env != 0 && a.M >= w4_min);
    int bm = 0, bn = 0, ks = 1;
    if (!w4 && a.A_lo != nullptr && a.M > 128) {                 // hi + lo prompts: kernels_gemm_tile.hip
        if (!gemm_tile_plan(a.M, a.N, a.K, a.ws ? a.ws_floats : 0, a.norm_w != nullptr, &bm, &bn, &ks, nullptr)) return false;
        a.ksplit = ks;
        if (!launch_gemm_tile(a, epi, bm, bn, s)) return false;
        if (ks > 1) leave_slices(a, epi, s);
        return true;
    }
    if (!gemm256_plan(a.M, a.N, a.K, a.A_lo != nullptr, a.ws ? a.ws_floats : 0, w4, &bn, &ks)) return false;
    a.ksplit = ks;
    if (w4) { if (!launch_gemmw4(a, epi, bn, s)) return false; }
    else if (!launch_gemm256(a, epi, bn, s)) return false;
    if (ks > 1) launch_splitk(a, epi, s);
    return true;
}

// rows of interleaved (gate_j, up_j) f32 columns -> silu(gate) * up as bf16 hi (+ lo) planes [M][N / 2] (the GEMM's GEPI_SILUMUL epilogue
// as a launch of its own: the two-pass GEMM over a hi + lo weight operand)
__global__ void silu_mul_split_kernel(const float* __restrict__ gu, uint16_t* __restrict__ hi, uint16_t* __restrict__ lo, size_t n4, int half4) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;          // 4 outputs = 8 interleaved inputs
    if (i >= n4) return;
    const size_t m = i / (size_t)half4, c = i % (size_t)half4;
    const float* p = gu + (m * (size_t)half4 + c) * 8;
    const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
    const float o[4] = {(a[0] / (1.0f + expf(-a[0]))) * a[1], (a[2] / (1.0f + expf(-a[2]))) * a[3],
                        (b[0] / (1.0f + expf(-b[0]))) * b[1], (b[2] / (1.0f + expf(-b[2]))) * b[3]};
    split_store4(hi, lo, i * 4, o);
}

static bool launch_gemm_inner(GemmArgs& a, int epi, hipStream_t s);
static bool launch_gemm_once(GemmArgs& a, int epi, hipStream_t s);
// the planes of a.norm_w's norm of C, where no reduction wrote them
static void launch_gemm_norm(const GemmArgs& a, hipStream_t s) {
    if (a.norm_b != nullptr) launch_layernorm_rows(a.C, a.norm_w, a.norm_b, a.norm_hi, a.norm_lo, a.M, a.N, a.norm_eps, s);
    else launch_rmsnorm_rows(a.C, a.norm_w, a.norm_hi, a.norm_lo, a.M, a.N, a.norm_eps, s);
}
bool launch_gemm(const GemmArgs& a0, int epi, hipStream_t s) {
    if (a0.N % 128 != 0 || a0.K % GBK != 0) return false;
    GemmArgs a = a0;
    if (a.norm_w != nullptr && (epi != GEPI_RESADD || a.ldc != a.N)) return false;
    if (a.W_lo != nullptr) {
        // hi + lo weight operand (a dequantised ggml matrix): C = A . W^T, then C += A_hi . W_lo^T (the A_lo . W_lo term is 2^-26);
        // the epilogue that is not linear in C (SiLU(gate) * up) runs on the f32 sums afterwards
        if (epi != GEPI_STORE && epi != GEPI_RESADD && epi != GEPI_SILUMUL) return false;
        if (epi == GEPI_SILUMUL && a.gu_tmp == nullptr) return false;
        GemmArgs p1 = a, p2 = a;
        p1.W_lo = nullptr; p1.norm_w = nullptr; p1.defer_ks = p2.defer_ks = nullptr;
        p2.W = a.W_lo; p2.W_lo = nullptr; p2.A_lo = nullptr; p2.norm_w = nullptr;
        if (epi == GEPI_SILUMUL) { p1.C = a.gu_tmp; p1.ldc = a.N; p2.C = a.gu_tmp; p2.ldc = a.N; }
        if (!launch_gemm_inner(p1, epi == GEPI_RESADD ? GEPI_RESADD : GEPI_STORE, s)) return false;
        if (!launch_gemm_inner(p2, GEPI_RESADD, s)) return false;
        if (epi == GEPI_SILUMUL) {
            const size_t n4 = (size_t)a.M * (a.N / 8);
            hipLaunchKernelGGL(silu_mul_split_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, a.gu_tmp, a.H_hi, a.H_lo, n4, a.N / 8);
        }
    } else
    if (!launch_gemm_inner(a, epi, s)) return false;
    // the planes of RMSNorm(C) were not written by the split-K reduction (no split, or switched off): the row kernel
    if (a.norm_w != nullptr) launch_gemm_norm(a, s);
    return true;
}

// 9 .. 128 rows: the tiles of kernels_gemm_rows.hip where its rule takes the sizes
static bool try_gemm_rows(GemmArgs& a, int epi, hipStream_t s) {
    static const int env = getenv("CM_GEMM256") ? atoi(getenv("CM_GEMM256")) : 1;
    if (!env || (a.wide256 != 1 && a.wide256 != 4) || a.A_lo == nullptr || epi == GEPI_ACT_SPLIT) return false;
    int bn = 0, ks = 0;
    if (!gemm_rows_plan(a.M, a.N, a.K, a.ws ? a.ws_floats : 0, &bn, &ks)) return false;
    a.ksplit = ks;
    if (!launch_gemm_rows(a, epi, bn, s)) return false;
    if (ks > 1) leave_slices(a, epi, s);
    return true;
}
static bool gemm_tail_columns(int M, int N) { return M >= 256 && N >= 512 && N % 192 != 0 && N % 256 == 128; }
// Prompt rows over a width that no tile of the LDS-DMA kernels divides because of its last 128 columns (the merged in_proj of a Gated-Delta-Net layer:
// 8192 columns and 32 gate columns padded to 128): the wide part there, the last columns alone.  8320 x 2048, 2048 rows: 180 -> 137 us (a prompt of
// 2048 / 1024 / 300 tokens 18.6 / 10.8 / 5.54 -> 17.8 / 10.2 / 5.49 ms; width 1024: 12.3 / 7.3 / 4.5 -> 12.0 / 7.2 / 4.5)
static bool try_gemm_tail(GemmArgs& a, int epi, hipStream_t s) {
    if (epi != GEPI_STORE || a.norm_w != nullptr || !gemm_tail_columns(a.M, a.N)) return false;
    GemmArgs most = a, rest = a;
    most.defer_ks = rest.defer_ks = nullptr;
    most.N = a.N - 128;
    if (!try_gemm256(most, epi, s)) return false;
    rest.W = a.W + (size_t)most.N * a.K; rest.C = a.C + most.N; rest.N = 128;
    if (a.bias != nullptr) rest.bias = a.bias + most.N;
    return launch_gemm_once(rest, epi, s);
}
// What M rows of a product with hi + lo activations take on the kernel that launch_gemm_once finds for them, in seconds: the tiles of kernels_gemm_tile.hip by their own figures; two blocks of
// 128 x 128 on a CU 1.6 us per 64-deep k-tile and 10 around them; one row tile of gemm256_kernel 1.44 us at 256 columns and 13; products of at most 128 rows by their weights, which the rows in
// front of them have just read (118 launches of 9 .. 128 rows over the widths of the 8B and 2B models: 5 % off in the mean square)
static double gemm_seconds(int M, int N, int K, int epi, size_t ws_floats, int ksplit_cap) {
    int bm = 0, bn = 0, ks = 0;
    const auto split = [&](int cols) { return ks > 1 ? (double)(2 * ks + 1) * M * cols * 4.0 / 5e12 + 4e-6 : 0.0; };
    if (epi != GEPI_ACT_SPLIT && gemm_rows_plan(M, N, K, ws_floats, &bn, &ks)) return 4.3e-6 + M * 62e-9 + (double)N * K * 2.0 / (M <= 64 ? 5.9e12 : 4.2e12);
    const int tiles_m = (M + 127) / 128;
    const bool tail = epi == GEPI_STORE && gemm_tail_columns(M, N);
    const int cols = N - (tail ? 128 : 0);
    double best = 0.0;
    if (gemm_tile_plan(M, cols, K, ws_floats, epi == GEPI_RESADD, &bm, &bn, &ks, &best)) return best + (tail ? 15e-6 : 0.0);
    if (M <= 128 && gemm256_plan(M, cols, K, true, ws_floats, false, &bn, &ks))
        return (tiles_m * (cols / bn) * ks + 255) / 256 * (K / 64 / ks * 1.44e-6 * bn / 256 + 13e-6) + split(cols);
    ks = gemm_ksplit(M, N, tiles_m * (N / 128), K / GBK, ws_floats, ksplit_cap);
    return (tiles_m * (N / 128) * ks + 511) / 512 * (K / 64 / ks * 1.6e-6 + 10e-6) + split(N);
}
// the rows of the first of two bands that take less time than all rows at once; 0: all at once
int gemm_band(int M, int N, int K, int epi, size_t ws_floats, int ksplit_cap) {
    if (M <= 256 || N % 128 != 0 || K % 64 != 0 || epi == GEPI_ACT_SPLIT) return 0;
    const double whole = gemm_seconds(M, N, K, epi, ws_floats, ksplit_cap);
    double least = std::min(0.95 * whole, whole - 8e-6);
    int rows = 0;
    for (int m = (M - 9) / 128 * 128; m >= 128 && M - m <= 1024; m -= 128) {
        const double t = gemm_seconds(m, N, K, epi, ws_floats, ksplit_cap) + gemm_seconds(M - m, N, K, epi, ws_floats, ksplit_cap) + 2e-6;
        if (t < least) { least = t; rows = m; }
    }
    return rows;
}
// A round of blocks that the last tiles fill to a part takes as long as a full one: a band of rows whose tiles fill their rounds first, the rows behind it on
// the kernel that suits so few.  What bounds either band is what bounded the whole; the second reads the weights again.  One launch / two, us of prompts through eight layers: width 4096, 645 tokens
// 4525 / 4388 (gate and up 512 + 133), 768 4726 / 4521, 1040 6877 / 5918 (1024 + 16 in three products), 1152 7053 / 6478, 1400 7814 / 7608 (down 384 + 1016); width 2048 with Gated-Delta-Net layers,
// 1290 3546 / 3378, 2060 5427 / 4848, 2304 5718 / 5475, 4165 9739 / 8647.  The line is a gain of 5 % and 8 us by the figures above, which are 5 % off: with 5 % alone the products of width
// 1024 lost, a launch and a reduction more for a round of 30 us.  Width 5120, whose sizes the tiles' prices were not fitted to: 19 of 21 lengths gain up to 10 %, 960 and 2000 tokens lose 1.6 %.
// Rows of products with an activation behind them and the
// vision tower's norm stay in one launch (not measured).
static bool try_gemm_bands(GemmArgs& a, int epi, hipStream_t s) {
    if (a.A_lo == nullptr || a.wide256 != 1 || a.norm_b != nullptr) return false;
    const int m = gemm_band(a.M, a.N, a.K, epi, a.ws ? a.ws_floats : 0, a.ksplit_cap);
    if (m == 0) return false;
    const size_t hcols = epi == GEPI_SILUMUL ? (size_t)a.N / 2 : (size_t)a.N;
    for (int part = 0; part < 2; ++part) {
        const size_t r0 = part ? (size_t)m : 0;
        GemmArgs b = a;
        b.defer_ks = nullptr;                                      // (slices of either band's rows)
        b.M = part ? a.M - m : m;
        b.A_hi += r0 * a.K; b.A_lo += r0 * a.K;
        if (a.C) b.C += r0 * a.ldc;
        if (a.H_hi) b.H_hi += r0 * hcols;
        if (a.H_lo) b.H_lo += r0 * hcols;
        if (a.norm_hi) b.norm_hi += r0 * a.N;
        if (a.norm_lo) b.norm_lo += r0 * a.N;
        if (!launch_gemm_once(b, epi, s)) return false;
        if (b.norm_w != nullptr) launch_gemm_norm(b, s);
    }
    a.norm_w = nullptr;
    return true;
}
static bool launch_gemm_inner(GemmArgs& a, int epi, hipStream_t s) { return try_gemm_bands(a, epi, s) || launch_gemm_once(a, epi, s); }
static bool launch_gemm_once(GemmArgs& a, int epi, hipStream_t s) {
    if (try_gemm_tail(a, epi, s) || try_gemm_rows(a, epi, s) || try_gemm256(a, epi, s)) return true;
    const int tiles_m = (a.M + GBM - 1) / GBM;
    const bool split = a.A_lo != nullptr;
    // 256-wide tiles (one 8-wave block per CU) when they give every CU at least two blocks (1024-token gate||up: 428 -> ~370 us;
    // fewer, and the tail of the last round costs more than the tile saves); CM_GEMM_BN = 128 | 256 forces a width (A/B)
    static const int bn_env = getenv("CM_GEMM_BN") ? atoi(getenv("CM_GEMM_BN")) : 0;
    const int t256 = tiles_m * (a.N / 256);
    static const int wide_lo = getenv("CM_GEMM_WIDE_LO") ? atoi(getenv("CM_GEMM_WIDE_LO")) : 192;      // (tuning)
    const bool wide = a.N % 256 == 0 && (bn_env == 256 || (bn_env == 0 && (t256 >= 512 || (t256 >= wide_lo && t256 <= 256))));
    if (wide) {
        const int tiles = tiles_m * (a.N / 256);
#define CM_GEMM(SP, EP) hipLaunchKernelGGL((gemm_bf16_kernel<SP, EP, 256>), dim3(tiles), dim3(512), 0, s, a)
        a.ksplit = 1;
        if (split) {
            if (epi == GEPI_STORE) CM_GEMM(2, GEPI_STORE); else if (epi == GEPI_RESADD) CM_GEMM(2, GEPI_RESADD);
            else if (epi == GEPI_ACT_SPLIT) CM_GEMM(2, GEPI_ACT_SPLIT); else CM_GEMM(2, GEPI_SILUMUL);
        } else {
            if (epi == GEPI_STORE) CM_GEMM(1, GEPI_STORE); else if (epi == GEPI_RESADD) CM_GEMM(1, GEPI_RESADD);
            else if (epi == GEPI_ACT_SPLIT) CM_GEMM(1, GEPI_ACT_SPLIT); else CM_GEMM(1, GEPI_SILUMUL);
        }
#undef CM_GEMM
        return true;
    }
    const int tiles = tiles_m * (a.N / 128);
    a.ksplit = a.ws != nullptr ? gemm_ksplit(a.M, a.N, tiles, a.K / GBK, a.ws_floats, a.ksplit_cap) : 1;
    if (a.ksplit > 1) {
        static const int bm_env = getenv("CM_GEMM_BM") ? atoi(getenv("CM_GEMM_BM")) : 0;       // 128: never the 64-row tile (A/B)
        if (a.M <= 64 && bm_env != 128) {        // one m-tile of <= 64 rows: the 64 x 128 tile (same block count, same partial layout)
            if (split) hipLaunchKernelGGL((gemm_bf16_kernel<2, GEPI_PARTIAL, 128, 64>), dim3(tiles * a.ksplit), dim3(256), 0, s, a);
            else hipLaunchKernelGGL((gemm_bf16_kernel<1, GEPI_PARTIAL, 128, 64>), dim3(tiles * a.ksplit), dim3(256), 0, s, a);
        } else
        if (split) hipLaunchKernelGGL((gemm_bf16_kernel<2, GEPI_PARTIAL, 128>), dim3(tiles * a.ksplit), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((gemm_bf16_kernel<1, GEPI_PARTIAL, 128>), dim3(tiles * a.ksplit), dim3(256), 0, s, a);
        launch_splitk(a, epi, s);
        return true;
    }
#define CM_GEMM(SP, EP) hipLaunchKernelGGL((gemm_bf16_kernel<SP, EP, 128>), dim3(tiles), dim3(256), 0, s, a)
    if (split) {
        if (epi == GEPI_STORE) CM_GEMM(2, GEPI_STORE); else if (epi == GEPI_RESADD) CM_GEMM(2, GEPI_RESADD);
        else if (epi == GEPI_ACT_SPLIT) CM_GEMM(2, GEPI_ACT_SPLIT); else CM_GEMM(2, GEPI_SILUMUL);
    } else {
        if (epi == GEPI_STORE) CM_GEMM(1, GEPI_STORE); else if (epi == GEPI_RESADD) CM_GEMM(1, GEPI_RESADD);
        else if (epi == GEPI_ACT_SPLIT) CM_GEMM(1, GEPI_ACT_SPLIT); else CM_GEMM(1, GEPI_SILUMUL);
    }
#undef CM_GEMM
    return true;
}
// kvt: KV_BF16 | KV_F16 | KV_F32 (the element type the kernel READS: f32 for the int8 / int4 shadow)
// shares of the keys for a launch of the fast path (key tiles of 64 tokens; at head_dim 256, whose waves take halves of them, counted in those): `fill` blocks keep the chip busy (two on a CU, one); a share of fewer than eight
// key tiles is not worth the merging launch, which costs more the more rows there are: at least a tile for every nine of the blocks that there are without shares.  us a layer of
// width 1024, whole / shared: 500 rows (256 blocks) behind 512 / 1024 / 2048 / 3584 tokens, 32 heads of 128: 132.5 / 135.9, 144.2 / 145.2, 167.3 / 163.5, 201.6 / 191.5; 384 rows (192)
// behind 1024 145.4 / 144.1; 256 rows (128) behind 1024 123.5 / 115.1; 64 rows behind 1024 / 3584 79.2 / 73.1, 136.7 / 78.4; 16 heads, 500 rows (128) behind 512 123.4 / 118.4;
// 8 heads of 256, 500 rows (64) behind 512 / 3584 738 / 705, 895 / 740 (four layers, one of them attention)
int attn_prefill_shares(int rows, int start, int heads, int D) {
    const int fill = D == 128 ? 512 : 256, kt = D == 128 ? 64 : 32, blocks = heads * ((rows + 63) / 64), tiles = (start + rows + kt - 1) / kt;
    return tiles * 9 < blocks ? 1 : std::max(1, std::min(std::min(fill / std::max(1, blocks), tiles / 8), 16));
}
static int prefill_split(const AttnPreArgs& a, int D) {
    if (a.tiles != nullptr || a.ws == nullptr) return 1;
    int n = attn_prefill_shares(a.S, a.start_pos, a.Hq, D);
    while (n > 1 && (size_t)n * a.S * a.Hq * (D + 2) > a.ws_floats) --n;
    return n;
}
// Which of the two head_dim-128 kernels takes query tiles whose walks are `walks` key tiles together (of one head) and `longest` at most.  attn_prefill_fast_kernel has 512 places; a launch of
// more tiles fills them again as the short ones end, so that what it takes is its longest walk until the work is more than about seven tenths of 512 of those: there attn_prompt_pair_kernel, with all
// its waves at once, is ahead.  us a layer, that kernel - this one: from the start of a prompt 16 heads 512 / 672 / 704 / 768 / 832 / 1024 tiles (0.52 / 0.67 / 0.70 / 0.77 / 0.83 / 1.02 of 512) -13 /
// -12 / 0 / +4 / +25 / +30, 32 heads 544 / 672 (0.69) / 704 (0.72) / 896 / 1024 -7 / -6 / +4 / +13 / +22, 24 heads 672 (0.68) / 720 (0.73) -6 / +8, 64 heads 640 (0.69) / 704 (0.75) -2 / +4, 8 heads 528 (0.53) -28; behind 512 tokens 16 heads
// 560 .. 608 (0.64 .. 0.70) -4 .. -1, 640 (0.74) 0, 32 heads 544 .. 608 (0.72 .. 0.78) -2 .. -1; behind 1024 16 heads 528 (0.69) +2, 576 (0.75) +5; behind 2048 16 heads 512 / 528 / 560 (0.76 / 0.78 / 0.82)
// -13 / +16 / +11, 32 heads 544 (0.88) +12 .. +16; several prompts of 32 heads 1200 and eight of 64 (0.65) -5, 1300 and 200 (0.72) -5 .. -1, 700 twice (0.75) +1, 300 six times (1.12) +2
static bool attn_pairs(int heads, int nrep, int tiles, long long walks, int longest) { return nrep % 2 == 0 && heads * tiles > 512 && heads * walks * 10 > 512LL * 7 * longest; }
bool attn_prompt_pairs(int rows, int start, int heads, int nrep) {
    const int tiles = (rows + 63) / 64;
    long long walks = 0;
    int longest = 0;
    for (int i = 0; i < tiles; ++i) walks += longest = (start + std::min(64 * (i + 1), rows) + 63) / 64;
    return attn_pairs(heads, nrep, tiles, walks, longest);
}
// causal prompts over 2-byte pages
static void launch_prefill_fast(AttnPreArgs a, int D, int kvt, hipStream_t s) {
    a.nsplit = prefill_split(a, D);
    const dim3 grid(a.Hq, a.tiles != nullptr ? a.ntiles : (a.S + 63) / 64, a.nsplit);
    if (D == 256) launch_attn_prompt_wide(a, kvt, s);
    else if (a.nsplit == 1 && (a.tiles != nullptr ? attn_pairs(a.Hq, a.nrep, a.ntiles, a.walks, a.longest) : attn_prompt_pairs(a.S, a.start_pos, a.Hq, a.nrep))) launch_attn_prompt_pair(a, kvt, s);
    else if (kvt == KV_F16) hipLaunchKernelGGL((attn_prefill_fast_kernel<KV_F16>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((attn_prefill_fast_kernel<KV_BF16>), grid, dim3(256), 0, s, a);
    if (a.nsplit == 1) return;
    const dim3 rows((unsigned)(((size_t)a.S * a.Hq + 1024 / D - 1) / (1024 / D)));
    if (D == 256) hipLaunchKernelGGL(attn_prefill_merge_kernel<256>, rows, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(attn_prefill_merge_kernel<128>, rows, dim3(256), 0, s, a);
}
void launch_attn_prefill(const AttnPreArgs& a, int D, int kvt, hipStream_t s) {
    const dim3 grid(a.Hq, a.tiles != nullptr ? a.ntiles : (a.S + 63) / 64);
    if (D == 128) {
        // the dense family's causal prompts over 2-byte pages: the fast path (CM_ATTN_PREFILL_FAST=0: the general kernel, A/B)
        static const int fast_env = getenv("CM_ATTN_PREFILL_FAST") ? atoi(getenv("CM_ATTN_PREFILL_FAST")) : 1;
        if (fast_env != 0 && a.gate == nullptr && (kvt == KV_F16 || kvt == KV_BF16) && a.page % 64 == 0 &&
            a.q_lo != nullptr) {
            launch_prefill_fast(a, D, kvt, s);
            return;
        }
        if (kvt == KV_F32) hipLaunchKernelGGL((attn_prefill_kernel<128, KV_F32>), grid, dim3(256), 0, s, a);
        else if (kvt == KV_F16) hipLaunchKernelGGL((attn_prefill_kernel<128, KV_F16>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((attn_prefill_kernel<128, KV_BF16>), grid, dim3(256), 0, s, a);
    } else {
        // the hybrid family's gated head_dim-256 attention: attn_prompt_wide_kernel
        static const int fast_env = getenv("CM_ATTN_PREFILL_FAST") ? atoi(getenv("CM_ATTN_PREFILL_FAST")) : 1;
        if (fast_env != 0 && (kvt == KV_F16 || kvt == KV_BF16) && a.page % 64 == 0 && a.q_lo != nullptr) {
            launch_prefill_fast(a, D, kvt, s);
            return;
        }
        if (kvt == KV_F32) hipLaunchKernelGGL((attn_prefill_kernel<256, KV_F32>), grid, dim3(256), 0, s, a);
        else if (kvt == KV_F16) hipLaunchKernelGGL((attn_prefill_kernel<256, KV_F16>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((attn_prefill_kernel<256, KV_BF16>), grid, dim3(256), 0, s, a);
    }
}

}  // namespace cm
