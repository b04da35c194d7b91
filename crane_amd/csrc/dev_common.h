// Device-side helpers shared by all gfx950 kernels (wave64, CDNA4).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cm {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(4))) short bf16x4;

constexpr int WAVE = 64;

// ---- bf16 <-> f32 (bit tricks; RNE on the way down, finite inputs) ---------
__device__ __forceinline__ float bf16_lo(uint32_t packed) { return __uint_as_float(packed << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t packed) { return __uint_as_float(packed & 0xFFFF0000u); }
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }
// gfx950 converts in hardware (v_cvt_pk_bf16_f32, round to nearest even): one instruction per PAIR instead of five
// integer ops per value
typedef __attribute__((ext_vector_type(2))) float cm_f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 cm_bf16x2;
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    const cm_bf16x2 v = __builtin_convertvector((cm_f32x2){lo, hi}, cm_bf16x2);
    uint32_t r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}
__device__ __forceinline__ uint16_t f32_to_bf16(float f) { return (uint16_t)(pack_bf16x2(f, 0.f) & 0xFFFFu); }
__device__ __forceinline__ float bf16_round(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// ---- f16 <-> f32 (CM_KV_F16 pages: K/V cached as IEEE binary16 -- the bytes of a bf16 page, 11 significand bits instead
// of 8; v_cvt_f16_f32 rounds to nearest even and keeps subnormals, the clamp saturates instead of overflowing to inf) ----
typedef __attribute__((ext_vector_type(2))) _Float16 cm_f16x2;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
__device__ __forceinline__ float f16_lo(uint32_t packed) { return (float)__builtin_bit_cast(cm_f16x2, packed)[0]; }
__device__ __forceinline__ float f16_hi(uint32_t packed) { return (float)__builtin_bit_cast(cm_f16x2, packed)[1]; }
__device__ __forceinline__ float f16_to_f32(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ uint16_t f32_to_f16(float f) {
    const _Float16 h = (_Float16)fminf(fmaxf(f, -65504.f), 65504.f);
    return __builtin_bit_cast(uint16_t, h);
}
// from memory into LDS without passing registers: every lane's 16 (4) bytes at its gsrc land at lds_base + 16 (4) * lane.  M0 carries the LDS base and
// belongs to the compiler: saved and restored around the instruction.  Counted by vmcnt like any load
__device__ __forceinline__ void lds_load16(const void* gsrc, uint32_t lds_base) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(gsrc), "s"(lds_base) : "memory");
}
// the same from base + off, the base in scalar registers
__device__ __forceinline__ void lds_load16_at(const char* base, uint32_t off, uint32_t lds_base) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_base) : "memory");
}
__device__ __forceinline__ void lds_load4(const void* gsrc, uint32_t lds_base) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(gsrc), "s"(lds_base) : "memory");
}
// internal KV-page element types (template parameter KVT of the attention kernels, Model::kv_mode)
enum { KV_BF16 = 0, KV_F32 = 1, KV_INT8 = 2, KV_INT4 = 3, KV_F16 = 4 };
// one cached 16-bit element pair -> f32 (bf16: bit shifts; f16: v_cvt_f32_f16)
template <int KVT> __device__ __forceinline__ float kv16_lo(uint32_t p) { return KVT == KV_F16 ? f16_lo(p) : bf16_lo(p); }
template <int KVT> __device__ __forceinline__ float kv16_hi(uint32_t p) { return KVT == KV_F16 ? f16_hi(p) : bf16_hi(p); }
template <int KVT> __device__ __forceinline__ uint16_t kv16_from_f32(float f) { return KVT == KV_F16 ? f32_to_f16(f) : f32_to_bf16(f); }
template <int KVT> __device__ __forceinline__ float kv16_to_f32(uint16_t h) { return KVT == KV_F16 ? f16_to_f32(h) : bf16_to_f32(h); }

// KVT = 4 (f16 pages): the same tiles on the f16 matrix-core instructions -- K rows and V^T fragments are the cached halves,
// q and p are split into f16 hi + lo (q is O(10) after the QK-norm, p <= 1: both far inside the binary16 range).
template <int KVT>
__device__ __forceinline__ f32x4 mma_k32(const bf16x8& a, const bf16x8& b, const f32x4& c) {
    if constexpr (KVT == KV_F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <int KVT>
__device__ __forceinline__ f32x4 mma_k16(const bf16x4& a, const bf16x4& b, const f32x4& c) {
    if constexpr (KVT == KV_F16) return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Workgroups go round the eight XCDs: the place of workgroup `id` of `all` where those of an XCD are neighbours
__device__ __forceinline__ int xcd_neighbours(int id, int all) { return (id & 7) * (all >> 3) + min(id & 7, all & 7) + (id >> 3); }

// four f32 as bf16 hi + lo planes; four weights as two terms of the pages' type
__device__ __forceinline__ void split_store4(uint16_t* hi, uint16_t* lo, size_t off, const float v[4]) {
    uint16_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = f32_to_bf16(v[i]);
        l[i] = f32_to_bf16(v[i] - bf16_to_f32(h[i]));
    }
    *(u32x2*)(hi + off) = (u32x2){(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
    if (lo) *(u32x2*)(lo + off) = (u32x2){(uint32_t)l[0] | ((uint32_t)l[1] << 16), (uint32_t)l[2] | ((uint32_t)l[3] << 16)};
}
template <int KVT>
__device__ __forceinline__ void p_split4(const float (&p)[4], bf16x4& hi, bf16x4& lo) {
    if constexpr (KVT == KV_F16) {
        typedef __attribute__((ext_vector_type(2))) _Float16 h2;
        const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(p[0], p[1]));
        const h2 b = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(p[2], p[3]));
        const h2 c = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(p[0] - (float)a[0], p[1] - (float)a[1]));
        const h2 d = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(p[2] - (float)b[0], p[3] - (float)b[1]));
        const u32x2 hv = {__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
        const u32x2 lv = {__builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)};
        hi = __builtin_bit_cast(bf16x4, hv); lo = __builtin_bit_cast(bf16x4, lv);
    } else {
        const uint32_t a = pack_bf16x2(p[0], p[1]), b = pack_bf16x2(p[2], p[3]);
        const uint32_t c = pack_bf16x2(p[0] - bf16_lo(a), p[1] - bf16_hi(a)), d = pack_bf16x2(p[2] - bf16_lo(b), p[3] - bf16_hi(b));
        const u32x2 hv = {a, b}, lv = {c, d};
        hi = __builtin_bit_cast(bf16x4, hv); lo = __builtin_bit_cast(bf16x4, lv);
    }
}

// ---- streaming (non-temporal) 16-byte load: weights are read once ----------
__device__ __forceinline__ u32x4 ld_nt16(const void* p) {
    return __builtin_nontemporal_load((const u32x4*)p);
}
__device__ __forceinline__ u32x4 ld16(const void* p) { return *(const u32x4*)p; }

// ---- DPP cross-lane (no LDS traffic) ----------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// The value of lane l ^ 1, 2, 4, 8, 16 without the LDS (a __shfl_xor is a ds_bpermute, about 100 cycles in a chain that waits for it; these are 4 .. 8).  Both lanes of a pair active.
// permlane16_swap(v, v): {rows 0 0 2 2, rows 1 1 3 3} of 16 lanes; permlane32_swap(v, v): {lower half twice, upper half twice}
typedef __attribute__((ext_vector_type(2))) unsigned int cm_u32x2;
__device__ __forceinline__ cm_u32x2 rows16(float v) { return __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false); }
__device__ __forceinline__ cm_u32x2 rows32(float v) { return __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false); }
template <int X>
__device__ __forceinline__ float lane_xor(float v) {
    static_assert(X == 1 || X == 2 || X == 4 || X == 8 || X == 16, "");
    if constexpr (X == 1) return dpp_mov<0xB1>(v);                    // quad_perm [1,0,3,2]
    else if constexpr (X == 2) return dpp_mov<0x4E>(v);               // quad_perm [2,3,0,1]
    else if constexpr (X == 4) return dpp_mov<0x141>(dpp_mov<0x1B>(v));   // row_half_mirror (l ^ 7) of quad_perm [3,2,1,0] (l ^ 3)
    else if constexpr (X == 8) return dpp_mov<0x128>(v);              // row_ror 8
    else { const cm_u32x2 r = rows16(v); return __uint_as_float(threadIdx.x & 16 ? r[0] : r[1]); }
}
// v summed, or its maximum taken, over lanes l, l ^ 16 and then l ^ 32
__device__ __forceinline__ float rows_sum(float v) {
    cm_u32x2 r = rows16(v);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = rows32(v);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float rows_max(float v) {
    cm_u32x2 r = rows16(v);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = rows32(v);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// sum over an aligned group of L lanes (a power of two), partners L / 2 apart first
__device__ __forceinline__ float group_sum(float v, int L) {
    if (L > 32) { const cm_u32x2 r = rows32(v); v = __uint_as_float(r[0]) + __uint_as_float(r[1]); }
    if (L > 16) { const cm_u32x2 r = rows16(v); v = __uint_as_float(r[0]) + __uint_as_float(r[1]); }
    if (L > 8) v += lane_xor<8>(v);
    if (L > 4) v += lane_xor<4>(v);
    if (L > 2) v += lane_xor<2>(v);
    if (L > 1) v += lane_xor<1>(v);
    return v;
}
// sum over each aligned group of 16 lanes ("row"); every lane of the row gets it
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_mov<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dpp_mov<0x141>(v);   // row_half_mirror
    v += dpp_mov<0x140>(v);   // row_mirror
    return v;
}
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_mov<0xB1>(v));
    v = fmaxf(v, dpp_mov<0x4E>(v));
    v = fmaxf(v, dpp_mov<0x141>(v));
    v = fmaxf(v, dpp_mov<0x140>(v));
    return v;
}
// full 64-lane sum, result wave-uniform
__device__ __forceinline__ float wave_sum(float v) {
    v = row16_sum(v);
    float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return (a + b) + (c + d);
}
__device__ __forceinline__ float wave_max(float v) {
    v = row16_max(v);
    float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// ---- synthetic weights (crane_amd/synth.py) ------------------------------------
__host__ __device__ __forceinline__ uint32_t fmix32(uint32_t h) {
    h ^= h >> 16; h *= 0x85EBCA6Bu; h ^= h >> 13; h *= 0xC2B2AE35u; h ^= h >> 16;
    return h;
}
__host__ __device__ __forceinline__ float synth_val(uint32_t idx, uint32_t tseed, float mul, float off) {
#pragma clang fp contract(off)      // (the _rn intrinsics below are plain operators in this ROCm: contraction is switched off by name)
    uint32_t h = fmix32(idx * 0x9E3779B1u + tseed);
    int c = (int)((h & 0xFF) + ((h >> 8) & 0xFF) + ((h >> 16) & 0xFF) + (h >> 24)) - 510;
#if defined(__HIP_DEVICE_COMPILE__)
    return __fadd_rn(off, __fmul_rn((float)c, mul));   // no FMA contraction: must match numpy bit-for-bit
#else
    volatile float prod = (float)c * mul;
    return off + prod;
#endif
}

// decode-step state living in HBM so a captured hipGraph can be replayed
struct StepState {
    uint32_t token;     // token to feed this step
    int32_t pos;        // its KV position
    uint32_t next;      // arg-max result of this step
    int32_t pad;        // token-ring write index
    int32_t slot;       // active sequence slot (indexes the per-sequence GDN state pools)
    int32_t rsv[3];     // rsv[0] = rotary position delta (MRoPE counter - cache position); rsv[1] = epoch base and
                        // rsv[2] = error code of the persistent chain kernel (kernels_engine.hip)
};

// sums that another XCD's block reads: written through to where all of them read, and read from there, so that their counter needs no fence (a fence writes back
// and drops a whole L2: the shares of lay_attn_tile_kernel 18 us a launch without, 52 with)
__device__ __forceinline__ void put_through(float* p, float x, float y) {
    __hip_atomic_store((unsigned long long*)p, (unsigned long long)__float_as_uint(y) << 32 | __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 get_through(const float* p) {
    const unsigned long long v = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}

}  // namespace cm
