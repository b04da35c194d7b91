// Device-side pieces shared by the layer-list decoders' kernel files.
#pragma once
#include "dev_common.h"
#include "layered.h"

namespace cm {

__device__ __forceinline__ float lay_act(float v, int act, float param = 1.f) {
    switch (act) {
        case LACT_RELU2: { const float r = fmaxf(v, 0.f); return r * r; }
        case LACT_LOGSIG: return param * (fminf(v, 0.f) - log1pf(expf(-fabsf(v))));      // ln sigmoid(v), no overflow either way
        case LACT_SOFTCAP: return param * tanhf(v / param);
        case LACT_SILU: return v / (1.f + __expf(-v));
        case LACT_SIGMOID: return 1.f / (1.f + __expf(-v));
        case LACT_GELU_TANH: {
            const float u = 0.7978845608028654f * (v + 0.044715f * v * v * v);
            return 0.5f * v * (1.f + tanhf(u));
        }
        default: return v;
    }
}
// capped gated product: g = min(g, cap), u = clamp(u, -cap, cap): g sigmoid(1.702 g) (u + 1)
__device__ __forceinline__ float lay_capglu(float g, float u, float cap) {
    g = fminf(g, cap);
    u = fminf(fmaxf(u, -cap), cap);
    return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
}

// a pair turned by an angle; spelled out, so that every kernel rounds it alike
__device__ __forceinline__ float2 lay_turn(float2 v, float cs, float sn) { return make_float2(fmaf(v.x, cs, -(v.y * sn)), fmaf(v.y, cs, v.x * sn)); }

// One wave turns the E logits of token t in zs into choices and weights.  zs: [E] logits, then choice scores (shared_gate: one more
// logit behind them); sc: [E] scores, [groups], [top].
__device__ __forceinline__ void lay_router_choose(float* zs, int t, int lane, int32_t* __restrict__ sel, float* __restrict__ wsel, int E, int top,
                                                  const RouterSpec& rs, const float* __restrict__ correction, int slots) {
    float* sc = zs + E + (rs.shared_gate ? 1 : 0);
    // wave 0: lane l owns outputs l, l + 64, ...; maxima, sums and the arg-max (lowest index among equals) are wave reductions
    auto arg_best = [&](bool want_max, int lo, int hi, float& bv) {      // over the live (not -inf) entries of zs[lo, hi)
        float v = 0.f; int at = 0x7fffffff;
        for (int ex = lo + lane; ex < hi; ex += 64) {
            const float z = zs[ex];
            if (z == -INFINITY) continue;
            if (at == 0x7fffffff || (want_max ? z > v : z < v)) { v = z; at = ex; }
        }
        for (int off = 32; off > 0; off >>= 1) {
            const float ov = __shfl_xor(v, off); const int oa = __shfl_xor(at, off);
            if (oa != 0x7fffffff && (at == 0x7fffffff || (want_max ? ov > v : ov < v) || (ov == v && oa < at))) { v = ov; at = oa; }
        }
        bv = v;
        return at;
    };
    // scores; the choice goes by score + correction (plain sigmoid scores: by the logits themselves, the same order -- unless groups are
    // compared by sums of scores)
    if (rs.softmax) {
        float mx = -INFINITY;
        for (int ex = lane; ex < E; ex += 64) mx = fmaxf(mx, zs[ex]);
        mx = wave_max(mx);
        float sum = 0.f;
        for (int ex = lane; ex < E; ex += 64) { const float p = expf(zs[ex] - mx); sc[ex] = p; sum += p; }
        sum = wave_sum(sum);
        for (int ex = lane; ex < E; ex += 64) sc[ex] /= sum;
    } else
        for (int ex = lane; ex < E; ex += 64) sc[ex] = 1.f / (1.f + expf(-zs[ex]));
    if (rs.softmax || correction || (rs.groups > 1 && rs.group_top > 1))
        for (int ex = lane; ex < E; ex += 64) zs[ex] = sc[ex] + (correction ? correction[ex] : 0.f);
    __builtin_amdgcn_wave_barrier();
    if (rs.groups > 1) {                   // keep the best groups: every pass removes the worst remaining one
        const int per = E / rs.groups;
        float* gb = sc + E;                // [groups] a group's score: its largest choice score, or the sum of its two largest (-inf: removed)
        for (int g = lane; g < rs.groups; g += 64) {
            float best = -INFINITY, second = -INFINITY;
            for (int j = 0; j < per; ++j) {
                const float v = zs[g * per + j];
                second = fmaxf(second, fminf(best, v));
                best = fmaxf(best, v);
            }
            gb[g] = rs.group_top > 1 && per > 1 ? best + second : best;
        }
        for (int drop = 0; drop < rs.groups - rs.keep_groups; ++drop) {
            // the worst live group, among equals the last one
            float v = 0.f; int at = -1;
            for (int g = lane; g < rs.groups; g += 64) {
                const float b = gb[g];
                if (b == -INFINITY) continue;
                if (at < 0 || b <= v) { v = b; at = g; }
            }
            for (int off = 32; off > 0; off >>= 1) {
                const float ov = __shfl_xor(v, off); const int oa = __shfl_xor(at, off);
                if (oa >= 0 && (at < 0 || ov < v || (ov == v && oa > at))) { v = ov; at = oa; }
            }
            if (at < 0) break;
            if (lane == 0) gb[at] = -INFINITY;
            for (int j = lane; j < per; j += 64) zs[at * per + j] = -INFINITY;
            __builtin_amdgcn_wave_barrier();      // LDS accesses of one wave complete in order; this keeps the compiler from moving them
        }
    }
    float* wl = sc + E + rs.groups;        // [top] the chosen scores
    float wsum = 0.f;
    // up to a wave's width: a score per lane, maxima by row operations and the lowest lane that has one (an exchange over the wave takes six steps of two
    // shuffles per choice, 1.6 us of four out of 14).  Scores that are no numbers take the exchange
    float own = lane < E ? zs[lane] : -INFINITY;
    const bool lanes = E <= 64 && !__any(own != own);
    for (int k = 0; k < top; ++k) {
        float bz;
        int best;
        if (lanes) {
            bz = wave_max(own);
            const unsigned long long at = bz == -INFINITY ? 0 : __ballot(own == bz);
            best = at ? __builtin_ctzll(at) : 0;
            if (lane == best) own = -INFINITY;
        } else {
            best = arg_best(true, 0, E, bz);
            if (best == 0x7fffffff) best = 0;
        }
        const float w = sc[best];
        wsum += w;
        if (lane == 0) {
            sel[(size_t)t * top + k] = best;
            wl[k] = w;
            zs[best] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
    }
    for (int k = lane; k < top; k += 64) wsel[(size_t)t * slots + k] = (rs.normalise ? wl[k] / (wsum + 1e-20f) : wl[k]) * rs.scale;
    for (int k = top + lane; k < slots; k += 64) wsel[(size_t)t * slots + k] = rs.shared_gate ? 1.f / (1.f + expf(-zs[E])) : 1.f;
}

// Choice `slot` of lay_router_choose by itself, for at most 64 outputs without correction or groups, in every wave that calls it and with nothing written: the lane with `slot` better
// scores, equal ones in the lanes' order, as that function's maxima come one after another.  -1: it goes by another rule there (scores that are no numbers, a choice of none).  Scores
// are made and compared here as they are there; a change to one is a change to the other
__device__ __forceinline__ int lay_router_choice(const float* zs, int lane, int slot, int E, const RouterSpec& rs) {
    const float z = lane < E ? zs[lane] : -INFINITY;
    float own = z;
    if (rs.softmax) {
        const float mx = wave_max(z), p = lane < E ? expf(z - mx) : 0.f;
        own = p / wave_sum(p);
    }
    if (__any(lane < E && !(own > -INFINITY))) return -1;
    int better = 0;
    for (int j = 0; j < E; ++j) {
        const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(own), j));
        better += v > own || (v == own && j < lane);
    }
    const unsigned long long at = __ballot(lane < E && better == slot);
    return at ? __builtin_ctzll(at) : -1;
}

}  // namespace cm
