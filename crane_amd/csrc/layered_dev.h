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

}  // namespace cm
