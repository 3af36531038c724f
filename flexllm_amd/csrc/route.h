// The choice of experts, shared by the kernels that make it.
#pragma once
#include "elem.h"

namespace fx {

constexpr int kMaxExperts = 1024, kMaxTop = 32;

// Expert choice of one token by one wave: softmax over the router outputs, the `top` largest (ties: lower index), their
// weights divided by their sum.  Lane k < top gets choice k, an expert's number whatever the outputs are, and its weight.
// NE: 64-expert pieces (experts <= 64 NE).
template <int NE>
__device__ __forceinline__ void route_wave_n(const float* __restrict__ z, int experts, int top, int& pick, float& weight) {
    const int lane = threadIdx.x & 63;
    float v[NE];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NE; i++) {
        v[i] = i * 64 + lane < experts ? z[i * 64 + lane] : -INFINITY;
        mx = fmaxf(mx, v[i]);
    }
    mx = wave_max(mx);
    float den = 0.0f;
#pragma unroll
    for (int i = 0; i < NE; i++) {
        v[i] = i * 64 + lane < experts ? exp_f<false>(v[i] - mx) : -1.0f;
        den += fmaxf(v[i], 0.0f);
    }
    den = wave_sum(den);
    float sum = 0.0f;
    pick = 0;
    weight = 0.0f;
    for (int k = 0; k < top; k++) {
        float best = v[0];
#pragma unroll
        for (int i = 1; i < NE; i++) best = fmaxf(best, v[i]);
        best = wave_max(best);
        int bi = -1;                                      // lowest index that holds the maximum
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const unsigned long long hit = __ballot(v[i] == best);
            if (bi < 0 && hit) {
                const int l = __builtin_ctzll(hit);
                bi = i * 64 + l;
                if (lane == l) v[i] = -1.0f;
            }
        }
        const float s = best / den;
        sum += s;
        if (lane == k) { pick = bi; weight = s; }
    }
    weight = weight / (sum + 1e-20f);
    // where outputs are not numbers there may be nothing left to take, or only lanes without an expert
    pick = min(max(pick, 0), experts - 1);
}
__device__ __forceinline__ void route_wave(const float* __restrict__ z, int experts, int top, int& pick, float& weight) {
    if (experts <= 64) route_wave_n<1>(z, experts, top, pick, weight);
    else if (experts <= 256) route_wave_n<4>(z, experts, top, pick, weight);
    else route_wave_n<kMaxExperts / 64>(z, experts, top, pick, weight);
}

}  // namespace fx
