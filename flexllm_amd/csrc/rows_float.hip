// Row kernels of the floating-point layers: weight packing, embedding rows, and the fused
// residual + norm after a sublayer + norm before the next one (with the mixture's weighted sum in front).
#include "float_ops.h"
#include "gemm_walk.h"

namespace fx {

// dst row i*row_step + row_off = source row i, widened or copied, zero beyond k (rows are kpad long)
template <typename ET>
__global__ __launch_bounds__(256) void pack_rows_kernel(const bf16_t* __restrict__ src, ET* __restrict__ dst, int k, int kpad, int row_step, int row_off) {
    const bf16_t* s = src + (size_t)blockIdx.x * k;
    ET* d = dst + ((size_t)blockIdx.x * row_step + row_off) * kpad;
    for (int i = threadIdx.x; i < kpad; i += 256) d[i] = i < k ? (ET)s[i] : (ET)0.0f;
}
template <typename ET>
int pack_rows(const bf16_t* src, ET* dst, int n, int k, int kpad, int row_step, int row_off, hipStream_t st) {
    FX_REQUIRE(src && dst && n > 0 && k > 0 && kpad >= k, "pack_rows: n=%d k=%d", n, k);
    pack_rows_kernel<ET><<<n, 256, 0, st>>>(src, dst, k, kpad, row_step, row_off);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}
template int pack_rows<bf16_t>(const bf16_t*, bf16_t*, int, int, int, int, int, hipStream_t);
template int pack_rows<float>(const bf16_t*, float*, int, int, int, int, int, hipStream_t);

static __global__ __launch_bounds__(256) void widen_rows_kernel(const bf16_t* __restrict__ src, float* __restrict__ dst, int n, float add) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = (float)src[i] + add;
}
int widen_rows(const bf16_t* src, float* dst, int n, float add, hipStream_t st) {
    FX_REQUIRE(src && dst && n > 0, "widen_rows: n=%d", n);
    widen_rows_kernel<<<(n + 255) / 256, 256, 0, st>>>(src, dst, n, add);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// Ids outside [0, vocab) are replaced by 0 and reported through *err = 2, as in embed_rows_kernel.
static __global__ __launch_bounds__(256) void embed_bf16_kernel(const bf16_t* __restrict__ table, float scale, const int* __restrict__ tokens, float* __restrict__ x,
                                                                int width, int vocab, int* __restrict__ err) {
    int tk = tokens[blockIdx.x];
    if ((unsigned)tk >= (unsigned)vocab) {
        if (err && threadIdx.x == 0) err[0] = 2;
        tk = 0;
    }
    const bf16_t* s = table + (size_t)tk * width;
    float* const to = x + (size_t)blockIdx.x * width;
    if (width % 8 == 0) {                                  // rows start on 16 bytes
        for (int i = threadIdx.x * 8; i < width; i += 256 * 8) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(s + i);
#pragma unroll
            for (int h = 0; h < 8; h += 4) *reinterpret_cast<f32x4*>(to + i + h) = f32x4{(float)v[h] * scale, (float)v[h + 1] * scale, (float)v[h + 2] * scale, (float)v[h + 3] * scale};
        }
        return;
    }
    for (int i = threadIdx.x; i < width; i += 256) to[i] = (float)s[i] * scale;
}
int embed_rows_bf16(const bf16_t* table, float scale, const int* tokens, int n, float* x, int width, int vocab, int* err, hipStream_t st) {
    embed_bf16_kernel<<<n, 256, 0, st>>>(table, scale, tokens, x, width, vocab, err);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

static __global__ void put_state_kernel(int* state, int pos, int step) { state[0] = pos; state[1] = step; }
static __global__ void advance_kernel(int* state, int n) { state[0] += n; }
int set_state_launch(int* state, int pos, int step, hipStream_t st) {
    put_state_kernel<<<1, 1, 0, st>>>(state, pos, step);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}
int advance_launch(int* state, int n, hipStream_t st) {
    advance_kernel<<<1, 1, 0, st>>>(state, n);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// y at `at`, its parts in order.
template <typename V>
__device__ __forceinline__ V sum_parts(const RowArgs& a, size_t at) {
    V v = *reinterpret_cast<const V*>(a.y + at);
#pragma unroll 4
    for (int p = 1; p < a.y_parts; p++) v += *reinterpret_cast<const V*>(a.y + p * a.y_stride + at);
    return v;
}

// One workgroup per row; the row stays in LDS between the two norms.
template <typename ET>
__global__ __launch_bounds__(256) void norm_rows_kernel(RowArgs a) {
    extern __shared__ float row[];
    __shared__ float red[4];
    const int t = threadIdx.x, r = blockIdx.x;
    const float* x = a.x + (size_t)(a.rows_src ? a.rows_src[r] : r) * a.width;
    float* x_new = (a.x_new ? a.x_new : a.x) + (size_t)r * a.width;
    const bool mix = a.ys != nullptr, have_y = a.y || mix;
    if (have_y || a.x0) {
        float sg = 1.0f;
        if (mix && a.y) sg = sigmoid_f(a.route[(size_t)r * a.ld_route + a.experts]);
        float ss = 0.0f;
        for (int i = t; i < a.width; i += 256) {
            float v = 0.0f;
            if (mix) {
                for (int k = 0; k < a.top; k++) v = fma_f(a.pick_w[r * a.top + k], a.ys[(size_t)a.pos_of[r * a.top + k] * a.ldy + i], v);
                if (a.y) v = fma_f(sg, sum_parts<float>(a, (size_t)r * a.ldy + i), v);
            } else if (a.y) {
                v = sum_parts<float>(a, (size_t)r * a.ldy + i);
            }
            row[i] = v;
            ss = fma_f(v, v, ss);
        }
        const bool post = have_y && a.gb;
        const float rs = post ? 1.0f / sqrtf(block_sum<4>(ss, red) / (float)a.width + a.eps) : 1.0f;
        for (int i = t; i < a.width; i += 256) {
            float v = x[i] + (post ? row[i] * rs * a.gb[i] : row[i]);
            if (a.x0) v += a.x0[(size_t)r * a.width + i];
            row[i] = v;
            if (!a.rows_src) x_new[i] = v;
        }
    } else {
        for (int i = t; i < a.width; i += 256) row[i] = x[i];
    }
    if (!a.h) return;
    float ss = 0.0f;
    for (int i = t; i < a.width; i += 256) ss = fma_f(row[i], row[i], ss);
    const float rx = 1.0f / sqrtf(block_sum<4>(ss, red) / (float)a.width + a.eps);
    if (a.h_f32) {
        float* h = static_cast<float*>(a.h) + (size_t)r * a.ldh;
        for (int i = t; i < a.width; i += 256) h[i] = row[i] * rx * a.g[i];
    } else {
        ET* h = static_cast<ET*>(a.h) + (size_t)r * a.ldh;
        for (int i = t; i < a.ldh; i += 256) h[i] = i < a.width ? (ET)(row[i] * rx * a.g[i]) : (ET)0.0f;
    }
}

// The same for widths that are a multiple of 4 and at most 256 * 4 * V: the row stays in registers, 16-byte accesses.
// What bounds it: up to a few hundred rows the chain of trips to memory, so that all that does not hang on another trip's answer is asked for at the
// start (norm weights, all parts of y, the places of a mixture's rows, then those rows together); with thousands of rows the memory's rate.
// us, requests: lopazen-1b 5 tokens 1024 -> 973, 100 tokens 1400 -> 1345, nifunex-1b-moe 64 tokens 2125 -> 2094; 1000 rows and more as before.
template <typename ET, int V, bool MIX>
__global__ __launch_bounds__(256) void norm_rows_vec_kernel(RowArgs a) {
    arguments(a.x, a.x_new, a.x0, a.y, a.ldy, a.y_parts, a.y_stride, a.gb, a.g, a.width, a.h, a.ldh, a.rows_src, a.ys, a.top);
    __shared__ float red[4];
    const int t = threadIdx.x, r = blockIdx.x, n4 = a.width >> 2;
    const bool have_y = a.y || MIX, post = have_y && a.gb;
    int at[V];                                             // a lane behind the row's end reads its last piece and has zeros
    bool in[V];
#pragma unroll
    for (int i = 0; i < V; i++) { in[i] = t + i * 256 < n4; at[i] = min(t + i * 256, n4 - 1) * 4; }
    auto get = [&](f32x4 (&d)[V], const float* from) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < V; i++) d[i] = *reinterpret_cast<const f32x4*>(from + at[i]);
    };
    f32x4 v[V], y[V], x0[V], gb[V], g[V];
    get(v, a.x + (size_t)(a.rows_src ? a.rows_src[r] : r) * a.width);
    if (a.y) get(y, a.y + (size_t)r * a.ldy);
    if (a.x0) get(x0, a.x0 + (size_t)r * a.width);
    if (post) get(gb, a.gb);
    if (a.h) get(g, a.g);
    if (a.y)
        for (int p = 1; p < a.y_parts; p += 3) {
            f32x4 u[3][V];
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (p + q < a.y_parts) get(u[q], a.y + (p + q) * a.y_stride + (size_t)r * a.ldy);
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (p + q < a.y_parts)
#pragma unroll
                    for (int i = 0; i < V; i++) y[i] += u[q][i];
        }
    if constexpr (MIX) {
        constexpr int K = V > 2 ? 4 : 8;
        const float sg = a.y ? sigmoid_f(a.route[(size_t)r * a.ld_route + a.experts]) : 1.0f;
        f32x4 sum[V];
#pragma unroll
        for (int i = 0; i < V; i++) sum[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int k0 = 0; k0 < a.top; k0 += K) {
            f32x4 u[K][V];
            float w[K];
            int pos[K];
#pragma unroll
            for (int k = 0; k < K; k++) {
                const int k1 = r * a.top + min(k0 + k, a.top - 1);
                w[k] = a.pick_w[k1];
                pos[k] = a.pos_of[k1];
            }
#pragma unroll
            for (int k = 0; k < K; k++)
                if (k0 + k < a.top) get(u[k], a.ys + (size_t)pos[k] * a.ldy);
#pragma unroll
            for (int k = 0; k < K; k++)
                if (k0 + k < a.top)
#pragma unroll
                    for (int i = 0; i < V; i++)
#pragma unroll
                        for (int e = 0; e < 4; e++) sum[i][e] = fma_f(w[k], u[k][i][e], sum[i][e]);
        }
#pragma unroll
        for (int i = 0; i < V; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) y[i][e] = a.y ? fma_f(sg, y[i][e], sum[i][e]) : sum[i][e];
    }
    if (have_y || a.x0) {
        float rs = 1.0f;
        if (post) {
            float ss = 0.0f;
#pragma unroll
            for (int i = 0; i < V; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) ss = in[i] ? fma_f(y[i][e], y[i][e], ss) : ss;
            rs = 1.0f / sqrtf(block_sum<4>(ss, red) / (float)a.width + a.eps);
        }
        float* x_new = (a.x_new ? a.x_new : a.x) + (size_t)r * a.width;
#pragma unroll
        for (int i = 0; i < V; i++) {
            if (have_y) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = v[i][e] + (post ? y[i][e] * rs * gb[i][e] : y[i][e]);
            }
            if (a.x0) v[i] += x0[i];
            if (in[i] && !a.rows_src) *reinterpret_cast<f32x4*>(x_new + at[i]) = v[i];
        }
    }
    if (!a.h) return;
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < V; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) ss = in[i] ? fma_f(v[i][e], v[i][e], ss) : ss;
    const float rx = 1.0f / sqrtf(block_sum<4>(ss, red) / (float)a.width + a.eps);
#pragma unroll
    for (int i = 0; i < V; i++) {
        if (!in[i]) continue;
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = v[i][e] * rx * g[i][e];
        if (a.h_f32 || std::is_same<ET, float>::value) {
            *reinterpret_cast<f32x4*>(static_cast<float*>(a.h) + (size_t)r * a.ldh + at[i]) = o;
        } else {
            bf16x4 b;
#pragma unroll
            for (int e = 0; e < 4; e++) b[e] = (bf16_t)o[e];
            *reinterpret_cast<bf16x4*>(static_cast<bf16_t*>(a.h) + (size_t)r * a.ldh + at[i]) = b;
        }
    }
}

template <typename ET>
int norm_rows(const RowArgs& a, hipStream_t st) {
    FX_REQUIRE(a.x && a.rows > 0 && a.width > 0 && a.width <= 16384 && (!a.h || (a.g && a.ldh >= a.width)), "norm_rows: rows=%d width=%d", a.rows, a.width);
    const bool vec = a.width % 4 == 0 && a.ldy % 4 == 0 && a.ldh % 4 == 0;
    auto launch = [&](auto mix) {
        constexpr bool MIX = decltype(mix)::value;
        if (a.width <= 1024) norm_rows_vec_kernel<ET, 1, MIX><<<a.rows, 256, 0, st>>>(a);
        else if (a.width <= 2048) norm_rows_vec_kernel<ET, 2, MIX><<<a.rows, 256, 0, st>>>(a);
        else norm_rows_vec_kernel<ET, 4, MIX><<<a.rows, 256, 0, st>>>(a);
    };
    if (vec && a.width <= 4096 && a.ys) launch(std::true_type());
    else if (vec && a.width <= 4096) launch(std::false_type());
    else norm_rows_kernel<ET><<<a.rows, 256, a.width * sizeof(float), st>>>(a);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}
template int norm_rows<bf16_t>(const RowArgs&, hipStream_t);
template int norm_rows<float>(const RowArgs&, hipStream_t);

}  // namespace fx
