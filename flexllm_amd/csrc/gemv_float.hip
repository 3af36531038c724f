// Linears of one token: y = W h with W of ET (bfloat16 or float32) streamed once, h float32 in LDS.
//
// A workgroup of 256 threads walks groups of R weight rows; thread t reads 16-byte pieces t, t + 256, ... of each row.
// The first two groups are requested before the prologue (residual, norms) runs, so that its latency lies under the weight
// stream, and two groups stay in flight after that.  The R sums are reduced together (multi_sum_step).
#include "float_ops.h"
#include "gemm_walk.h"
#include "route.h"
#include <atomic>

namespace fx {

constexpr size_t kGemvTokensLds = 128 * 1024;             // vectors of gemv_tokens_kernel

// VEC: the prologue keeps its vectors in registers as float4 (k a multiple of 4, at most what the S pieces per thread cover);
// else any k, through LDS.  NT: the weights are read once on this chip and are requested as such (non-temporal): what they
// would push out of the caches stays, and the stream itself runs faster (16384 x 2048 bfloat16: 14.6 -> 13.9 us, the head of
// 128256 x 2048 90 -> 82 us).  With several tokens the grid rows share the weights through L2 and the ordinary loads stay.
template <typename ET, int R, int S, int PRO, bool VEC, bool NT>
__global__ __launch_bounds__(256) void gemv_float_kernel(GemvArgs g) {
    constexpr int CE = Chunk<ET>::N;
    extern __shared__ __attribute__((aligned(16))) float xs[];     // [kpad] the vector, and a piece of zeros for threads without one
    __shared__ float red[2][4 * R];
    __shared__ float nred[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int tok = PRO == 2 ? blockIdx.y / g.top : blockIdx.y;
    const ET* w = static_cast<const ET*>(g.w);
    const float* x = g.x + (size_t)tok * g.ldx;
    // ---- requests for the vector go out first: loads return in order, and the weights behind them are a long stream
    constexpr int Q = VEC ? S * CE / 4 : 1;               // float4 per thread
    f32x4 xv[Q], yv[Q], gb[Q], gv[Q];
    const int k4 = g.k >> 2;
    const bool have_y = PRO == 1 && g.y != nullptr, post = have_y && g.gb != nullptr;
    // gb holds the weight of the norm after the sublayer, or where there is none the other vector to add
    const float* extra = post ? g.gb : g.x0 ? g.x0 + (size_t)tok * g.ldx : nullptr;
    if constexpr (VEC) {
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        const float* y = g.y + (size_t)tok * g.ldy;
#pragma unroll
        for (int i = 0; i < Q; i++) {
            const int c = t + 256 * i;
            const bool in = c < k4;
            if constexpr (PRO == 1) yv[i] = in && have_y ? *reinterpret_cast<const f32x4*>(y + 4 * c) : zero;
            xv[i] = in ? *reinterpret_cast<const f32x4*>(x + 4 * c) : zero;
            if constexpr (PRO == 1) {
                gb[i] = in && extra ? *reinterpret_cast<const f32x4*>(extra + 4 * c) : zero;
                gv[i] = in ? *reinterpret_cast<const f32x4*>(g.g + 4 * c) : zero;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (PRO == 2) {
        int pick;                                         // every wave chooses for itself: no barrier before the weights
        float weight;
        route_wave(g.route + (size_t)tok * g.ld_route, g.experts, g.top, pick, weight);
        const int slot = blockIdx.y % g.top;
        w += (size_t)__builtin_amdgcn_readlane(pick, slot) * g.w_stride;
        if (blockIdx.x == 0 && t == slot) { g.pick[blockIdx.y] = pick; g.pick_w[blockIdx.y] = weight; }
    }
    const int nchunk = g.kpad / CE;                       // 16-byte pieces of a row
    const int ng = (g.n + R - 1) / R, G = gridDim.x;      // groups of R rows, dealt to the workgroups in turn
    i32x4 buf[2][R][S];
    auto piece = [&](int row, int c) {
        const i32x4* p = reinterpret_cast<const i32x4*>(w + (size_t)min(row, g.n - 1) * g.kpad + c * CE);
        if constexpr (NT) return __builtin_nontemporal_load(p);
        else return *p;
    };
    auto load = [&](int b, int grp) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int s = 0; s < S; s++) {
                const int c = s * 256 + t;
                buf[b][r][s] = c < nchunk ? piece(grp * R + r, c) : i32x4{0, 0, 0, 0};
            }
    };
    const int g0 = blockIdx.x;
    load(0, g0);
    if (g0 + G < ng) load(1, g0 + G);
    __builtin_amdgcn_sched_barrier(0);
    if (t < CE) xs[g.kpad + t] = 0.0f;
    // ---- the vector
    if constexpr (PRO == 1 && VEC) {
        float rs = 0.0f;
        if (post) {
            float ss = 0.0f;
#pragma unroll
            for (int i = 0; i < Q; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) ss = fma_f(yv[i][e], yv[i][e], ss);
            rs = 1.0f / sqrtf(block_sum<4>(ss, nred) / (float)g.k + g.eps);
        }
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < Q; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                xv[i][e] = post ? xv[i][e] + yv[i][e] * rs * gb[i][e] : xv[i][e] + yv[i][e] + gb[i][e];
                ss = fma_f(xv[i][e], xv[i][e], ss);
            }
        const float rx = 1.0f / sqrtf(block_sum<4>(ss, nred) / (float)g.k + g.eps);
#pragma unroll
        for (int i = 0; i < Q; i++) {
            const int c = t + 256 * i;
            f32x4 h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = xv[i][e] * rx * gv[i][e];
            if (4 * c < g.kpad) *reinterpret_cast<f32x4*>(xs + 4 * c) = h;
            if (blockIdx.x == 0 && c < k4) {
                if (g.x_new) *reinterpret_cast<f32x4*>(g.x_new + (size_t)tok * g.ldx + 4 * c) = xv[i];
                if (g.h_out) *reinterpret_cast<f32x4*>(g.h_out + (size_t)tok * g.ldh + 4 * c) = h;
            }
        }
    } else if constexpr (PRO == 1) {
        float rs = 0.0f;
        if (have_y) {
            const float* y = g.y + (size_t)tok * g.ldy;
            float ss = 0.0f;
            for (int i = t; i < g.k; i += 256) { const float v = y[i]; xs[i] = v; ss = fma_f(v, v, ss); }
            if (post) rs = 1.0f / sqrtf(block_sum<4>(ss, nred) / (float)g.k + g.eps);
        }
        float ss = 0.0f;
        for (int i = t; i < g.k; i += 256) {
            float v = x[i];
            if (post) v = v + xs[i] * rs * extra[i];
            else {
                if (have_y) v += xs[i];
                if (extra) v += extra[i];
            }
            xs[i] = v;
            ss = fma_f(v, v, ss);
            if (blockIdx.x == 0 && g.x_new) g.x_new[(size_t)tok * g.ldx + i] = v;
        }
        const float rx = 1.0f / sqrtf(block_sum<4>(ss, nred) / (float)g.k + g.eps);
        for (int i = t; i < g.kpad; i += 256) {
            const float v = i < g.k ? xs[i] * rx * g.g[i] : 0.0f;
            xs[i] = v;
            if (blockIdx.x == 0 && g.h_out && i < g.k) g.h_out[(size_t)tok * g.ldh + i] = v;
        }
    } else if constexpr (VEC) {
#pragma unroll
        for (int i = 0; i < Q; i++)
            if (4 * (t + 256 * i) < g.kpad) *reinterpret_cast<f32x4*>(xs + 4 * (t + 256 * i)) = xv[i];
    } else {
        for (int i = t; i < g.kpad; i += 256) xs[i] = i < g.k ? x[i] : 0.0f;
    }
    __syncthreads();
    // ---- the products
    auto dot = [&](int c, const i32x4& u, float& acc) {
        float wv[CE];
        Chunk<ET>::unpack(make_uint4(u[0], u[1], u[2], u[3]), wv);
#pragma unroll
        for (int q = 0; q < CE / 4; q++) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(xs + c * CE + q * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) acc = fma_f(wv[q * 4 + e], v[e], acc);
        }
    };
    auto process = [&](int b, int grp) {
        float acc[R];
        float bias[2] = {0.0f, 0.0f};                     // of the rows that this thread hands out below
        if (g.bias && t < R) {
            bias[0] = g.bias[min(grp * R + t, g.n - 1)];
            bias[1] = g.bias[min(grp * R + t + 1, g.n - 1)];
        }
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = 0.0f;
#pragma unroll
        for (int s = 0; s < S; s++) {
            const int c = min(s * 256 + t, nchunk);       // pieces beyond the row meet the zeros
#pragma unroll
            for (int r = 0; r < R; r++) dot(c, buf[b][r][s], acc[r]);
        }
        for (int c = S * 256 + t; c < nchunk; c += 256)
#pragma unroll
            for (int r = 0; r < R; r++) dot(c, piece(grp * R + r, c), acc[r]);
        multi_sum_step<R, 1>(acc, lane);
        if (lane < R) red[b][wave * R + multi_row<R>(lane)] = acc[0];
        __syncthreads();                                  // red alternates with the buffer: one barrier per group is enough
        if (t < R) {
            const int row = grp * R + t;
            float v[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int r = min(t + i, R - 1);
                v[i] = (red[b][r] + red[b][R + r]) + (red[b][2 * R + r] + red[b][3 * R + r]) + bias[i];
            }
            if (row < g.n) {
                const size_t o = blockIdx.y;
                if (row >= g.n_split) g.out32[o * g.ldo32 + row - g.n_split] = v[0];
                else if (!g.glu) g.out[o * g.ldo + row] = v[0];
                else if ((row & 1) == 0) g.out[o * g.ldo + (row >> 1)] = glu_f(g.glu, v[0], v[1], g.limit);
            }
        }
    };
    for (int grp = g0; grp < ng; grp += 2 * G) {
        process(0, grp);
        if (grp + 2 * G < ng) load(0, grp + 2 * G);
        if (grp + G < ng) {
            process(1, grp + G);
            if (grp + 3 * G < ng) load(1, grp + 3 * G);
        }
    }
}

template <typename ET, int R, int S>
static int launch_gemv_rs(const GemvArgs& g, int pro, int tokens, hipStream_t st) {
    const int rows_y = pro == 2 ? tokens * g.top : tokens;
    // workgroups that share the chip at a time (two per CU where the vector takes a third of LDS or more); each walks its
    // groups with the next one's weights in flight
    int wgs = (S > 4 ? 512 : 1024) / rows_y;
    if (wgs < 128) wgs = 128;
    // the workgroups of one walk for all tokens belong on one die, whose L2 hands the weights on: dies take workgroups in turn
    // (three tokens of 16 layers of 2048, 341 workgroups each: 1107 us, 336: 1031)
    if (tokens > 1) wgs &= ~7;
    const int ng = (g.n + R - 1) / R;
    const dim3 grid(ng < wgs ? ng : wgs, rows_y);
    const size_t lds = (size_t)(g.kpad + Chunk<ET>::N) * sizeof(float);
    const bool vec = g.k % 4 == 0 && g.ldx % 4 == 0 && g.ldy % 4 == 0 && g.ldh % 4 == 0 && g.kpad <= 256 * Chunk<ET>::N * S;
#define FX_GEMV(PRO)                                                                               \
    do {                                                                                           \
        if (vec && tokens == 1) gemv_float_kernel<ET, R, S, PRO, true, true><<<grid, 256, lds, st>>>(g); \
        else if (vec) gemv_float_kernel<ET, R, S, PRO, true, false><<<grid, 256, lds, st>>>(g);    \
        else gemv_float_kernel<ET, R, S, PRO, false, false><<<grid, 256, lds, st>>>(g);            \
    } while (0)
    if (pro == 0) FX_GEMV(0);
    if constexpr (S <= 4) {                               // longer rows: gemv_float asks for the plain linear only
        if (pro == 1) FX_GEMV(1);
        if (pro == 2) FX_GEMV(2);
    }
#undef FX_GEMV
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// The same linear for TT tokens at a time (prologue 0): a piece of a weight row in registers meets the TT vectors in LDS, so the
// weights are read once per TT tokens instead of once per token.  A thread's floats of the vectors lie in planes of 4 (one for
// float32, two for bfloat16 pieces of 8), so that neighbouring lanes read neighbouring 16 bytes.
template <typename ET, int TT, int R, int S>
__global__ __launch_bounds__(256) void gemv_tokens_kernel(GemvArgs g, int tokens) {
    constexpr int CE = Chunk<ET>::N, PL = CE / 4;
    constexpr int SUMS = R * TT <= 4 ? 4 : R * TT <= 8 ? 8 : R * TT <= 16 ? 16 : 32;
    static_assert(R * TT <= 32, "sums per lane");
    extern __shared__ __attribute__((aligned(16))) float xs[];     // [TT][PL][nchunk + 1][4], the last piece zeros for threads without one
    __shared__ float red[2][4 * SUMS];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, tok0 = blockIdx.y * TT;
    const ET* w = static_cast<const ET*>(g.w);
    const int nchunk = g.kpad / CE, ng = (g.n + R - 1) / R, G = gridDim.x;
    // the vectors first: loads return in order, and the weights behind them are a long stream
    const bool vec = (g.k & 3) == 0 && (g.ldx & 3) == 0;
#pragma unroll
    for (int j = 0; j < TT; j++) {
        const float* x = g.x + (size_t)min(tok0 + j, tokens - 1) * g.ldx;
        for (int c = t; c < g.kpad / 4; c += 256) {
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (vec) {
                if (4 * c < g.k) v = *reinterpret_cast<const f32x4*>(x + 4 * c);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = 4 * c + e < g.k ? x[4 * c + e] : 0.0f;
            }
            *reinterpret_cast<f32x4*>(xs + ((size_t)(j * PL + c % PL) * (nchunk + 1) + c / PL) * 4) = v;
        }
    }
    if (t < TT * PL) *reinterpret_cast<f32x4*>(xs + ((size_t)t * (nchunk + 1) + nchunk) * 4) = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    i32x4 buf[2][R][S];
    auto piece = [&](int row, int c) { return *reinterpret_cast<const i32x4*>(w + (size_t)min(row, g.n - 1) * g.kpad + c * CE); };
    auto load = [&](int b, int grp) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int s = 0; s < S; s++) {
                const int c = s * 256 + t;
                buf[b][r][s] = c < nchunk ? piece(grp * R + r, c) : i32x4{0, 0, 0, 0};
            }
    };
    const int g0 = blockIdx.x;
    load(0, g0);
    if (g0 + G < ng) load(1, g0 + G);
    __syncthreads();
    // piece c of R rows (u[.][s]) meets the vectors' piece c
    auto take = [&](const i32x4 (&u)[R][S], int s, int c, float (&acc)[SUMS]) {
        float wv[R][CE];
#pragma unroll
        for (int r = 0; r < R; r++) Chunk<ET>::unpack(make_uint4(u[r][s][0], u[r][s][1], u[r][s][2], u[r][s][3]), wv[r]);
#pragma unroll
        for (int j = 0; j < TT; j++)
#pragma unroll
            for (int q = 0; q < PL; q++) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(xs + ((j * PL + q) * (nchunk + 1) + c) * 4);
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[r * TT + j] = fma_f(wv[r][q * 4 + e], v[e], acc[r * TT + j]);
            }
    };
    auto process = [&](int b, int grp) {
        float acc[SUMS];
#pragma unroll
        for (int i = 0; i < SUMS; i++) acc[i] = 0.0f;
#pragma unroll
        for (int s = 0; s < S; s++) take(buf[b], s, min(s * 256 + t, nchunk), acc);     // pieces beyond the row meet the zeros
        for (int c = S * 256 + t; c < nchunk; c += 256) {
            i32x4 more[R][S];
#pragma unroll
            for (int r = 0; r < R; r++) more[r][0] = piece(grp * R + r, c);
            take(more, 0, c, acc);
        }
        multi_sum_step<SUMS, 1>(acc, lane);
        if (lane < SUMS) red[b][wave * SUMS + multi_row<SUMS>(lane)] = acc[0];
        __syncthreads();                                  // red alternates with the buffer: one barrier per group is enough
        const int r = t / TT, j = t - r * TT, row = grp * R + r, tok = tok0 + j;
        if (t < R * TT && row < g.n && tok < tokens) {
            auto total = [&](int i) {
                const float* p = red[b] + min(r + i, R - 1) * TT + j;
                const float v = (p[0] + p[SUMS]) + (p[2 * SUMS] + p[3 * SUMS]);
                return g.bias ? v + g.bias[min(row + i, g.n - 1)] : v;
            };
            if (row >= g.n_split) g.out32[(size_t)tok * g.ldo32 + row - g.n_split] = total(0);
            else if (!g.glu) g.out[(size_t)tok * g.ldo + row] = total(0);
            else if ((row & 1) == 0) g.out[(size_t)tok * g.ldo + (row >> 1)] = glu_f(g.glu, total(0), total(1), g.limit);
        }
    };
    for (int grp = g0; grp < ng; grp += 2 * G) {
        process(0, grp);
        if (grp + 2 * G < ng) load(0, grp + 2 * G);
        if (grp + G < ng) {
            process(1, grp + G);
            if (grp + 3 * G < ng) load(1, grp + 3 * G);
        }
    }
}

template <typename ET, int TT, int R, int S>
static int launch_gemv_tokens(const GemvArgs& g, int tokens, hipStream_t st) {
    const size_t lds = (size_t)TT * (g.kpad + Chunk<ET>::N) * sizeof(float);
    static std::atomic<bool> opted_in{false};
    if (!opted_in.load(std::memory_order_acquire)) {
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemv_tokens_kernel<ET, TT, R, S>), hipFuncAttributeMaxDynamicSharedMemorySize, kGemvTokensLds));
        opted_in.store(true, std::memory_order_release);
    }
    const int groups = (tokens + TT - 1) / TT, per_cu = lds <= 37 * 1024 ? 4 : lds <= 73 * 1024 ? 2 : 1, ng = (g.n + R - 1) / R;
    const int wgs = 256 * per_cu / groups;                // what is resident at a time
    gemv_tokens_kernel<ET, TT, R, S><<<dim3(ng < wgs ? ng : wgs, groups), 256, lds, st>>>(g, tokens);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// R x S pieces per thread and group as for one token, TT as many tokens as LDS holds.
template <typename ET, int R, int S>
static int gemv_tokens_rs(const GemvArgs& g, int tokens, hipStream_t st) {
    const int fit = (int)(kGemvTokensLds / ((g.kpad + Chunk<ET>::N) * sizeof(float))), most = fit < 32 / R ? fit : 32 / R;
    const int cap = most >= 8 ? 8 : most >= 6 ? 6 : most >= 4 ? 4 : 2, groups = (tokens + cap - 1) / cap, tt = (tokens + groups - 1) / groups;
    // rows that the others are called with are too long for eight vectors
    if constexpr (std::is_same<ET, float>::value && R > 1) if (tt > 6) return launch_gemv_tokens<ET, 8, R, S>(g, tokens, st);
    if (tt > 4) return launch_gemv_tokens<ET, 6, R, S>(g, tokens, st);
    if (tt > 2) return launch_gemv_tokens<ET, 4, R, S>(g, tokens, st);
    return launch_gemv_tokens<ET, 2, R, S>(g, tokens, st);
}

template <typename ET>
static int gemv_tokens(const GemvArgs& g, int tokens, hipStream_t st) {
    const int per = 256 * Chunk<ET>::N, steps = (g.kpad + per - 1) / per;
    if constexpr (std::is_same<ET, float>::value) {       // bfloat16: beyond what gemv_mfma_kernel takes, more than two pieces
        if (steps == 1) return gemv_tokens_rs<ET, 4, 1>(g, tokens, st);
        if (steps == 2) return gemv_tokens_rs<ET, 2, 2>(g, tokens, st);
    }
    if (steps <= 4 || g.glu) return gemv_tokens_rs<ET, 2, 4>(g, tokens, st);      // a pair of the gated unit lies in one group
    return gemv_tokens_rs<ET, 1, 8>(g, tokens, st);
}

// bfloat16 weights on the matrix cores: a float32 vector is the sum of three bfloat16 parts to 24 bits and their products with the
// weights are exact in float32, so two instructions per 16 rows x 32 k (at most 8 tokens: two parts lie side by side) give what the float32 products give (vector
// instructions: 16384 x 2048 for 5 tokens 24 us, the weights' stream is 10).  A workgroup of eight waves walks tiles of 16 rows; the
// waves share a unit of UK of k, of which a tile has UNITS, and meet through LDS per tile.
// What bounds it: the weights' stream, and that hangs on how it is asked for.  The operand of the instruction is 64 bytes of each of 16 rows; asked
// for like that, 67 MB take 17.5 us without any arithmetic, as 1 KiB of one row per request 11.5.  So the weights go to LDS in
// such requests (16-byte chunk c of row r at place c ^ r, for reads without conflicts), two units of 64 KiB of them in flight, and a
// unit's place is free for the next but one as soon as its operands are in registers.  The vectors' parts stay in registers, each wave's
// own stretch of k.
// Before (operands straight from memory) and now, 5 tokens, us: 16384 x 2048 21.5 and 14.4, 2048 x 8192 13.2 and 9.3, 28672 x 4096 49.8 and
// 39.6 (8 tokens 81 and 44), 4096 x 14336 28.0 and 21.0.
// ONE: where a workgroup has one tile of one unit there is no stream, only a chain of trips, and the weights come to registers in the operands' own
// shape: asked for together with the vectors they are a trip less than through LDS.  us, 5 tokens, before the stream through LDS, on it, now: 2048 x 2048 7.2, 6.7,
// 5.9, in two parts 5.3, 5.7, 4.8; 4096 x 2048 8.0, 7.5, 6.8; 1024 x 1024 4.9, 5.1, 4.5; 4000 x 1088 6.4, 6.6, 6.1; 4096 x 256 4.2, 5.1, 4.5 (what is left there is
// that each wave takes its vectors apart by itself, and at k of 256 two of eight have any).
constexpr int kMfmaTokens = 8, kMfmaWaves = 8;
template <int UK, int UNITS, bool ONE>
__global__ __launch_bounds__(kMfmaWaves * 64, 2) void gemv_mfma_kernel(GemvArgs g, int tokens, int group) {
    static_assert(!ONE || UNITS == 1, "ONE: a workgroup has one tile of one unit at most");
    arguments(g.w, g.x, g.n, g.k, g.kpad, g.ldx, g.parts, tokens, group, gridDim.x);
    constexpr int STRETCH = UK * UNITS, SW = UK / kMfmaWaves / 32, SL = UK / kMfmaWaves;      // matrix k-steps and k of a wave in a unit
    constexpr int UB = UK * 2, SLOT = 16 * UB, SLOTS = ONE ? 1 : 128 * 1024 / SLOT, PER = SLOT / 1024 / kMfmaWaves;   // PER: requests of a wave per unit
    static_assert(kMfmaTokens * SL * 4 <= PER * 1024, "a wave's vectors fit into its part of a unit's place");
    extern __shared__ __attribute__((aligned(16))) int8_t ring[];
    __shared__ float red[2][kMfmaWaves][16 * 17];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int part = blockIdx.x % g.parts, walker = blockIdx.x / g.parts, walkers = gridDim.x / g.parts;
    const int tok0 = blockIdx.y * group, nt = min(group, tokens - tok0), k0 = part * STRETCH, tiles = (g.n + 15) / 16;
    const int mine = (tiles - walker + walkers - 1) / walkers, total = mine * UNITS;          // tiles and units of this workgroup
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)ring;
    auto request_unit = [&](int u) __attribute__((always_inline)) {
        const int tile = walker + u / UNITS * walkers, h = u % UNITS, last = min(16, g.n - tile * 16) - 1;
        const int8_t* base = static_cast<const int8_t*>(g.w) + (size_t)tile * 16 * g.kpad * 2;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int p = wave * PER + q, r = p / (UB / 1024), seg = p % (UB / 1024);
            // what is behind the row's end (any of its bytes will do) meets zeros
            const int kb = min((k0 + h * UK) * 2 + seg * 1024 + (lane ^ r) * 16, g.kpad * 2 - 16);
            load_to_lds<true>(base, (unsigned)(min(r, last) * g.kpad * 2 + kb), lds0 + (u % SLOTS) * SLOT + p * 1024);      // the vectors are read by every workgroup
        }
    };
    // a wave's vectors [token][SL], in the last place's part that only this wave's requests write
    int8_t* const xs = ring + (SLOTS - 1) * SLOT + wave * (PER * 1024);
    constexpr int XC = SL / 4, XN = kMfmaTokens * XC / 64;    // 16-byte chunks of a token, and of a lane
    const bool vec = (g.k & 3) == 0 && (g.ldx & 3) == 0 && (reinterpret_cast<uintptr_t>(g.x) & 15) == 0;
    auto request_vectors = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XN; i++) {
            const int c = i * 64 + lane, j = min(c / XC, nt - 1), k = k0 + h * UK + wave * SL + c % XC * 4;
            if (i * 64 < nt * XC) load_to_lds(g.x + (size_t)tok0 * g.ldx, (unsigned)(j * g.ldx + min(k, g.k - 4)) * 4u, lds0 + (unsigned)(xs - ring) + i * 1024);
        }
    };
    // The instruction has 16 columns for at most 8 tokens: columns 0 to 7 are the tokens' first and third part, 8 to 15 their second.
    bf16x8 xf[UNITS * SW][2];
    const int j0 = min(lane & 7, nt - 1), second = (lane >> 3) & 1, gq = lane >> 4;
    constexpr int JI = 64 / XC;                               // tokens that a round of the wave's lanes covers
    const int put0 = ((((lane % XC) >> 1) ^ (lane / XC)) << 4) + (lane & 1) * 8 + lane / XC * (SL * 2), row0 = second * kMfmaTokens + j0;
    const int8_t* const get0 = xs + row0 * (SL * 2);
    bf16x8 direct[ONE ? SW : 1];
    auto take_vectors = [&](int h) __attribute__((always_inline)) {
        const int first = k0 + h * UK + wave * SL;            // k of the wave's stretch
        f32x4 v[XN];
        auto row_of = [&](int i) __attribute__((always_inline)) { return g.x + (size_t)(tok0 + min(i * JI + lane / XC, nt - 1)) * g.ldx; };
        if (vec) {
#pragma unroll
            for (int i = 0; i < XN; i++) {
                if (i * JI >= nt) break;
                v[i] = ONE ? *reinterpret_cast<const f32x4*>(row_of(i) + min(first + lane % XC * 4, g.k - 4)) : *reinterpret_cast<const f32x4*>(xs + (i * 64 + lane) * 16);
            }
        } else {
#pragma unroll
            for (int i = 0; i < XN; i++) {
                if (i * JI >= nt) break;
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = row_of(i)[min(first + lane % XC * 4 + e, g.k - 1)];
            }
        }
        if constexpr (ONE) {
            const bf16_t* row = static_cast<const bf16_t*>(g.w) + (size_t)min(walker * 16 + (lane & 15), g.n - 1) * g.kpad;
#pragma unroll
            for (int s = 0; s < SW; s++) direct[s] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(row + min(first + s * 32 + gq * 8, g.kpad - 8)));
            __builtin_amdgcn_sched_barrier(0);
        }
        if (first + SL > g.k) {
#pragma unroll
            for (int i = 0; i < XN; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = first + lane % XC * 4 + e < g.k ? v[i][e] : 0.0f;
        }
        // A part is the upper half of the bits, so three of them are the value and none rounds up to infinity.  What is left of an infinity
        // is not a number, which makes the sums such (see `whole`).  Parts lie as [2][token][SL], chunk c of 16 bytes at place c ^ row:
        // the 16 columns of an operand read are on different banks.
        auto put = [&](int i, int to) __attribute__((always_inline)) {
            const int row = to * kMfmaTokens + i * JI;
            uint2 o;
            o.x = __builtin_amdgcn_perm(__float_as_uint(v[i][1]), __float_as_uint(v[i][0]), 0x07060302u);
            o.y = __builtin_amdgcn_perm(__float_as_uint(v[i][3]), __float_as_uint(v[i][2]), 0x07060302u);
            *reinterpret_cast<uint2*>(xs + (put0 ^ (row << 4)) + row * (SL * 2)) = o;
#pragma unroll
            for (int e = 0; e < 4; e++) v[i][e] -= __uint_as_float(__float_as_uint(v[i][e]) & 0xFFFF0000u);
        };
        auto get = [&](int s) { return *reinterpret_cast<const bf16x8*>(get0 + (((s * 4 + gq) ^ row0) << 4)); };
#pragma unroll
        for (int i = 0; i < XN; i++) {
            if (i * JI >= nt) break;
            put(i, 0);
            put(i, 1);
        }
#pragma unroll
        for (int s = 0; s < SW; s++) xf[h * SW + s][0] = get(s);
#pragma unroll
        for (int i = 0; i < XN; i++) {
            if (i * JI >= nt) break;
            put(i, 0);
        }
        const uint32_t keep = second ? 0u : ~0u;
#pragma unroll
        for (int s = 0; s < SW; s++) {
            i32x4 b = __builtin_bit_cast(i32x4, get(s));
#pragma unroll
            for (int e = 0; e < 4; e++) b[e] &= keep;
            xf[h * SW + s][1] = __builtin_bit_cast(bf16x8, b);
        }
    };
    auto all_read = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    if constexpr (ONE) {
        take_vectors(0);
    } else {
        if (vec) request_vectors(0);
#pragma unroll
        for (int u = 0; u < SLOTS - 1; u++)
            if (u < total) request_unit(u);
        if (vec) {
            if (total >= SLOTS - 1) wait_vmcnt<(SLOTS - 1) * PER>();
            else if (total == 2) wait_vmcnt<2 * PER>();
            else wait_vmcnt<PER>();
        }
        take_vectors(0);
        if constexpr (UNITS == 2) {
            all_read();
            if (vec) { request_vectors(1); wait_vmcnt<0>(); }
            take_vectors(1);
        }
        all_read();
        if (SLOTS - 1 < total) request_unit(SLOTS - 1);
    }
    // Not a number may be of the parts' own making, where an infinite weight meets parts of zero or of both signs (or, behind the row's
    // end, zeros) or a value is infinite: the same sum with a float32 product per weight has the right of it.
    auto whole = [&](int row, int j) __attribute__((always_inline)) {
        const bf16_t* wr = static_cast<const bf16_t*>(g.w) + (size_t)row * g.kpad;
        const float* x = g.x + (size_t)(tok0 + j) * g.ldx;
        float s = 0.0f;
        for (int k = k0; k < min(k0 + STRETCH, g.k); k++) s = fma_f((float)wr[k], x[k], s);
        return s;
    };
    auto finish = [&](int i) __attribute__((always_inline)) {
        const int r = t & 15, j = t >> 4, row = (walker + i * walkers) * 16 + r, tok = tok0 + j;
        if (j < nt && row < g.n) {
            auto sum = [&](int o) {
                const float* p = red[i & 1][0] + (r + o) * 17 + j;
                float v[kMfmaWaves];
#pragma unroll
                for (int q = 0; q < kMfmaWaves; q++) v[q] = p[q * 16 * 17] + p[q * 16 * 17 + 8];
                float s = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
                if (isnan(s)) s = whole(min(row + o, g.n - 1), j);
                return g.bias ? s + g.bias[min(row + o, g.n - 1)] : s;
            };
            if (row >= g.n_split) g.out32[part * g.part_stride + (size_t)tok * g.ldo32 + row - g.n_split] = sum(0);
            else if (!g.glu) g.out[(size_t)tok * g.ldo + row] = sum(0);
            else if ((row & 1) == 0) g.out[(size_t)tok * g.ldo + (row >> 1)] = glu_f(g.glu, sum(0), sum(1), g.limit);
        }
    };
    if constexpr (ONE) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < SW; s++)
#pragma unroll
            for (int p = 1; p >= 0; p--) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(direct[s], xf[s][p], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) red[0][wave][(gq * 4 + e) * 17 + (lane & 15)] = acc[e];
        __syncthreads();
        return finish(0);
    }
    const int8_t* const mine_in = ring + (lane & 15) * UB;
    for (int i = 0; i < mine; i++) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int h = 0; h < UNITS; h++) {
            const int u = i * UNITS + h, younger = total - 1 - u;
            if (younger >= SLOTS - 1) wait_vmcnt<(SLOTS - 1) * PER>();
            else if (SLOTS > 3 && younger == 2) wait_vmcnt<2 * PER>();
            else if (SLOTS > 2 && younger == 1) wait_vmcnt<PER>();
            else wait_vmcnt<0>();
            all_read();                                        // the last tile's sums have left
            barrier();
            bf16x8 wf[SW];
            const int8_t* in = mine_in + (u % SLOTS) * SLOT;
#pragma unroll
            for (int s = 0; s < SW; s++) {
                const int c = wave * (SL / 8) + s * 4 + gq;      // chunk of the row, in KiB of 64 chunks that are rotated each by itself
                wf[s] = *reinterpret_cast<const bf16x8*>(in + (c ^ (lane & 15)) * 16);
            }
            all_read();
            barrier();
            if (u + SLOTS < total) request_unit(u + SLOTS);
            if (h == 0 && i > 0) finish(i - 1);
#pragma unroll
            for (int s = 0; s < SW; s++)
#pragma unroll
                for (int p = 1; p >= 0; p--)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], xf[h * SW + s][p], acc, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) red[i & 1][wave][(gq * 4 + e) * 17 + (lane & 15)] = acc[e];
    }
    __syncthreads();
    finish(mine - 1);
}

template <int UK, int UNITS, bool ONE>
static int launch_gemv_mfma(const GemvArgs& g, int tokens, int walkers, int groups, hipStream_t st) {
    constexpr int lds = ONE ? UK * 32 : 128 * 1024;
    static std::atomic<bool> opted_in{false};
    if (!opted_in.load(std::memory_order_acquire)) {
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemv_mfma_kernel<UK, UNITS, ONE>), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        opted_in.store(true, std::memory_order_release);
    }
    gemv_mfma_kernel<UK, UNITS, ONE><<<dim3(walkers * g.parts, groups), kMfmaWaves * 64, lds, st>>>(g, tokens, (tokens + groups - 1) / groups);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}
static int gemv_mfma(const GemvArgs& g, int tokens, int stretch, hipStream_t st) {
    const int groups = (tokens + kMfmaTokens - 1) / kMfmaTokens, tiles = (g.n + 15) / 16;
    int walkers = 256 / (g.parts * groups);               // one workgroup per CU
    if (walkers < 1) walkers = 1;
    const bool one = tiles <= walkers;
    if (one) walkers = tiles;
    if (stretch <= 1024) return one ? launch_gemv_mfma<1024, 1, true>(g, tokens, walkers, groups, st) : launch_gemv_mfma<1024, 1, false>(g, tokens, walkers, groups, st);
    if (stretch <= 2048) return one ? launch_gemv_mfma<2048, 1, true>(g, tokens, walkers, groups, st) : launch_gemv_mfma<2048, 1, false>(g, tokens, walkers, groups, st);
    return launch_gemv_mfma<2048, 2, false>(g, tokens, walkers, groups, st);
}

// k of a workgroup: 1024, 2048 or 4096.  Parts of a product whose reader adds them: as few as that takes, one more doubling where the
// rows alone leave CUs without a tile (2048 x 2048).
template <>
int gemv_parts<bf16_t>(int n, int kpad, int most) {
    int parts = (kpad + 2047) / 2048;
    if (parts > most) return 1;
    if (parts * 2 <= most && kpad >= parts * 2048 && (n + 15) / 16 * parts < 256) parts *= 2;
    return parts;
}
template <>
int gemv_parts<float>(int, int, int) { return 1; }

template <typename ET>
int gemv_float(const GemvArgs& g, int pro, int tokens, hipStream_t st) {
    FX_REQUIRE(g.w && g.x && g.n > 0 && g.k > 0 && g.kpad >= g.k && g.kpad % kKPad == 0 && tokens > 0, "gemv_float: n=%d k=%d", g.n, g.k);
    FX_REQUIRE(g.kpad <= 15360, "gemv_float: k=%d beyond 15360 (the vector is held in LDS)", g.k);
    FX_REQUIRE(pro != 2 || (g.experts > 0 && g.experts <= kMaxExperts && g.top > 0 && g.top <= kMaxTop && g.top <= g.experts),
               "gemv_float: %d experts, top %d (at most %d, %d)", g.experts, g.top, kMaxExperts, kMaxTop);
    FX_REQUIRE(g.parts == 1 || (std::is_same<ET, bf16_t>::value && pro == 0 && tokens > 1 && g.n_split == 0 && !g.bias), "gemv_float: %d parts", g.parts);
    if (pro == 0 && tokens > 1 && !g.per_token) {
        if constexpr (std::is_same<ET, bf16_t>::value) {
            const int stretch = (g.kpad + g.parts - 1) / g.parts;
            if (stretch <= 4096) return gemv_mfma(g, tokens, stretch, st);
            FX_REQUIRE(g.parts == 1, "gemv_float: %d parts of k=%d", g.parts, g.k);
        }
        return gemv_tokens<ET>(g, tokens, st);
    }
    const int per = 256 * Chunk<ET>::N, steps = (g.kpad + per - 1) / per;
    // Rows per group: four pieces per thread and group where workgroups walk several groups (a group's sums and barrier then
    // overlap the next group's loads: 16384 x 2048 13.9 us with eight, 12.9 with four; 28672 x 4096 42.2 -> 37.7 us), eight
    // where a workgroup has a single group anyway (4096 x 4096: 7.65 us with eight, 7.96 with four) and for rows so long
    // that two rows are eight pieces (2048 x 8192: 8.2 us, 8.4 one row at a time; 4096 x 14336: 21.1 and 23.1).
    // Several tokens wait for the L2, with eight in flight again: of rows of two pieces always, of one piece from the third token on (four
    // tokens of 16 layers of 2048, bfloat16, half of them recurrences: 1349 us with eight, 1444 with four; two tokens 1058 and 1030).
    if (steps == 1 && pro != 2 && tokens > 2 && (g.n + 7) / 8 * tokens >= 512) return launch_gemv_rs<ET, 8, 1>(g, pro, tokens, st);
    if (steps == 1) return launch_gemv_rs<ET, 4, 1>(g, pro, tokens, st);
    if (steps == 2) return (g.n + 3) / 4 <= 1024 || tokens > 1 ? launch_gemv_rs<ET, 4, 2>(g, pro, tokens, st) : launch_gemv_rs<ET, 2, 2>(g, pro, tokens, st);
    if (steps > 4 && pro == 0) return launch_gemv_rs<ET, 2, 8>(g, pro, tokens, st);
    return launch_gemv_rs<ET, 2, 4>(g, pro, tokens, st);
}
template int gemv_float<bf16_t>(const GemvArgs&, int, int, hipStream_t);
template int gemv_float<float>(const GemvArgs&, int, int, hipStream_t);

// Down projections of the chosen experts and of the shared one, summed with their weights.  The sources lie one after
// the other in a list of 16-byte pieces, which the threads walk together; R = 4 output rows per workgroup.  The trips to
// memory bound it: a pick, the weights behind it, the sum.  So a thread requests B = 4 pieces of each row, and what they
// meet, before it takes the first one in.  Six experts of 2048 x 1024 and a shared one of 2048, one token, 33.5 MB: 12.4 us
// with one piece after the other, 9.6 us so (3.5 TB/s).  NT: one token, whose weights are read once; several tokens share
// them through the L2.
template <typename ET, bool NT>
__global__ __launch_bounds__(256) void moe_down_kernel(MoeDownArgs a) {
    constexpr int CE = Chunk<ET>::N, R = 4, B = 4;
    __shared__ float red[4 * R];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, tok = blockIdx.y, row0 = blockIdx.x * R;
    const int ce = a.kpad / CE, cs = a.ws ? a.ks_pad / CE : 0, total = a.top * ce + cs;
    const bool vec = ((a.k | a.ldh) & 3) == 0 && (!a.ws || ((a.ks | a.ldhs) & 3) == 0);
    float acc[R] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i0 = t; i0 < total; i0 += 256 * B) {
        i32x4 u[B][R];
        float x[B][CE], wt[B];
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int it = min(i0 + 256 * b, total - 1);
            const bool sh = it >= a.top * ce;
            const int slot = sh ? 0 : it / ce, c = sh ? it - a.top * ce : it - slot * ce, kp = sh ? a.ks_pad : a.kpad;
            const ET* w = sh ? static_cast<const ET*>(a.ws) : static_cast<const ET*>(a.w) + (size_t)a.pick[tok * a.top + slot] * a.w_stride;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const i32x4* p = reinterpret_cast<const i32x4*>(w + (size_t)min(row0 + r, a.n - 1) * kp + c * CE);
                if constexpr (NT) u[b][r] = __builtin_nontemporal_load(p);
                else u[b][r] = *p;
            }
        }
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int it = min(i0 + 256 * b, total - 1);
            const bool sh = it >= a.top * ce;
            const int slot = sh ? 0 : it / ce, c = sh ? it - a.top * ce : it - slot * ce, kk = sh ? a.ks : a.k;
            const float* h = sh ? a.hs + (size_t)tok * a.ldhs : a.h + (size_t)(tok * a.top + slot) * a.ldh;
            wt[b] = sh ? a.route[(size_t)tok * a.ld_route + a.experts] : a.pick_w[tok * a.top + slot];
            if (vec) {
#pragma unroll
                for (int q = 0; q < CE; q += 4) {
                    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                    if (c * CE + q < kk) v = *reinterpret_cast<const f32x4*>(h + c * CE + q);
#pragma unroll
                    for (int e = 0; e < 4; e++) x[b][q + e] = v[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < CE; e++) x[b][e] = c * CE + e < kk ? h[c * CE + e] : 0.0f;
            }
            if (sh) wt[b] = sigmoid_f(wt[b]);
        }
#pragma unroll
        for (int b = 0; b < B; b++) {
            if (i0 + 256 * b >= total) break;
#pragma unroll
            for (int r = 0; r < R; r++) {
                float wv[CE], s = 0.0f;
                Chunk<ET>::unpack(make_uint4(u[b][r][0], u[b][r][1], u[b][r][2], u[b][r][3]), wv);
#pragma unroll
                for (int e = 0; e < CE; e++) s = fma_f(wv[e], x[b][e], s);
                acc[r] = fma_f(wt[b], s, acc[r]);
            }
        }
    }
    multi_sum_step<R, 1>(acc, lane);
    if (lane < R) red[wave * R + multi_row<R>(lane)] = acc[0];
    __syncthreads();
    if (t < R && row0 + t < a.n)
        a.y[(size_t)tok * a.ldy + row0 + t] = (red[t] + red[R + t]) + (red[2 * R + t] + red[3 * R + t]);
}

template <typename ET>
int moe_down_small(const MoeDownArgs& a, int tokens, hipStream_t st) {
    FX_REQUIRE(a.w && a.h && a.pick && a.pick_w && a.y && a.n > 0 && tokens > 0, "moe_down: null pointer");
    const dim3 grid((a.n + 3) / 4, tokens);
    if (tokens == 1) moe_down_kernel<ET, true><<<grid, 256, 0, st>>>(a);
    else moe_down_kernel<ET, false><<<grid, 256, 0, st>>>(a);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}
template int moe_down_small<bf16_t>(const MoeDownArgs&, int, hipStream_t);
template int moe_down_small<float>(const MoeDownArgs&, int, hipStream_t);

// ---- the plan of a mixture over many rows --------------------------------------------------------------------------
static __global__ __launch_bounds__(256) void moe_clear_kernel(int* counts, int n) {
    for (int i = threadIdx.x; i < n; i += 256) counts[i] = 0;
}
constexpr int kPlanT = 1024, kRouteRows = 32;              // rows per workgroup of the route kernel
static __global__ __launch_bounds__(kPlanT) void moe_route_kernel(const float* __restrict__ route, int ld, int rows, int experts, int top,
                                                                  int* __restrict__ pick, float* __restrict__ pick_w, int* __restrict__ counts) {
    __shared__ int hist[kMaxExperts];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    for (int e = t; e < experts; e += kPlanT) hist[e] = 0;
    __syncthreads();
    for (int i = 0; i < kRouteRows / (kPlanT / 64); i++) {
        const int row = blockIdx.x * kRouteRows + i * (kPlanT / 64) + wave;
        if (row >= rows) break;
        int e;
        float w;
        route_wave(route + (size_t)row * ld, experts, top, e, w);
        if (lane < top) {
            pick[row * top + lane] = e;
            pick_w[row * top + lane] = w;
            atomicAdd(&hist[e], 1);
        }
    }
    __syncthreads();
    for (int e = t; e < experts; e += kPlanT)
        if (hist[e]) atomicAdd(&counts[e], hist[e]);
}
// Place every (row, choice) in its expert's run: a workgroup reserves room for its entries with one atomic per expert.
// Workgroup 0 also cuts the runs into tiles.
static __global__ __launch_bounds__(kPlanT) void moe_place_kernel(int rows, int experts, int top, int tile_rows, const int* __restrict__ pick,
                                                                  int* __restrict__ counts, int* __restrict__ pos_of, int* __restrict__ row_src,
                                                                  int4* __restrict__ tiles, int* __restrict__ n_tiles) {
    __shared__ int first[kMaxExperts], tile0[kMaxExperts], hist[kMaxExperts];
    __shared__ int part[kPlanT], part_t[kPlanT];
    const int t = threadIdx.x;
    static_assert(kPlanT >= kMaxExperts, "one thread per expert");
    const int n = t < experts ? counts[t] : 0, nt = (n + tile_rows - 1) / tile_rows;
    part[t] = n; part_t[t] = nt;
    if (t < experts) hist[t] = 0;
    __syncthreads();
    for (int m = 1; m < kPlanT; m <<= 1) {                // inclusive scan
        const int a = t >= m ? part[t - m] : 0, b = t >= m ? part_t[t - m] : 0;
        __syncthreads();
        part[t] += a; part_t[t] += b;
        __syncthreads();
    }
    const int idx = blockIdx.x * kPlanT + t, e = idx < rows * top ? pick[idx] : -1;
    const int local = e >= 0 ? atomicAdd(&hist[e], 1) : 0;
    if (t < experts) tile0[t] = part_t[t] - nt;
    __syncthreads();
    if (t < experts) first[t] = part[t] - n + (hist[t] ? atomicAdd(&counts[experts + t], hist[t]) : 0);
    __syncthreads();
    if (e >= 0) {
        const int pos = first[e] + local;
        pos_of[idx] = pos;
        row_src[pos] = idx / top;
    }
    if (blockIdx.x == 0) {
        if (t < experts)
            for (int i = 0; i < nt; i++) tiles[tile0[t] + i] = make_int4(t, part[t] - n + i * tile_rows, part[t] - n + min(n, (i + 1) * tile_rows), 0);
        if (t == 0) n_tiles[0] = part_t[kPlanT - 1];
    }
}

int moe_plan(const float* route, int ld_route, int rows, int experts, int top, int tile_rows, const MoePlan& p, hipStream_t st) {
    FX_REQUIRE(experts > 0 && experts <= kMaxExperts && top > 0 && top <= kMaxTop && top <= experts, "moe_plan: %d experts, top %d (at most %d, %d)",
               experts, top, kMaxExperts, kMaxTop);
    moe_clear_kernel<<<1, 256, 0, st>>>(p.counts, 2 * experts);
    moe_route_kernel<<<(rows + kRouteRows - 1) / kRouteRows, kPlanT, 0, st>>>(route, ld_route, rows, experts, top, p.pick, p.pick_w, p.counts);
    moe_place_kernel<<<(rows * top + kPlanT - 1) / kPlanT, kPlanT, 0, st>>>(rows, experts, top, tile_rows, p.pick, p.counts, p.pos_of, p.row_src, p.tiles, p.n_tiles);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

}  // namespace fx

using namespace fx;

extern "C" {

int flexllm_linear_float_step(const float* x, const void* w, const float* bias, float* y, float* y32, int tokens, int k, int n, int n_split, int glu, float limit,
                              int parts, int dtype, void* stream) {
    FX_REQUIRE((dtype == 0 || dtype == 1) && glu >= 0 && glu <= 1 + FLEXLLM_GLU_GELU, "linear_float_step: dtype=%d glu=%d", dtype, glu);
    FX_REQUIRE(tokens > 0 && tokens <= 8 && k > 0 && n > 0 && n_split >= 0 && n_split <= n && (n_split == 0 || y) && (n_split == n || y32) && (!glu || n_split % 2 == 0),
               "linear_float_step: tokens=%d k=%d n=%d n_split=%d", tokens, k, n, n_split);
    FX_REQUIRE(parts >= 1 && parts <= 8 && (size_t)x % 16 == 0 && (size_t)w % 16 == 0, "linear_float_step: %d parts, or an operand off 16 bytes", parts);
    GemvArgs g;
    g.w = w; g.n = n; g.k = k; g.kpad = pad_k(k); g.x = x; g.ldx = k; g.bias = bias;
    g.out = y; g.ldo = glu ? n_split / 2 : n_split; g.out32 = y32; g.ldo32 = n - n_split; g.n_split = n_split; g.glu = glu; g.limit = limit;
    g.parts = parts; g.part_stride = (size_t)tokens * n;
    return dtype == 0 ? gemv_float<bf16_t>(g, 0, tokens, as_stream(stream)) : gemv_float<float>(g, 0, tokens, as_stream(stream));
}

}  // extern "C"
