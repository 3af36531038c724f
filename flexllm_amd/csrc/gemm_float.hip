// Floating-point GEMMs for prefill: C[m][n] = sum_k A[m][k] * W[n][k], both operands K-contiguous, on the walk of gemm_walk.h.
// Rows of A may be gathered, groups of rows may have a weight matrix each (experts), the epilogue adds a bias, splits the columns
// between an ET and a float32 output and applies the gated unit to interleaved gate/up columns.
#include <atomic>
#include "float_ops.h"
#include "gemm_walk.h"
#include "gemm_few.h"

namespace fx {

// One row's four consecutive columns col..col+3.
template <typename ET>
__device__ __forceinline__ void gemm_store4(const GemmArgs& g, int row, int col, float (&v)[4], bool vec) {
    ET* y = static_cast<ET*>(g.y);
    if (vec) {
        if (col >= g.n) return;
        if (col >= g.n_split) {
            *reinterpret_cast<float4*>(g.y32 + (size_t)row * g.ldy32 + (col - g.n_split)) = make_float4(v[0], v[1], v[2], v[3]);
        } else if (g.glu) {
            ET* d = y + (size_t)row * g.ldy + (col >> 1);
            d[0] = (ET)glu_f(g.glu, v[0], v[1], g.limit);
            d[1] = (ET)glu_f(g.glu, v[2], v[3], g.limit);
        } else if constexpr (std::is_same<ET, float>::value) {
            *reinterpret_cast<float4*>(y + (size_t)row * g.ldy + col) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (bf16_t)v[e];
            *reinterpret_cast<bf16x4*>(y + (size_t)row * g.ldy + col) = o;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int c = col + e;
        if (c >= g.n) return;
        if (c >= g.n_split) g.y32[(size_t)row * g.ldy32 + (c - g.n_split)] = v[e];
        else if (!g.glu) y[(size_t)row * g.ldy + c] = (ET)v[e];
        else if ((c & 1) == 0) y[(size_t)row * g.ldy + (c >> 1)] = (ET)glu_f(g.glu, v[e], v[(e + 1) & 3], g.limit);
    }
}

// How the outputs of a product may leave.  kWide: columns below n_split, or those from there on, in whole 16-byte pieces (rows and outputs
// start on such a border); kQuad: four columns never straddle the split and every store address is a multiple of the store's size;
// kSingle: one by one.
enum GemmStores { kSingle = 0, kQuad = 1, kWide = 2 };

// A wave's outputs that all lie on one side of the split: J blocks of 16 columns at a time become 64 consecutive bytes of a row, 16 per
// lane (GLU: the unit, 0: none; OT: type of the outputs).
// cols: those that there are from the wave's first one on, a multiple of what 16 bytes of output are made of.
template <typename OT, class W, int GLU, bool BIAS>
__device__ __forceinline__ void gemm_out_wide(OT* y, int ldy, const float* bias, float limit, int row0, int row_end, int cols, f32x4 (&acc)[W::MIv][W::NIv]) {
    constexpr int R = (int)sizeof(OT) / (GLU ? 2 : 1), J = 4 / R, NI = W::NIv, MI = W::MIv;   // R: words of a lane's four columns
    const int lane = threadIdx.x & 63, row_bytes = ldy * (int)sizeof(OT);
    const TileRows out(y + (size_t)row0 * ldy, row_end - row0, MI * 16, row_bytes);
    const int at = (lane & 15) * row_bytes + (lane >> 4) * 16;
#pragma unroll
    for (int j0 = 0; j0 < NI; j0 += J) {
        f32x4 b[J];
        if constexpr (BIAS) {
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) b[j][e] = bias[min((j0 + j) * 16 + (lane >> 4) * 4 + e, cols - 1)];
        }
        const bool there = j0 * 16 + (lane >> 4) * (4 * J) < cols;
#pragma unroll
        for (int i = 0; i < MI; i++) {
            uint32_t w[J][R];
#pragma unroll
            for (int j = 0; j < J; j++) {
                f32x4 v = acc[i][j0 + j];
                if constexpr (BIAS) v += b[j];
                else asm volatile("" : "+v"(v));                  // out of the accumulation registers here, a block at a time
                OT o[GLU ? 2 : 4];
                if constexpr (GLU != 0) {
                    o[0] = (OT)glu_f(GLU, v[0], v[1], limit);
                    o[1] = (OT)glu_f(GLU, v[2], v[3], limit);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) o[e] = (OT)v[e];
                }
                __builtin_memcpy(w[j], o, sizeof(o));
            }
            join_blocks<R>(w);
            out.put(&w[0][0], there ? at + i * 16 * row_bytes + j0 * 16 * (int)sizeof(OT) / (GLU ? 2 : 1) : kNowhere);
            __builtin_amdgcn_sched_barrier(0);                 // one piece after the other: all at once are more than the registers hold
        }
    }
}

// Outputs of any form: up to 64 columns of the wave's rows at a time turn through LDS, so that a loop can take them and lanes side by side store what
// is side by side.  (Before, a loop of a lane's own four columns: sixteen rows per store.)
template <typename ET, class W>
__device__ __forceinline__ void gemm_out_loose(const GemmArgs& g, int row0, int row_end, int col0, int stores, int8_t* smem, f32x4 (&acc)[W::MIv][W::NIv]) {
    constexpr int MI = W::MIv, NI = W::NIv, J = NI < 4 || 4 * MI * 16 * 68 * 4 > W::kLds ? 2 : 4, C = J * 16, P = C + 4;      // P: of 16 rows no two begin on the same banks
    static_assert(NI % J == 0 && 4 * MI * 16 * P * 4 <= W::kLds, "a patch per wave");
    const int lane = threadIdx.x & 63, fg = lane >> 4, fr = lane & 15, rows = min(MI * 16, row_end - row0);
    __syncthreads();                                           // the walk has left LDS behind in this wave alone
    float* const patch = reinterpret_cast<float*>(smem) + W::wave() * (MI * 16 * P);
    auto settled = []() __attribute__((always_inline)) {       // a wave's own LDS operations complete in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
#pragma unroll
    for (int j0 = 0; j0 < NI; j0 += J) {
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int i = 0; i < MI; i++) *reinterpret_cast<f32x4*>(patch + (i * 16 + fr) * P + j * 16 + fg * 4) = acc[i][j0 + j];
        settled();
        if (stores == kSingle && !g.glu) {
            constexpr int R = 64 / C;
            const int c = lane % C, col = col0 + j0 * 16 + c;
            const float b = g.bias ? g.bias[min(col, g.n - 1)] : 0.0f;
            auto each = [&](auto* to, int ld) __attribute__((always_inline)) {
#pragma unroll 4
                for (int r = lane / C; r < rows; r += R) {
                    float v = patch[r * P + c];
                    if (g.bias) v += b;
                    to[(size_t)r * ld] = v;
                }
            };
            if (col < g.n_split) each(static_cast<ET*>(g.y) + (size_t)row0 * g.ldy + col, g.ldy);
            else if (col < g.n) each(g.y32 + (size_t)row0 * g.ldy32 + (col - g.n_split), g.ldy32);
        } else {
            constexpr int L = C / 4, R = 64 / L;
            const int c = lane % L * 4, col = col0 + j0 * 16 + c;
            f32x4 b = {0.0f, 0.0f, 0.0f, 0.0f};
            if (g.bias)
#pragma unroll
                for (int e = 0; e < 4; e++) b[e] = g.bias[min(col + e, g.n - 1)];
#pragma unroll 2
            for (int r = lane / L; r < rows; r += R) {
                f32x4 q = *reinterpret_cast<const f32x4*>(patch + r * P + c);
                if (g.bias) q += b;
                float v[4] = {q[0], q[1], q[2], q[3]};
                gemm_store4<ET>(g, row0 + r, col, v, stores != kSingle);
            }
        }
        settled();
    }
}

// OUT: forms of the outputs that a kernel of tiles of 256 columns is made for (all of them in one are more than its registers hold beside the
// sums, and spilled sums have come back wrong: the build refuses such kernels).  kOutAny: all, at run time; kOutLoose: what does not leave in
// whole 16-byte pieces.
enum GemmOut { kOutAny = 0, kOutPlain = 1, kOutBias = 2, kOutClamped = 3, kOutGelu = 4, kOutLoose = 5 };
template <typename ET, class W, int OUT>
__device__ __forceinline__ void gemm_out(const GemmArgs& g, int row0, int row_end, int col0, int stores, int8_t* smem, f32x4 (&acc)[W::MIv][W::NIv]) {
    constexpr int NI = W::NIv, J = std::is_same<ET, float>::value ? 2 : 4;
    const int end = col0 + NI * 16;
    const float* bias = g.bias + col0;
    ET* const y = static_cast<ET*>(g.y);
    float* const y32 = g.y32 + (col0 - g.n_split);
    const int cols = g.n_split - col0, cols32 = g.n - col0;
    if constexpr (OUT == kOutClamped || OUT == kOutGelu) {
        return gemm_out_wide<ET, W, OUT == kOutGelu ? kGluGelu : kGluClamped, false>(y + (col0 >> 1), g.ldy, nullptr, g.limit, row0, row_end, cols, acc);
    } else if constexpr (OUT == kOutPlain || OUT == kOutBias) {
        if (col0 >= g.n_split) gemm_out_wide<float, W, 0, OUT == kOutBias>(y32, g.ldy32, bias, 0.0f, row0, row_end, cols32, acc);
        else gemm_out_wide<ET, W, 0, OUT == kOutBias>(y + col0, g.ldy, bias, 0.0f, row0, row_end, cols, acc);
        return;
    } else if constexpr (OUT == kOutAny) {
        if (stores == kWide && col0 >= g.n_split) {
            if (g.bias) return gemm_out_wide<float, W, 0, true>(y32, g.ldy32, bias, 0.0f, row0, row_end, cols32, acc);
            return gemm_out_wide<float, W, 0, false>(y32, g.ldy32, bias, 0.0f, row0, row_end, cols32, acc);
        }
        if constexpr (NI % J == 0) {
            if (stores == kWide && (end <= g.n_split || g.n_split == g.n) && !(g.bias && g.glu)) {
                if (g.glu == kGluClamped) return gemm_out_wide<ET, W, kGluClamped, false>(y + (col0 >> 1), g.ldy, bias, g.limit, row0, row_end, cols, acc);
                if (g.glu == kGluGelu) return gemm_out_wide<ET, W, kGluGelu, false>(y + (col0 >> 1), g.ldy, bias, g.limit, row0, row_end, cols, acc);
                if (g.bias) return gemm_out_wide<ET, W, 0, true>(y + col0, g.ldy, bias, 0.0f, row0, row_end, cols, acc);
                return gemm_out_wide<ET, W, 0, false>(y + col0, g.ldy, bias, 0.0f, row0, row_end, cols, acc);
            }
        }
    }
    gemm_out_loose<ET, W>(g, row0, row_end, col0, stores, smem, acc);
}

template <typename ET, int WM, int MI, int NI, int NA, int NB, bool ONCE = false>
struct FloatWalk : GemmWalk<ET, WM, MI, NI, NA, NB, ONCE> {
    static constexpr int MIv = MI, NIv = NI;
    static constexpr bool kMany = std::is_same<ET, bf16_t>::value && NI == 4 && (ONCE || MI == 4) && GemmWalk<ET, WM, MI, NI, NA, NB, ONCE>::kLds > 80 * 1024;   // of groups
};

template <typename ET, class W, int OUT>
__global__ __launch_bounds__(256, W::per_cu()) void gemm_float_walk_kernel(GemmArgs g, int tiles_m, int tiles_n, int stores) {
    extern __shared__ __attribute__((aligned(16))) int8_t gemm_smem[];
    if constexpr (!W::kSumsApart) arguments(g.a, g.w, g.lda, g.ldw, g.m, g.n, g.k, g.row_src, g.tiles, g.n_tiles, g.w_stride, g.parts, g.part_stride, tiles_m, tiles_n);
    int tm, tn, group = 0, row0, row_end;
    gemm_tile_of<W::kOnce ? 1 : 8>(blockIdx.x, tiles_m, tiles_n, tm, tn);
    if (g.tiles) {
        if (tm >= g.n_tiles[0]) return;
        const int4 e = g.tiles[tm];
        group = e.x; row0 = e.y; row_end = e.z;
    } else {
        row0 = tm * W::BM; row_end = min(g.m, row0 + W::BM);
    }
    const int col0 = tn * W::BN;
    const int part = blockIdx.y, stages = g.k * (int)sizeof(ET) / 128;
    int k0 = 0, k1 = stages;
    if (g.parts > 1) {
        // scalar registers: divisions are made in vector ones, and the loop would carry them along
        k0 = __builtin_amdgcn_readfirstlane(part * stages / g.parts);
        k1 = __builtin_amdgcn_readfirstlane((part + 1) * stages / g.parts);
    }
    g.y32 += part * g.part_stride;
    unsigned offa[W::AI], offb[W::BI];
#pragma unroll
    for (int j = 0; j < W::AI; j++) {
        const int r = W::load_row_a(j);
        int row = min(row0 + r, row_end - 1);
        if (g.row_src) row = g.row_src[row];
        offa[j] = (unsigned)row * (unsigned)(g.lda * sizeof(ET)) + W::load_byte(r);
    }
#pragma unroll
    for (int j = 0; j < W::BI; j++) {
        const int r = W::load_row_b(j);
        offb[j] = (unsigned)min(col0 + r, g.n - 1) * (unsigned)(g.ldw * sizeof(ET)) + W::load_byte(r);
    }
    f32x4 acc[W::MIv][W::NIv];
    const int8_t *const a = static_cast<const int8_t*>(g.a) + (size_t)k0 * 128, *const w = static_cast<const int8_t*>(g.w) + (size_t)group * g.w_stride * sizeof(ET) + (size_t)k0 * 128;
    W::run(a, w, offa, offb, k1 - k0, gemm_smem, acc, OneTile());
    const int r0 = row0 + W::row_of_wave(), c0 = col0 + W::col_of_wave();
    gemm_out<ET, W, OUT>(g, r0, row_end, c0, stores, gemm_smem, acc);
}

// Tiles of groups of rows, those of a CU in one workgroup.  A tile of an expert has 16 to 32 stages, and with a workgroup of its own it took 5 us besides: where its
// rows lie is three trips (tile table, row numbers, rows), then the ring filled and the outputs left.  A workgroup makes the trips once for kListed tiles
// (the offsets of their rows and what else there is to a tile stand in LDS behind the ring), and the ring goes on from one to the next.  Whole prompts of 8 layers
// of 64 experts, top 6, us: 500 tokens 2850 -> 2698, 700 3120 -> 2950, 1024 3565 -> 3470, 2000 4920 -> 4690, 4000 8040 -> 7610 (of these, where experts are one tile, 1.5 to 2 %
// were tiles that began at different stages of k, which they do no more).  The weights come at 4.1 TB/s where the tiles of 1024 tokens are 4.2 to 5 rounds of 256.
constexpr int kListed = 16;
template <typename ET, class W, int OUT>
struct GroupTiles {
    static constexpr bool kMany = true;
    static constexpr int kRowsAt = W::kLds, kTileAt = kRowsAt + kListed * W::BM * 4, kLds = kTileAt + kListed * 16;
    static_assert(kLds <= 160 * 1024, "ring and list");
    const GemmArgs& g;
    const int8_t* smem;
    int count, at = 0;
    __device__ __forceinline__ int4 tile(int i) const {
        const int4 t = reinterpret_cast<const int4*>(smem + kTileAt)[i];
        return make_int4(__builtin_amdgcn_readfirstlane(t.x), __builtin_amdgcn_readfirstlane(t.y), __builtin_amdgcn_readfirstlane(t.z), __builtin_amdgcn_readfirstlane(t.w));
    }
    __device__ __forceinline__ bool more() const { return at + 1 < count; }
    __device__ __forceinline__ void rows_of(int i, unsigned (&offa)[W::AI]) const {
        const unsigned* const off = reinterpret_cast<const unsigned*>(smem + kRowsAt) + i * W::BM;
#pragma unroll
        for (int j = 0; j < W::AI; j++) offa[j] = off[W::load_row_a(j)] + W::load_byte(W::load_row_a(j));
    }
    __device__ __forceinline__ void cols_of(int i, unsigned (&offb)[W::BI], const int8_t*& w) const {
        const int4 t = tile(i);
        w = static_cast<const int8_t*>(g.w) + (size_t)t.x * g.w_stride * sizeof(ET);
#pragma unroll
        for (int j = 0; j < W::BI; j++) {
            const int r = W::load_row_b(j);
            offb[j] = (unsigned)min(t.w * W::BN + r, g.n - 1) * (unsigned)(g.ldw * sizeof(ET)) + W::load_byte(r);
        }
    }
    __device__ __forceinline__ void rows(unsigned (&offa)[W::AI]) const { rows_of(at + 1, offa); }
    __device__ __forceinline__ void cols(unsigned (&offb)[W::BI], const int8_t*& w) const { cols_of(at + 1, offb, w); }
    __device__ __forceinline__ void out(f32x4 (&acc)[W::MIv][W::NIv]) {
        const int4 t = tile(at++);
        gemm_out<ET, W, OUT>(g, t.y + W::row_of_wave(), t.z, t.w * W::BN + W::col_of_wave(), kWide, nullptr, acc);
    }
};

template <typename ET, class W, int OUT>
__global__ __launch_bounds__(256, 1) void gemm_float_groups_kernel(GemmArgs g, int tiles_n) {
    extern __shared__ __attribute__((aligned(16))) int8_t gemm_smem[];
    static_assert(W::BM == W::RA, "a row number per row in LDS");
    using Tiles = GroupTiles<ET, W, OUT>;
    const int t = threadIdx.x, tiles_m = g.n_tiles[0], total = tiles_m * tiles_n;
    int4* const list = reinterpret_cast<int4*>(gemm_smem + Tiles::kTileAt);
    unsigned* const off = reinterpret_cast<unsigned*>(gemm_smem + Tiles::kRowsAt);
    for (int id0 = blockIdx.x; id0 < total; id0 += kListed * gridDim.x) {
        const int count = min(kListed, (total - id0 + (int)gridDim.x - 1) / (int)gridDim.x);
        __syncthreads();
        if (t < count) {
            int tm, tn;
            gemm_tile_of_lane<W::kOnce ? 1 : 8>(id0 + t * gridDim.x, tiles_m, tiles_n, tm, tn);
            const int4 e = g.tiles[tm];
            list[t] = make_int4(e.x, e.y, e.z, tn);
        }
        __syncthreads();
#pragma unroll 4
        for (int i = t; i < count * W::BM; i += 256) {
            const int4 e = list[i / W::BM];
            int row = min(e.y + i % W::BM, e.z - 1);
            if (g.row_src) row = g.row_src[row];
            off[i] = (unsigned)row * (unsigned)(g.lda * sizeof(ET));
        }
        __syncthreads();
        Tiles tiles{g, gemm_smem, count};
        unsigned offa[W::AI], offb[W::BI];
        const int8_t* w;
        tiles.rows_of(0, offa);
        tiles.cols_of(0, offb, w);
        f32x4 acc[W::MIv][W::NIv];
        W::run(static_cast<const int8_t*>(g.a), w, offa, offb, g.k * (int)sizeof(ET) / 128, gemm_smem, acc, tiles);
    }
}

// Whole pieces: rows and outputs start on 16 bytes, and both sides of the split are a multiple of the columns that a piece is made of.
template <typename ET>
static int gemm_stores(const GemmArgs& g) {
    const int piece = 16 / (int)sizeof(ET);
    if ((g.n & 3) || (g.n_split & 3) || (g.ldy & 3) || (g.ldy32 & 3)) return kSingle;
    const bool wide = rows_fit(g.ldy, sizeof(ET)) && rows_fit(g.ldy32, 4) && g.ldy % piece == 0 && g.n_split % (g.glu ? 2 * piece : piece) == 0 &&
                      ((reinterpret_cast<uintptr_t>(g.y) | reinterpret_cast<uintptr_t>(g.y32)) & 15) == 0;
    return wide ? kWide : kQuad;
}
// Tiles of 256 columns have kernels of their own for these forms; a wave's 128 columns lie on one side of the split, and with a gated unit there is
// only one.
static bool gemm_wide_ok(const GemmArgs& g) {
    return gemm_stores<bf16_t>(g) == kWide && (g.n_split == g.n || (!g.glu && g.n_split % 128 == 0)) && !(g.bias && g.glu);
}

// A workgroup's LDS beyond 64 KiB has to be asked for, once per kernel.
template <typename K>
static int opt_in(std::atomic<bool>& done, K kernel, int bytes) {
    if (!done.load(std::memory_order_acquire)) {
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        done.store(true, std::memory_order_release);
    }
    return FLEXLLM_OK;
}

template <typename ET, class W, int OUT>
static int launch_walk_out(const GemmArgs& g, hipStream_t st) {
    static std::atomic<bool> opted_in{false};
    if (const int rc = opt_in(opted_in, gemm_float_walk_kernel<ET, W, OUT>, W::kLds)) return rc;
    const int tm = g.tiles ? g.max_tiles : (g.m + W::BM - 1) / W::BM, tn = (g.n + W::BN - 1) / W::BN;
    gemm_float_walk_kernel<ET, W, OUT><<<dim3(tm * tn, g.parts), 256, W::kLds, st>>>(g, tm, tn, gemm_stores<ET>(g));
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

template <typename ET, class W, int OUT>
static int launch_groups_out(const GemmArgs& g, hipStream_t st) {
    static std::atomic<bool> opted_in{false};
    constexpr int lds = GroupTiles<ET, W, OUT>::kLds;
    if (const int rc = opt_in(opted_in, gemm_float_groups_kernel<ET, W, OUT>, lds)) return rc;
    const int tn = (g.n + W::BN - 1) / W::BN;
    gemm_float_groups_kernel<ET, W, OUT><<<min(256, g.max_tiles * tn), 256, lds, st>>>(g, tn);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

template <typename ET, int WM, int MI, int NI, int NA, int NB, bool ONCE = false>
static int launch_walk(const GemmArgs& g, hipStream_t st) {
    using W = FloatWalk<ET, WM, MI, NI, NA, NB, ONCE>;
    if constexpr (W::kMany) {
        if (g.tiles && gemm_wide_ok(g) && g.k * (int)sizeof(ET) / 128 >= NA && !g.bias) {
            if (g.glu == kGluClamped) return launch_groups_out<ET, W, kOutClamped>(g, st);
            if (!g.glu) return launch_groups_out<ET, W, kOutPlain>(g, st);
        }
    }
    if constexpr (W::kSumsApart) {
        if (!gemm_wide_ok(g)) return launch_walk_out<ET, W, kOutLoose>(g, st);
        if (g.glu == kGluClamped) return launch_walk_out<ET, W, kOutClamped>(g, st);
        if (g.glu == kGluGelu) return launch_walk_out<ET, W, kOutGelu>(g, st);
        return g.bias ? launch_walk_out<ET, W, kOutBias>(g, st) : launch_walk_out<ET, W, kOutPlain>(g, st);
    } else {
        return launch_walk_out<ET, W, kOutAny>(g, st);
    }
}

// A few float32 output columns (router rows, low-rank gate inputs): 16 rows x 16 columns per workgroup on
// v_mfma_f32_16x16x32_bf16, the four waves sharing k; operands straight from memory, eight k-steps in flight.
__global__ __launch_bounds__(256) void gemm_bf16_narrow_kernel(GemmArgs g, int n0) {
    __shared__ float part[4][16 * 17];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, row0 = blockIdx.x * 16, col0 = n0 + blockIdx.y * 16;
    const int r = min(row0 + (lane & 15), g.m - 1), c = min(col0 + (lane & 15), g.n - 1), kq = (lane >> 4) * 8;
    const bf16_t* a = static_cast<const bf16_t*>(g.a) + (size_t)r * g.lda + kq;
    const bf16_t* w = static_cast<const bf16_t*>(g.w) + (size_t)c * g.ldw + kq;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int B = 8;
    for (int k0 = wave * 32 * B; k0 < g.k; k0 += 4 * 32 * B) {
        bf16x8 fa[B], fb[B];
#pragma unroll
        for (int i = 0; i < B; i++) {
            const int k = min(k0 + i * 32, g.k - 32);     // k is a multiple of 64; steps beyond it are left out below
            fa[i] = *reinterpret_cast<const bf16x8*>(a + k);
            fb[i] = *reinterpret_cast<const bf16x8*>(w + k);
        }
#pragma unroll
        for (int i = 0; i < B; i++)
            if (k0 + i * 32 < g.k) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[i], acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) part[wave][((lane >> 4) * 4 + i) * 17 + (lane & 15)] = acc[i];
    __syncthreads();
    const int rr = t >> 4, cc = t & 15;
    const float v = (part[0][rr * 17 + cc] + part[1][rr * 17 + cc]) + (part[2][rr * 17 + cc] + part[3][rr * 17 + cc]);
    if (row0 + rr < g.m && col0 + cc < g.n) g.y32[(size_t)(row0 + rr) * g.ldy32 + (col0 + cc - g.n_split)] = g.bias ? v + g.bias[col0 + cc] : v;
}

// 128 rows where most of a group's rows fill most of them.  bfloat16, 8 layers of 64 experts, a whole prompt on 64 and on 128 rows: 65 rows per expert 3261 and 3125 us, 93
// rows 4025 and 3526.
template <typename ET>
int gemm_group_tile_rows(int rows_per_group) { return rows_per_group >= (sizeof(ET) == 2 ? 60 : 96) ? 128 : 64; }
template int gemm_group_tile_rows<bf16_t>(int);
template int gemm_group_tile_rows<float>(int);

static int gemm_check(GemmArgs& g, size_t a_rows, int es) {
    if (!g.ldw) g.ldw = g.k;
    FX_REQUIRE(g.a && g.w && g.m > 0 && g.n > 0 && g.k > 0 && g.k % kKPad == 0 && g.lda >= g.k && g.lda % 8 == 0 && g.ldw >= g.k && g.ldw % 8 == 0,
               "gemm_float: m=%d n=%d k=%d lda=%d", g.m, g.n, g.k, g.lda);
    FX_REQUIRE((size_t)a_rows * g.lda * es < (1ull << 31) && (size_t)g.n * g.ldw * es < (1ull << 31), "gemm_float: operands beyond 2 GiB");
    FX_REQUIRE(g.n_split >= 0 && g.n_split <= g.n && (g.n_split == 0 || g.y) && (g.n_split == g.n || g.y32), "gemm_float: output pointers");
    FX_REQUIRE(!g.glu || g.n_split % 2 == 0, "gemm_float: odd number of gate/up rows");
    FX_REQUIRE(!g.tiles || (g.n_tiles && g.max_tiles > 0), "gemm_float: tile table");
    FX_REQUIRE(g.parts >= 1 && (g.parts == 1 || (g.n_split == 0 && !g.bias && !g.tiles && g.parts <= g.k * es / 128)), "gemm_float: %d parts of k=%d", g.parts, g.k);
    return FLEXLLM_OK;
}

// The tile whose rounds over the chip take the least time.  cost: of one stage of a round, and `round` once per round, in 0.01 us, as
// measured where all CUs are busy; per_cu: workgroups that the rule counts with per CU.  The bfloat16 ones were set by 520 sizes of 1
// to 4096 rows and 64 to 14336 k on an earlier kernel; on this one the tiles picked are 1.1 % from the best ones on average over 44 sizes.  What a
// round costs besides its stages decides where k is short and the outputs' stores bound the product: 2806 x 6656 x 512 29 us on 160 rows
// of 256 columns and on 128 x 128 twice per CU, 37 on 128 x 256 and 38 on 128 x 128.
//
// bfloat16 (64 k): 777 x 28672 x 4096 takes 256 columns (169 us; 128 x 128: 222 us), 1531 x 16384 x 2048 too (86 us; 123), 777 x 4096 x 14336
// 128 x 128 (1 round, 99 us; 128 x 256: 159 us), 1024 x 2048 x 2048 64 x 128 (16.0 us; 128 x 128: 21.4 us).  128 x 128 with two stages fits
// twice into a CU: 1389 x 6528 x 640 22.5 us, 27.5 on the one with more stages.  (Four stages on the others: 777 x 2560 x 2048 18.6 us, five 19.4,
// three 19.7; 41 x 2048 x 8192 in eight parts on 64 x 64 9.1, six 9.3, three 10.0.)
// float32 (32 k): 333 x 16384 x 2048 takes 64 x 128 (196 us; 128 x 128: 244 us), 333 x 2048 x 8192 64 x 64 (135 us; 64 x 128: 248 us).
struct GemmTileCost { int bm, bn, cost, round, per_cu; };
template <typename ET> struct GemmTiles;
template <> struct GemmTiles<bf16_t> {
    static constexpr GemmTileCost list[] = {{256, 256, 190, 520, 1}, {128, 256, 107, 180, 1}, {128, 128, 64, 150, 1}, {64, 128, 51, 170, 1}, {64, 64, 37, 40, 1}, {128, 128, 120, 120, 2}};
};
template <> struct GemmTiles<float> { static constexpr GemmTileCost list[] = {{128, 128, 235, 0, 1}, {64, 128, 126, 100, 1}, {64, 64, 66, 0, 1}}; };

template <typename ET>
static int gemm_cheapest_tile(const GemmArgs& g, int parts, long& best) {
    const long stages = (long)g.k * sizeof(ET) / 128;
    int pick = -1, i = 0;
    for (const GemmTileCost& t : GemmTiles<ET>::list) {
        const long n = (long)((g.m + t.bm - 1) / t.bm) * ((g.n + t.bn - 1) / t.bn) * parts, slots = 256 * t.per_cu;
        const long cost = (n + slots - 1) / slots * (t.cost * ((stages + parts - 1) / parts) + t.round);
        if (pick < 0 || cost < best) { best = cost; pick = i; }
        i++;
    }
    return pick;
}

// bfloat16 products whose tile has 256 columns share their rows out anew: any multiple of 32 from 96 to 256 rows is a tile of its own on the
// same walk, and the one whose rounds cost least is taken (as above, in 0.01 us; the choices of 44 sizes of 120 to 4096 rows are 0.2 % from
// the best ones on average).  777 x 28672 x 4096 takes 224 rows (170 us; 256: 185, 128: 211), 1531 x 16384 x 2048 192 (88 us; 256: 111,
// 128: 103), 2596 x 3712 x 2560 160 (51 us; 256: 63, 128: 69), 722 x 10496 x 10112 128 (140 us; 160: 171, 256: 186),
// 2528 x 2048 x 8192 96 (90 us; 128: 97, 160: 114; 64 rows, a trip of W for half the products, 139).
struct GemmWideRows { int rows, stage, round; };
constexpr GemmWideRows kGemmWideRows[] = {{256, 135, 1100}, {224, 119, 1000}, {192, 105, 900}, {160, 99, 800}, {128, 83, 700}, {96, 70, 620}};
static int gemm_wide_rows(int m, int k, int n, int parts) {
    const long stages = ((long)k * 2 / 128 + parts - 1) / parts;
    long best = 0;
    int rows = 0;
    for (const GemmWideRows& t : kGemmWideRows) {
        const long tiles = (long)((m + t.rows - 1) / t.rows) * ((n + 255) / 256) * parts, cost = (tiles + 255) / 256 * (t.stage * stages + t.round);
        if (!rows || cost < best) { best = cost; rows = t.rows; }
    }
    return rows;
}

// Few rows of a long k leave most CUs without a tile, so k is shared out.  A part costs its sums' way to memory and back (8 bytes
// each at 5 TB/s, besides the launch that it does not add) and has at least a ring of stages to walk.  The costs are good to a few
// per cent, so that more parts have to be a 32nd cheaper; and the sums of all parts have to fit into the 32 MiB of the dies' L2 caches: beyond
// them they cost more than that.  Whole prompts of the layers of width 4096 (four) and 2048 (sixteen), with the parts taken here and
// in one part: 200 rows 1024 and 1120 us, 1700 and 1949; 1024 rows 2459 and 2532, 3596 and 3688; 1531 rows 3644 in two parts and 3516 in one (50
// MB of sums: one), 4879 and 5040 (25 MB).
template <typename ET>
int gemm_parts(const GemmArgs& g, int most) {
    constexpr size_t kSums = (size_t)32 << 20;
    long best = 0;
    int parts = 1;
    for (int p = 1; p <= most && p * 4 <= (int)(g.k * sizeof(ET) / 128); p *= 2) {
        if (p > 1 && (size_t)p * g.m * g.n * sizeof(float) > kSums) break;
        long cost;
        gemm_cheapest_tile<ET>(g, p, cost);
        cost += (long)p * g.m * g.n * 8 / 50000;
        if (p == 1 || cost < best - best / 32) { best = cost; parts = p; }
    }
    return parts;
}
template int gemm_parts<bf16_t>(const GemmArgs&, int);
template int gemm_parts<float>(const GemmArgs&, int);

template <>
int gemm_float<bf16_t>(const GemmArgs& args, hipStream_t st) {
    GemmArgs g = args;
    int rc = gemm_check(g, g.m, 2);
    if (rc) return rc;
    FX_REQUIRE(!g.tiles, "gemm_float: a tile table goes to gemm_grouped");
    // a few float32 columns behind whole tiles would cost a tile column of their own: they get the narrow kernel
    const int extra = g.n - g.n_split;
    if (g.n_split > 0 && extra > 0 && extra <= 256 && (g.n + 127) / 128 > (g.n_split + 127) / 128) {
        gemm_bf16_narrow_kernel<<<dim3((g.m + 15) / 16, (extra + 15) / 16), 256, 0, st>>>(g, g.n_split);
        FX_LAUNCH_CHECK();
        g.n = g.n_split;
    }
    if (!g.row_src && gemm_few_ok(g.m, g.k, g.n, g.parts)) return gemm_few(g, st);
    // With one row tile the weights are read once: past what the caches hold of the rows, unless the caches hold the weights too.  Whole prompts, us, weights read by
    // ordinary loads and past the caches: layers of 2048 (16), 33 rows 1196 and 1157, 64 1268 and 1252, 128 1416 and 1417; of 4096 (4), 33 760 and 734, 64 786 and 771, 128
    // 867 and 852.  Layers of 1024, 64 rows, by all weights: 125 MB 261 and 283, 243 MB 444 and 484, 365 MB 668 and 634, 487 MB 868 and 825.
    const bool one = g.from_memory && g.m <= 64, one_wide = g.from_memory && g.m <= 128;
    long cost;
    switch (gemm_cheapest_tile<bf16_t>(g, g.parts, cost)) {
        case 0: case 1: switch (gemm_wide_rows(g.m, g.k, g.n, g.parts)) {
            case 256: return launch_walk<bf16_t, 2, 8, 8, 3, 2>(g, st);
            case 224: return launch_walk<bf16_t, 2, 7, 8, 3, 2>(g, st);
            case 192: return launch_walk<bf16_t, 2, 6, 8, 3, 2>(g, st);
            case 160: return launch_walk<bf16_t, 2, 5, 8, 3, 2>(g, st);
            case 128: return launch_walk<bf16_t, 2, 4, 8, 4, 3>(g, st);
            default: return launch_walk<bf16_t, 2, 3, 8, 4, 3>(g, st);
        }
        case 2: return one_wide ? launch_walk<bf16_t, 2, 4, 4, 4, 4, true>(g, st) : launch_walk<bf16_t, 2, 4, 4, 4, 4>(g, st);
        case 3: return one ? launch_walk<bf16_t, 2, 2, 4, 4, 4, true>(g, st) : launch_walk<bf16_t, 2, 2, 4, 4, 4>(g, st);
        case 4: return one ? launch_walk<bf16_t, 2, 2, 2, 4, 4, true>(g, st) : launch_walk<bf16_t, 2, 2, 2, 4, 4>(g, st);
        default: return launch_walk<bf16_t, 2, 4, 4, 2, 2>(g, st);
    }
}

// Experts: their weights are read once and little else, so the tiles keep as many bytes in flight as LDS holds (1024 tokens, top 6 of
// 64 experts of 2048 x 2048 and 2048 x 1024: 143 and 90 us; the weights alone are 98 and 49 at 5.5 TB/s).  With fewer than 45 rows
// per expert most of a wide tile's rows are none, and three workgroups per CU on 64 x 64 hide more of each other's trips.  Where an expert's rows are
// one tile its weights are read once, past what the caches hold of the rows, and a die takes all columns of an expert: 64 rows 2394 -> 2265 us (a whole
// prompt of 8 layers), 500 2886 -> 2793, 1024 3588 -> 3537.  Up to 112 rows on average on 128: at 122 many experts have two tiles (4230 -> 4239 us), at 188 4918 -> 5284.
// Not where the caches hold all weights: 125 MB in two layers of 16 experts, 64 tokens 275 us and 290, 200 299 and 314; 250 MB 507 and 493, 536 and 528.
template <int BM>
static int gemm_grouped_bf16(const GemmArgs& args, hipStream_t st) {
    GemmArgs g = args;
    int rc = gemm_check(g, g.m, 2);
    if (rc) return rc;
    if constexpr (BM == 128) return g.from_memory && g.group_rows <= 112 ? launch_walk<bf16_t, 2, 4, 4, 4, 4, true>(g, st) : launch_walk<bf16_t, 2, 4, 4, 4, 4>(g, st);
    else if (g.group_rows < 45) return g.from_memory ? launch_walk<bf16_t, 2, 2, 2, 3, 3, true>(g, st) : launch_walk<bf16_t, 2, 2, 2, 3, 3>(g, st);
    else return g.from_memory ? launch_walk<bf16_t, 2, 2, 4, 4, 4, true>(g, st) : launch_walk<bf16_t, 2, 2, 4, 4, 4>(g, st);
}

// ---- float32 -----------------------------------------------------------------------------------------------------
template <>
int gemm_float<float>(const GemmArgs& args, hipStream_t st) {
    GemmArgs g = args;
    int rc = gemm_check(g, g.m, 4);
    if (rc) return rc;
    FX_REQUIRE(!g.tiles, "gemm_float: a tile table goes to gemm_grouped");
    long cost;
    switch (gemm_cheapest_tile<float>(g, g.parts, cost)) {
        case 0: return launch_walk<float, 2, 4, 4, 4, 4>(g, st);
        case 1: return launch_walk<float, 2, 2, 4, 4, 4>(g, st);
        default: return launch_walk<float, 2, 2, 2, 3, 3>(g, st);
    }
}

template <int BM>
static int gemm_grouped_f32(const GemmArgs& args, hipStream_t st) {
    GemmArgs g = args;
    int rc = gemm_check(g, g.m, 4);
    if (rc) return rc;
    if constexpr (BM == 128) return launch_walk<float, 2, 4, 2, 3, 3>(g, st);
    else return launch_walk<float, 2, 2, 2, 3, 3>(g, st);
}

template <typename ET>
int gemm_grouped(const GemmArgs& g, int tile_rows, hipStream_t st) {
    FX_REQUIRE(g.tiles && (tile_rows == 64 || tile_rows == 128), "gemm_grouped: tile table of %d rows", tile_rows);
    if constexpr (std::is_same<ET, float>::value) return tile_rows == 128 ? gemm_grouped_f32<128>(g, st) : gemm_grouped_f32<64>(g, st);
    else return tile_rows == 128 ? gemm_grouped_bf16<128>(g, st) : gemm_grouped_bf16<64>(g, st);
}
template int gemm_grouped<bf16_t>(const GemmArgs&, int, hipStream_t);
template int gemm_grouped<float>(const GemmArgs&, int, hipStream_t);

}  // namespace fx

using namespace fx;

extern "C" {

int flexllm_linear_float_gemm(const void* a, const void* w, const float* bias, void* y, float* y32, int m, int k, int n, int n_split, int glu, float limit,
                              int dtype, void* stream) {
    FX_REQUIRE((dtype == 0 || dtype == 1) && glu >= 0 && glu <= 1 + FLEXLLM_GLU_GELU, "linear_float_gemm: dtype=%d glu=%d", dtype, glu);
    GemmArgs g;
    g.a = a; g.w = w; g.lda = k; g.m = m; g.n = n; g.k = k; g.n_split = n_split; g.glu = glu; g.limit = limit; g.bias = bias;
    g.y = y; g.ldy = glu ? n_split / 2 : n_split; g.y32 = y32; g.ldy32 = n - n_split;
    g.from_memory = n > 0 && k > 0 && (size_t)n * k * (dtype ? 4 : 2) > kCacheBytes;
    return dtype == 0 ? gemm_float<bf16_t>(g, as_stream(stream)) : gemm_float<float>(g, as_stream(stream));
}

int flexllm_linear_float_gemm_tile(int m, int k, int n, int dtype, int* rows, int* cols, int* per_cu) {
    FX_REQUIRE((dtype == 0 || dtype == 1) && m > 0 && n > 0 && k > 0 && k % kKPad == 0 && rows && cols && per_cu, "linear_float_gemm_tile: m=%d k=%d n=%d dtype=%d", m, k, n, dtype);
    GemmArgs g;
    g.m = m; g.k = k; g.n = n;
    long cost;
    const GemmTileCost& t = dtype == 0 ? GemmTiles<bf16_t>::list[gemm_cheapest_tile<bf16_t>(g, 1, cost)] : GemmTiles<float>::list[gemm_cheapest_tile<float>(g, 1, cost)];
    *rows = t.bm;
    *cols = t.bn;
    *per_cu = t.per_cu;
    return FLEXLLM_OK;
}

int flexllm_linear_float_gemm_rows(int m, int k, int n, int dtype, int parts) {
    FX_REQUIRE((dtype == 0 || dtype == 1) && m > 0 && n > 0 && k > 0 && k % kKPad == 0 && parts > 0, "linear_float_gemm_rows: m=%d k=%d n=%d dtype=%d", m, k, n, dtype);
    GemmArgs g;
    g.m = m; g.k = k; g.n = n;
    long cost;
    if (dtype) return GemmTiles<float>::list[gemm_cheapest_tile<float>(g, parts, cost)].bm;
    if (gemm_few_ok(m, k, n, parts)) return m <= 16 ? 16 : 32;
    const GemmTileCost& t = GemmTiles<bf16_t>::list[gemm_cheapest_tile<bf16_t>(g, parts, cost)];
    return t.bn == 256 ? gemm_wide_rows(m, k, n, parts) : t.bm;
}

int flexllm_linear_float_gemm_parts(int m, int k, int n, int dtype, int most) {
    FX_REQUIRE((dtype == 0 || dtype == 1) && m > 0 && n > 0 && k > 0 && k % kKPad == 0 && most > 0, "linear_float_gemm_parts: m=%d k=%d n=%d dtype=%d", m, k, n, dtype);
    GemmArgs g;
    g.m = m; g.k = k; g.n = n;
    return dtype == 0 ? gemm_parts<bf16_t>(g, most) : gemm_parts<float>(g, most);
}

}  // extern "C"
