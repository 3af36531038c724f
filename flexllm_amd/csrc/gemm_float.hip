// Floating-point GEMMs for prefill: C[m][n] = sum_k A[m][k] * W[n][k], both operands K-contiguous.
//
// bfloat16: the direct-load kernel of the int8 path (gemm_i8.h) on v_mfma_f32_32x32x16_bf16.  A lane's operand is the
// same 16 bytes of a row as in the int8 instruction, so the LDS stage layout, the chunk rotation and the software
// pipeline carry over with K counted in bytes.  Additions: rows of A may be gathered, groups of rows may have a weight
// matrix each (experts), the epilogue adds a bias, splits the columns between an ET and a float32 output and applies the
// gated unit to interleaved gate/up columns.
//
// float32: the same kernel on v_mfma_f32_32x32x2_f32 (full float32 products and sums).  The 16 bytes that a lane holds are four k of
// a row, and instruction e of four takes its e-th: the two halves of the wave then stand for k apart, the same ones in
// both operands, and a sum does not mind.  (A register-staged 64 x 64 tile, which this took the place of: 333 x 2048 x 8192 345 us,
// now 173; 2048 x 4096 x 4096 950 us, now 602.)
#include "float_ops.h"
#include "gemm_i8.h"

namespace fx {

struct GemmTile { int row0, row_end, group; };

// Which tile this workgroup works on: row tiles fastest inside a range of weight columns per XCD, as in gemm_i8_kernel.
template <int BM, int BN>
__device__ __forceinline__ bool gemm_pick_tile(const GemmArgs& g, int tiles_m, int tiles_n, GemmTile& t, int& col0) {
    const int tile = blockIdx.x;
    int tm, tn;
    if ((tiles_n & 7) == 0) {
        const int xcd = tile & 7, idx = tile >> 3;
        tn = xcd * (tiles_n >> 3) + idx / tiles_m;
        tm = idx % tiles_m;
    } else {
        tm = tile % tiles_m;
        tn = tile / tiles_m;
    }
    col0 = tn * BN;
    if (g.tiles) {
        if (tm >= g.n_tiles[0]) return false;
        const int4 e = g.tiles[tm];
        t.group = e.x; t.row0 = e.y; t.row_end = e.z;
    } else {
        t.group = 0; t.row0 = tm * BM; t.row_end = min(g.m, t.row0 + BM);
    }
    return true;
}

// One row's four consecutive columns col..col+3 of the accumulator tile.
template <typename ET>
__device__ __forceinline__ void gemm_store4(const GemmArgs& g, int row, int col, float (&v)[4], bool vec) {
    ET* y = static_cast<ET*>(g.y);
    if (g.bias) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += g.bias[min(col + e, g.n - 1)];
    }
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

// The accumulator tile of a wave turns through a private LDS patch so that a lane owns four consecutive columns.
template <typename ET, int TM, int TN>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, const GemmTile& t, int col0, int wm, int wn, int lane, float* patch,
                                              f32x16 (&acc)[TM][TN]) {
    constexpr int EP = 36;
    const int pr = lane >> 3, pc = (lane & 7) * 4;
    // four columns never straddle the split, and every store address is a multiple of the store's size
    const bool vec = (g.n & 3) == 0 && (g.n_split & 3) == 0 && (g.ldy & 3) == 0 && (g.ldy32 & 3) == 0;
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++) {
#pragma unroll
            for (int r = 0; r < 16; r++) patch[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * EP + (lane & 31)] = acc[i][j][r];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const int lr = p * 8 + pr, row = t.row0 + wm + i * 32 + lr;
                const f32x4 q = *reinterpret_cast<const f32x4*>(patch + lr * EP + pc);
                float v[4] = {q[0], q[1], q[2], q[3]};
                if (row < t.row_end) gemm_store4<ET>(g, row, col0 + wn + j * 32 + pc, v, vec);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
}

// A stage is 128 bytes of k of the tile's rows and columns; STAGES of them form the ring in LDS.
// What bounds it: with one workgroup per CU the trip of a stage's bytes, so that everything LDS holds is in flight (two stages of
// 128 x 128 in four waves, of which a CU could hold two: 213 us for 777 x 4096 x 14336, 224 tiles; four stages, eight waves: 117 us), and for the
// largest tile LDS itself, which hands out 6 KiB of operands for 8 matrix instructions per wave.
template <typename ET, int BM, int BN, int STAGES, int WPE, int NW>
__global__ __launch_bounds__(NW * 64, WPE) void gemm_float_dma_kernel(GemmArgs g, int tiles_m, int tiles_n) {
    constexpr int BKB = 128, GW = NW, WGN = GW / 2;
    constexpr int WM = BM / 2, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    constexpr int CPR = BKB / 16, RPI = 64 / CPR;
    constexpr int A_INSTR = BM / (GW * RPI), B_INSTR = BN / (GW * RPI);
    static_assert(A_INSTR >= 1 && B_INSTR >= 1 && TM >= 1 && TN >= 1, "tile too small for this wave count");
    constexpr int STAGE = (BM + BN) * BKB, KS = BKB / 32;
    auto rot = [](int r) { return (r >> 1) & 7; };
    extern __shared__ __attribute__((aligned(16))) int8_t gemm_smem[];

    GemmTile tl;
    int col0;
    // scalar registers for the ends of the part: divisions are made in vector ones, and the loop would carry them along
    const int part = blockIdx.y, stages = g.k * (int)sizeof(ET) / BKB;
    const int k0 = __builtin_amdgcn_readfirstlane(part * stages / g.parts);
    if (!gemm_pick_tile<BM, BN>(g, tiles_m, tiles_n, tl, col0)) return;
    g.y32 += part * g.part_stride;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
    const int8_t* const a = static_cast<const int8_t*>(g.a) + (size_t)k0 * BKB;
    const int8_t* const w = static_cast<const int8_t*>(g.w) + (size_t)tl.group * g.w_stride * sizeof(ET) + (size_t)k0 * BKB;

    unsigned offa[A_INSTR], offb[B_INSTR];
#pragma unroll
    for (int j = 0; j < A_INSTR; j++) {
        const int r = (wave * A_INSTR + j) * RPI + lane / CPR;
        int row = min(tl.row0 + r, tl.row_end - 1);
        if (g.row_src) row = g.row_src[row];
        offa[j] = (unsigned)row * (unsigned)(g.lda * sizeof(ET)) + (unsigned)(((lane % CPR) ^ rot(r)) * 16);
    }
#pragma unroll
    for (int j = 0; j < B_INSTR; j++) {
        const int r = (wave * B_INSTR + j) * RPI + lane / CPR;
        offb[j] = (unsigned)min(col0 + r, g.n - 1) * (unsigned)(g.ldw * sizeof(ET)) + (unsigned)(((lane % CPR) ^ rot(r)) * 16);
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)gemm_smem;
    auto issue_stage = [&](int kt) {
        const unsigned sb = lds0 + (unsigned)(kt % STAGES) * STAGE;
        const size_t koff = (size_t)kt * BKB;
#pragma unroll
        for (int j = 0; j < A_INSTR; j++) gemm_dma_issue(a + koff, offa[j], sb + (wave * A_INSTR + j) * 1024);
#pragma unroll
        for (int j = 0; j < B_INSTR; j++) gemm_dma_issue(w + koff, offb[j], sb + BM * BKB + (wave * B_INSTR + j) * 1024);
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    const int nk = __builtin_amdgcn_readfirstlane((part + 1) * stages / g.parts) - k0;
    constexpr int PER = A_INSTR + B_INSTR;
    // everything the compiler loaded itself (tile table, gathered row numbers) has to be in before the counted loads start
    gemm_wait_vmcnt<0>();
#pragma unroll
    for (int s0 = 0; s0 < STAGES - 1; s0++)
        if (s0 < nk) issue_stage(s0);
    const int fr = lane & 31, fg = lane >> 5;
    using Frag = std::conditional_t<std::is_same<ET, float>::value, f32x4, bf16x8>;
    auto read_frags = [&](int kt, int ks, Frag (&fa)[TM], Frag (&fb)[TN]) {
        const int8_t* sa = gemm_smem + (kt % STAGES) * STAGE;
        const int8_t* sb = sa + BM * BKB;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int r = wm + i * 32 + fr;
            fa[i] = *reinterpret_cast<const Frag*>(sa + r * BKB + (((ks * 2 + fg) ^ rot(r)) * 16));
        }
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int r = wn + j * 32 + fr;
            fb[j] = *reinterpret_cast<const Frag*>(sb + r * BKB + (((ks * 2 + fg) ^ rot(r)) * 16));
        }
    };
    auto mma = [&](const Frag (&fa)[TM], const Frag (&fb)[TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if constexpr (std::is_same<ET, float>::value) {
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][e], fb[j][e], acc[i][j], 0, 0, 0);
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
                }
            }
    };
    auto wait_stage = [&](int kt) {
        const int younger = min(STAGES - 2, nk - 1 - kt);
        if (younger >= 2) gemm_wait_vmcnt<2 * PER>();
        else if (younger == 1) gemm_wait_vmcnt<PER>();
        else gemm_wait_vmcnt<0>();
    };
    static_assert(STAGES <= 4 && 2 * PER < 64, "the wait distinguishes up to two younger stages");

    Frag fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    wait_stage(0);
    __syncthreads();
    read_frags(0, 0, fa0, fb0);
    // The last stage stands by itself, a branch less in the loop: 2 x 72 x 9024, one tile of 141 stages, 36.7 -> 31.0 us.
    auto stage = [&](int kt, auto more) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < KS; ks += 2) {
            read_frags(kt, ks + 1, fa1, fb1);
            if (more && ks == 0 && kt + STAGES - 1 < nk) issue_stage(kt + STAGES - 1);
            __builtin_amdgcn_sched_barrier(0);
            mma(fa0, fb0);
            __builtin_amdgcn_sched_barrier(0);
            if (ks + 2 < KS) {
                read_frags(kt, ks + 2, fa0, fb0);
            } else if (more) {
                wait_stage(kt + 1);
                __syncthreads();
                read_frags(kt + 1, 0, fa0, fb0);
            }
            __builtin_amdgcn_sched_barrier(0);
            mma(fa1, fb1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int kt = 0; kt < nk - 1; kt++) stage(kt, std::true_type());
    stage(nk - 1, std::false_type());
    __syncthreads();
    gemm_epilogue<ET, TM, TN>(g, tl, col0, wm, wn, lane, reinterpret_cast<float*>(gemm_smem) + wave * (32 * 36), acc);
}

constexpr int gemm_float_lds(int bm, int bn, int stages, int nw) {
    const int ring = stages * (bm + bn) * 128, epi = nw * 32 * 36 * 4;
    return ring > epi ? ring : epi;
}

template <typename ET, int BM, int BN, int STAGES, int WPE, int NW>
static int launch_dma(const GemmArgs& g, hipStream_t st) {
    constexpr int lds = gemm_float_lds(BM, BN, STAGES, NW);
    static std::atomic<bool> opted_in{false};
    if (!opted_in.load(std::memory_order_acquire)) {
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_float_dma_kernel<ET, BM, BN, STAGES, WPE, NW>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        opted_in.store(true, std::memory_order_release);
    }
    const int tm = g.tiles ? g.max_tiles : (g.m + BM - 1) / BM, tn = (g.n + BN - 1) / BN;
    gemm_float_dma_kernel<ET, BM, BN, STAGES, WPE, NW><<<dim3(tm * tn, g.parts), NW * 64, lds, st>>>(g, tm, tn);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
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

int gemm_group_tile_rows(int rows_per_group) { return rows_per_group >= 96 ? 128 : 64; }

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
// measured where all CUs are busy; per_cu: workgroups that a CU holds at a time.  The bfloat16 ones are those that lose least over 520 sizes of 1
// to 4096 rows and 64 to 14336 k: the tiles picked are 0.6 % from the best ones on average.  What a round costs besides its stages decides where k
// is short and the outputs' stores bound the product: 2409 x 5608 x 256 23.7 us on 256 x 256, 20.5 on 128 x 128 twice per CU,
// where 1621 x 22276 x 320 takes 54.8 us on 128 x 256 and 63.4 on those; 2070 x 9468 x 5632 293 us on 128 x 128, 253 on 128 x 256.
//
// bfloat16 (64 k): 777 x 28672 x 4096 takes 256 x 256 (2 rounds, 230 us; 128 x 128: 7 rounds, 255 us), 1531 x 16384 x 2048 128 x 256 (3
// rounds, 113 us; 256 x 256: 2 rounds, 141 us), 777 x 4096 x 14336 128 x 128 (1 round, 117 us; 128 x 256: 170 us), 1024 x 2048 x 2048
// 64 x 128 (14.4 us; 128 x 128: 19.4 us).  128 x 128 in four waves with two stages fits twice into a CU: 3700 x 2064 x 8576, 493 tiles,
// takes one round of it (130 us; two rounds of the one with four stages: 181 us).
// float32 (32 k): 333 x 16384 x 2048 takes 64 x 128 (251 us; 64 x 64: 265, 128 x 128: 289 us), 333 x 2048 x 8192 64 x 64 (173 us; 64 x 128:
// 276 us), 2048 x 4096 x 4096 128 x 128 (602 us, 114 TFLOP/s; 64 x 64: 656 us).
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
    long cost;
    switch (gemm_cheapest_tile<bf16_t>(g, g.parts, cost)) {
        case 0: return launch_dma<bf16_t, 256, 256, 2, 2, 8>(g, st);
        case 1: return launch_dma<bf16_t, 128, 256, 3, 2, 8>(g, st);
        case 2: return launch_dma<bf16_t, 128, 128, 4, 2, 8>(g, st);
        case 3: return launch_dma<bf16_t, 64, 128, 4, 2, 8>(g, st);
        case 4: return launch_dma<bf16_t, 64, 64, 4, 2, 4>(g, st);
        default: return launch_dma<bf16_t, 128, 128, 2, 2, 4>(g, st);
    }
}

// Experts: their weights are read once and little else, so the tiles keep as many bytes in flight as LDS holds (64 experts of
// 2048 x 2048 and 2048 x 1024, 1024 tokens, top 6: 134 us on average with two stages in four waves, 122 with four in eight;
// the weights alone are 73 us at 5.5 TB/s).  With fewer than 45 rows per expert most of a wide tile's rows are none, and three workgroups per
// CU on 64 x 64 hide more of each other's trips (the mixture's whole prompt of 9 rows 1711 -> 1666 us, 333 rows 2743 -> 2669, 450 rows
// 2830 -> 2772; 500 rows, 47 per expert, 2841 and 2850, 600 rows 3093 and 3143).
template <int BM>
static int gemm_grouped_bf16(const GemmArgs& args, hipStream_t st) {
    GemmArgs g = args;
    int rc = gemm_check(g, g.m, 2);
    if (rc) return rc;
    if constexpr (BM == 128) return launch_dma<bf16_t, 128, 128, 4, 2, 8>(g, st);
    else if (g.group_rows < 45) return launch_dma<bf16_t, 64, 64, 3, 3, 4>(g, st);
    else return launch_dma<bf16_t, 64, 128, 4, 2, 8>(g, st);
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
        case 0: return launch_dma<float, 128, 128, 4, 2, 8>(g, st);
        case 1: return launch_dma<float, 64, 128, 4, 2, 8>(g, st);
        default: return launch_dma<float, 64, 64, 4, 2, 4>(g, st);
    }
}

template <int BM>
static int gemm_grouped_f32(const GemmArgs& args, hipStream_t st) {
    GemmArgs g = args;
    int rc = gemm_check(g, g.m, 4);
    if (rc) return rc;
    if constexpr (BM == 128) return launch_dma<float, 128, 64, 4, 2, 4>(g, st);
    else return launch_dma<float, 64, 64, 4, 2, 4>(g, st);
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

int flexllm_linear_float_gemm_parts(int m, int k, int n, int dtype, int most) {
    FX_REQUIRE((dtype == 0 || dtype == 1) && m > 0 && n > 0 && k > 0 && k % kKPad == 0 && most > 0, "linear_float_gemm_parts: m=%d k=%d n=%d dtype=%d", m, k, n, dtype);
    GemmArgs g;
    g.m = m; g.k = k; g.n = n;
    return dtype == 0 ? gemm_parts<bf16_t>(g, most) : gemm_parts<float>(g, most);
}

}  // extern "C"
