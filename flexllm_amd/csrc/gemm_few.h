// bfloat16 GEMM of few rows (prompts of 9 to 32 tokens per pass over the weights): C[m][n] = sum_k A[m][k] * W[n][k].
//
// The weights' one pass through the chip bounds it, and that hangs on how they are asked for: in requests of 1 KiB of one row they
// stream at 5.8 TB/s (67 MB in 11.5 us), in the eight rows of 128 bytes that a stage of the wide GEMMs is made of at 4.4.  So the schedule is that of the
// steps of several tokens (gemv_mfma_kernel): eight waves share a unit of UK of k of 16 rows of W, which goes to LDS in requests of 1 KiB
// (16-byte chunk c of row r at place c ^ r, for reads without conflicts); a tile has UNITS of them, two are in flight, and a unit's place is
// free for the next but one as soon as its operands are in registers.  A stays in registers, each wave's own stretch of k of all rows.
// The waves' sums meet through LDS per tile.
#pragma once
#include "float_ops.h"
#include "gemm_walk.h"

namespace fx {

constexpr int kFewMost = 32;                              // rows of A in a pass over the weights

template <int UK, int UNITS, int NG>                      // 16 * NG rows of A
__global__ __launch_bounds__(512, 2) void gemm_few_kernel(GemmArgs g) {
    constexpr int NW = 8, SL = UK / NW, SW = SL / 32;      // k and matrix k-steps of a wave in a unit
    constexpr int UB = UK * 2, SLOT = 16 * UB, SLOTS = 128 * 1024 / SLOT, PER = SLOT / 1024 / NW;      // PER: requests of a wave per unit
    extern __shared__ __attribute__((aligned(16))) int8_t ring[];
    __shared__ float red[NW][NG][16 * 17];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), gq = lane >> 4;
    const int walker = blockIdx.x, walkers = gridDim.x, tiles = (g.n + 15) / 16;
    const int mine = (tiles - walker + walkers - 1) / walkers, total = mine * UNITS;          // tiles and units of this workgroup
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)ring;
    auto request_unit = [&](int u) __attribute__((always_inline)) {
        const int tile = walker + u / UNITS * walkers, h = u % UNITS, last = min(16, g.n - tile * 16) - 1;
        const int8_t* base = static_cast<const int8_t*>(g.w) + (size_t)tile * 16 * g.ldw * 2;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int p = wave * PER + q, r = p / (UB / 1024), seg = p % (UB / 1024);
            // what is behind the row's end (any of its bytes will do) is not looked at
            const int kb = min(h * UK * 2 + seg * 1024 + (lane ^ r) * 16, g.k * 2 - 16);
            load_to_lds<true>(base, (unsigned)(min(r, last) * g.ldw * 2 + kb), lds0 + (u % SLOTS) * SLOT + p * 1024);
        }
    };
    bf16x8 af[UNITS * SW][NG];
    int steps[UNITS];                                     // k-steps of this wave that there are
#pragma unroll
    for (int h = 0; h < UNITS; h++) {
        const int first = h * UK + wave * SL;
        steps[h] = max(0, min(SW, (g.k - first) / 32));
#pragma unroll
        for (int s = 0; s < SW; s++)
#pragma unroll
            for (int q = 0; q < NG; q++)
                af[h * SW + s][q] = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(g.a) + (size_t)min(q * 16 + (lane & 15), g.m - 1) * g.lda +
                                                                     min(first + s * 32, g.k - 32) + gq * 8);
    }
    wait_vmcnt<0>();                                      // results come in the order of the requests
#pragma unroll
    for (int u = 0; u < SLOTS; u++)
        if (u < total) request_unit(u);
    auto all_done = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    // thread = column r of the tile, row j of A; with the gated unit every other one has a neighbour's sum besides
    const int r = t & 15, j = t >> 4;
    auto sums = [&]() __attribute__((always_inline)) {
        if (j >= 16 * NG) return 0.0f;
        float v[NW];
#pragma unroll
        for (int q = 0; q < NW; q++) v[q] = red[q][j >> 4][r * 17 + (j & 15)];
        return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    };
    auto finish = [&](int i, float s) __attribute__((always_inline)) {
        const int col = (walker + i * walkers) * 16 + r;
        if (g.bias) s += g.bias[min(col, g.n - 1)];
        const float up = lane_xor_f<1>(s);
        if (j >= g.m || col >= g.n) return;
        bf16_t* y = static_cast<bf16_t*>(g.y);
        if (col >= g.n_split) g.y32[(size_t)j * g.ldy32 + col - g.n_split] = s;
        else if (!g.glu) y[(size_t)j * g.ldy + col] = (bf16_t)s;
        else if ((col & 1) == 0) y[(size_t)j * g.ldy + (col >> 1)] = (bf16_t)glu_f(g.glu, s, up, g.limit);
    };
    const int8_t* const in0 = ring + (lane & 15) * UB;
    for (int i = 0; i < mine; i++) {
        f32x4 acc[NG];
#pragma unroll
        for (int q = 0; q < NG; q++) acc[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        float before = 0.0f;
#pragma unroll
        for (int h = 0; h < UNITS; h++) {
            const int u = i * UNITS + h, younger = total - 1 - u;
            if (younger >= SLOTS - 1) wait_vmcnt<(SLOTS - 1) * PER>();
            else if (SLOTS > 3 && younger == 2) wait_vmcnt<2 * PER>();
            else if (SLOTS > 2 && younger == 1) wait_vmcnt<PER>();
            else wait_vmcnt<0>();
            all_done();                                   // the last tile's sums have left
            barrier();
            bf16x8 wf[SW];
            const int8_t* in = in0 + (u % SLOTS) * SLOT;
#pragma unroll
            for (int s = 0; s < SW; s++) {
                const int c = wave * (SL / 8) + s * 4 + gq;
                wf[s] = *reinterpret_cast<const bf16x8*>(in + (c ^ (lane & 15)) * 16);
            }
            if (h == 0 && i > 0) before = sums();
            all_done();
            barrier();
            if (u + SLOTS < total) request_unit(u + SLOTS);
            if (h == 0 && i > 0) finish(i - 1, before);
#pragma unroll
            for (int s = 0; s < SW; s++)
                if (s < steps[h])
#pragma unroll
                    for (int q = 0; q < NG; q++) acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], af[h * SW + s][q], acc[q], 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < NG; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) red[wave][q][(gq * 4 + e) * 17 + (lane & 15)] = acc[q][e];
    }
    __syncthreads();
    finish(mine - 1, sums());
}

// Products of at most 32 rows run here where a workgroup has two tiles or more, so that their weights' stream is long enough to pay for
// the start (A into registers) and the sums, and where k fills the units: a place in the ring that is half empty is half as much in flight, and an
// instruction on nothing takes as long as another.  The tiles of the wide GEMMs and this, us: 16384 x 2048, 9 rows 17.6 and 13.8, 32 rows 18.0 and 16.9; 28672 x
// 4096 53 and 38, 53 and 44; 8192 x 512, 16 rows 6.3 and 5.2, 32 rows 6.5 and 6.4 (stays).  Units that are not full: 12300 x 3072, 16 rows 18.6 and 17.6, 17 rows
// 19.0 and 20.1 (stays); 20480 x 2112, 16 rows 19.3 and 21.0 (stays); 16384 x 1088, 32 rows 10.2 and 12.2 (stays).  k below 512: 8192 x 64, 16 rows
// 3.9 and 5.0 (stays).  Over 240 sizes of 8 to 32 rows, 64 to 4096 k and 8192 to 28672 columns the choice is 1.1 % from the better one on average, and at
// most 1.6 % behind the tiles.
inline bool gemm_few_ok(int m, int k, int n, int parts) {
    if (m > kFewMost || parts != 1 || k > 4096 || n < 8192) return false;
    const int units = k <= 1024 ? 1024 : k <= 2048 ? 2048 : 4096;
    return m <= 16 ? k >= 512 && (k <= 1024 || k * 4 >= units * 3) : k > 1024 && k * 8 >= units * 7;
}

template <int UK, int UNITS, int NG>
static int launch_few(const GemmArgs& g, hipStream_t st) {
    constexpr int lds = 128 * 1024;
    static std::atomic<bool> opted_in{false};
    if (!opted_in.load(std::memory_order_acquire)) {
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_few_kernel<UK, UNITS, NG>), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        opted_in.store(true, std::memory_order_release);
    }
    gemm_few_kernel<UK, UNITS, NG><<<256, 512, lds, st>>>(g);      // one workgroup per CU, of two tiles or more
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}
inline int gemm_few(const GemmArgs& g, hipStream_t st) {
    if (g.m <= 16) return g.k <= 1024 ? launch_few<1024, 1, 1>(g, st) : g.k <= 2048 ? launch_few<2048, 1, 1>(g, st) : launch_few<2048, 2, 1>(g, st);
    return g.k <= 2048 ? launch_few<2048, 1, 2>(g, st) : launch_few<2048, 2, 2>(g, st);
}

}  // namespace fx
