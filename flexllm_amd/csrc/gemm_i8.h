// int8 x int8 -> int32 GEMM for prefill on gfx950 matrix cores: C[m][n] = sum_k A[m][k]*W[n][k].
//
// Both operands are K-contiguous, which is exactly the per-lane operand shape of
// v_mfma_i32_32x32x32_i8 (lane l supplies 16 consecutive k-bytes of row/column l%32, k-group l/32), so
// tiles go global -> registers -> LDS (16-byte chunks, k-chunk-major planes) -> MFMA operands with plain
// 128-bit reads and no transposition.  Integer accumulation: exact in any order.
//
// Workgroup tile BM x BN x 64, 256 threads = 4 waves in a 2x2 grid, each wave (BM/2)x(BN/2) as 32x32 MFMA
// tiles, double-buffered LDS, four k-steps of global loads in flight in registers.
#pragma once
#include "attn_decode_kernels.h"
#include "common.h"
#include "gemm_walk.h"
#include <atomic>
#include <type_traits>

namespace fx {

constexpr int kGemmBK = 64;        // k-bytes per stage
// LDS tile layout: [16-byte k-chunk (4 per stage)][row][16 B], i.e. for one k-chunk the rows are contiguous.
// A wave-wide 128-bit fragment read then touches two contiguous 512-byte runs; the +32 B on the plane pitch
// spreads the four chunks of one row, written by four neighbouring lanes, over all banks.
__host__ __device__ constexpr int gemm_plane(int rows) { return rows * 16 + 32; }

enum GemmEpi { kGemmRaw = 0, kGemmDequant = 1, kGemmDequantAsym = 2 };

// 16 nibbles (8 bytes, low nibble = even index) -> 16 bytes in index order; SIGNED: two's-complement nibbles
// are sign-extended (the weights), otherwise they stay 0..15 (the activations).
template <bool SIGNED>
__device__ __forceinline__ i32x4 unpack16_nibbles(uint2 p) {
    i32x4 r;
    const uint32_t src[2] = {p.x, p.y};
#pragma unroll
    for (int h = 0; h < 2; h++) {
        uint32_t lo = src[h] & 0x0F0F0F0Fu, hi = (src[h] >> 4) & 0x0F0F0F0Fu;       // elements 0,2,4,6 and 1,3,5,7
        if constexpr (SIGNED) {
            lo |= (lo & 0x08080808u) * 30u;                                          // 0x08 -> 0xF8: sign bits of the byte
            hi |= (hi & 0x08080808u) * 30u;
        }
        r[2 * h] = (int)__builtin_amdgcn_perm(hi, lo, 0x05010400u);                 // bytes lo0, hi0, lo1, hi1
        r[2 * h + 1] = (int)__builtin_amdgcn_perm(hi, lo, 0x07030602u);             // bytes lo2, hi2, lo3, hi3
    }
    return r;
}

// PACKED: both operands hold two 4-bit values per byte (rows of k/2 bytes; activations unsigned, weights signed);
// they are widened to int8 between the global load and the LDS store, the MFMA path is the same.
template <int BM, int BN, int EPI, int D, bool PACKED = false>
__global__ __launch_bounds__(256) void gemm_i8_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ w,
                                                      int32_t* __restrict__ c_out, const float* __restrict__ s_x,
                                                      const float* __restrict__ w_s, const float* __restrict__ residual,
                                                      float* __restrict__ y, int m, int k, int n, int tiles_m, int tiles_n,
                                                      const float* __restrict__ b_x = nullptr, const float* __restrict__ w_sum = nullptr) {
    constexpr int WM = BM / 2, WN = BN / 2;          // wave tile
    constexpr int TM = WM / 32, TN = WN / 32;        // 32x32 MFMA tiles per wave
    constexpr int A_CHUNKS = BM * 4 / 256;           // 16-byte chunks per thread per stage
    constexpr int B_CHUNKS = BN * 4 / 256;
    constexpr int PA = gemm_plane(BM), PB = gemm_plane(BN);
    __shared__ __attribute__((aligned(16))) int8_t lds_a[2][4 * PA];
    __shared__ __attribute__((aligned(16))) int8_t lds_b[2][4 * PB];

    // XCD-aware tile order.  Consecutive workgroup ids land on different XCDs (8 of them, each with its own
    // 4 MiB L2).  Give every XCD a contiguous range of weight columns and walk the token-row tiles fastest,
    // so that a weight block is fetched from HBM by one XCD only and is shared there by all token-row tiles
    // (the activations, M x K, are small and are read by every XCD).
    int tm, tn;
    if ((tiles_n & 7) == 0) {
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        tn = xcd * (tiles_n >> 3) + idx / tiles_m;
        tm = idx % tiles_m;
    } else {
        tm = blockIdx.x / tiles_n;
        tn = blockIdx.x % tiles_n;
    }
    const int row0 = tm * BM, col0 = tn * BN;

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;

    // global -> register staging: chunk id c = t + 256*i -> row c/4, 16-byte column c%4.  D k-steps of global
    // loads are kept in flight in registers (an L2/HBM round trip is several k-steps long).
    i32x4 ra[D][A_CHUNKS], rb[D][B_CHUNKS];
    const int8_t* a_ptr[A_CHUNKS];
    const int8_t* b_ptr[B_CHUNKS];
#pragma unroll
    for (int i = 0; i < A_CHUNKS; i++) {
        const int c = t + 256 * i;
        a_ptr[i] = PACKED ? a + (size_t)min(row0 + (c >> 2), m - 1) * (k >> 1) + (c & 3) * 8
                          : a + (size_t)min(row0 + (c >> 2), m - 1) * k + (c & 3) * 16;
    }
#pragma unroll
    for (int i = 0; i < B_CHUNKS; i++) {
        const int c = t + 256 * i;
        b_ptr[i] = PACKED ? w + (size_t)min(col0 + (c >> 2), n - 1) * (k >> 1) + (c & 3) * 8
                          : w + (size_t)min(col0 + (c >> 2), n - 1) * k + (c & 3) * 16;
    }
    auto load_global = [&](int k0, i32x4 (&xa)[A_CHUNKS], i32x4 (&xb)[B_CHUNKS]) {
#pragma unroll
        for (int i = 0; i < A_CHUNKS; i++) {
            if constexpr (PACKED) xa[i] = unpack16_nibbles<false>(*reinterpret_cast<const uint2*>(a_ptr[i] + (k0 >> 1)));
            else xa[i] = *reinterpret_cast<const i32x4*>(a_ptr[i] + k0);
        }
#pragma unroll
        for (int i = 0; i < B_CHUNKS; i++) {
            if constexpr (PACKED) xb[i] = unpack16_nibbles<true>(*reinterpret_cast<const uint2*>(b_ptr[i] + (k0 >> 1)));
            else xb[i] = *reinterpret_cast<const i32x4*>(b_ptr[i] + k0);
        }
    };
    auto store_lds = [&](int buf, const i32x4 (&xa)[A_CHUNKS], const i32x4 (&xb)[B_CHUNKS]) {
#pragma unroll
        for (int i = 0; i < A_CHUNKS; i++) {
            const int c = t + 256 * i;
            *reinterpret_cast<i32x4*>(&lds_a[buf][(c & 3) * PA + (c >> 2) * 16]) = xa[i];
        }
#pragma unroll
        for (int i = 0; i < B_CHUNKS; i++) {
            const int c = t + 256 * i;
            *reinterpret_cast<i32x4*>(&lds_b[buf][(c & 3) * PB + (c >> 2) * 16]) = xb[i];
        }
    };

    i32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

    const int nk = k / kGemmBK;            // a multiple of D (checked by the launcher)
#pragma unroll
    for (int d = 0; d < D; d++)
        if (d < nk) load_global(d * kGemmBK, ra[d], rb[d]);
    store_lds(0, ra[0], rb[0]);
    __syncthreads();
    const int frag_row = (lane & 31) * 16, frag_g = lane >> 5;
    for (int kt0 = 0; kt0 < nk; kt0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int kt = kt0 + d;
            const int buf = kt & 1;
            // slot d held k-step kt, which is already in LDS: refill it with k-step kt+D
            if (kt + D < nk) load_global((kt + D) * kGemmBK, ra[d], rb[d]);
#pragma unroll
            for (int ks = 0; ks < kGemmBK / 32; ks++) {
                i32x4 fa[TM], fb[TN];
#pragma unroll
                for (int i = 0; i < TM; i++)
                    fa[i] = *reinterpret_cast<const i32x4*>(&lds_a[buf][(ks * 2 + frag_g) * PA + (wm + i * 32) * 16 + frag_row]);
#pragma unroll
                for (int j = 0; j < TN; j++)
                    fb[j] = *reinterpret_cast<const i32x4*>(&lds_b[buf][(ks * 2 + frag_g) * PB + (wn + j * 32) * 16 + frag_row]);
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
            }
            if (kt + 1 < nk) {
                store_lds(buf ^ 1, ra[(d + 1) % D], rb[(d + 1) % D]);   // the other buffer was last read before the previous barrier
                __syncthreads();
            }
        }
    }

    // epilogue: 32x32 accumulator layout - lane l holds column l%32, register r holds row 8*(r/4) + 4*(l/32) + r%4
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = col0 + wn + j * 32 + (lane & 31);
            if (col >= n) continue;
            float ws = 0.0f, wsm = 0.0f;
            if constexpr (EPI != kGemmRaw) ws = w_s[col];
            if constexpr (EPI == kGemmDequantAsym) wsm = w_sum[col];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = row0 + wm + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (row >= m) continue;
                if constexpr (EPI != kGemmRaw) {
                    float v = (float)acc[i][j][r] * s_x[row] * ws;
                    if constexpr (EPI == kGemmDequantAsym) v = v + b_x[row] * wsm;      // zero point times the row sum of W
                    if (residual) v = v + residual[(size_t)row * n + col];
                    y[(size_t)row * n + col] = v;
                } else {
                    c_out[(size_t)row * n + col] = acc[i][j][r];
                }
            }
        }
}

// ---------------------------------------------------------------------------------------------------------
// Second kernel: tiles go global -> LDS by direct loads (global_load_lds_dwordx4), bypassing registers, two to four
// stages deep.  Tile BM x BN, BKB = 64 or 128 k-bytes per row and stage, four waves (2x2) or eight (2x4); the wave tile is a grid of 32x32 MFMA tiles, and the wider it is the more MFMAs every fragment
// read from LDS feeds (a 128x64 wave tile: six reads for eight MFMAs).
//
// LDS stage layout: row-major, BKB bytes (= BKB/16 16-byte k-chunks) per tile row.  A direct load writes lane i
// at base + 16*i, i.e. 64/(BKB/16) rows per instruction, which is also the coalesced order in global memory.  To
// keep the MFMA fragment reads (32 rows x one chunk) free of bank conflicts the chunks of a row are stored rotated:
// slot s of row r holds k-chunk s ^ ((r >> 2) & 3) for 64-byte rows, s ^ ((r >> 1) & 7) for 128-byte rows.  The
// rotation is applied on the global side of the direct load (the LDS side is fixed by the hardware).
//
// The loads are issued from inline assembly: the compiler does not track them, so the k-loop waits for them
// with explicit counters (results return in issue order).
enum GemmDmaEpi { kDmaRaw = 0, kDmaDequant = 1, kDmaSwiglu = 2, kDmaQkv = 3, kDmaDequantAsym = 4, kDmaSwigluAsym = 5 };

// The stage ring, or the epilogue: a patch per wave, for q/k/v the dequantised tile.
__host__ __device__ constexpr int gemm_dma_lds_bytes(int bm, int bn, int stages, int bkb, int nw, int epilogue) {
    const int ring = stages * (bm + bn) * bkb, epi = epilogue == kDmaQkv ? bm * (bn + 1) * 4 : nw * 32 * 36 * 4;
    return ring > epi ? ring : epi;
}

// Arguments of the q/k/v epilogue: 64 columns of the fused [q | k | v] projection are one attention head, a tile holds whole heads,
// so RoPE (pairs k, k+32), the static int8 quantisation and the store into q8 / the K cache / the transposed V
// cache blocks all happen on the tile, 64 tokens x 64 channels at a time (a V cache block is 64 positions x 64 channels).
struct QkvEpiArgs {
    const float *sin_t = nullptr, *cos_t = nullptr, *q_s = nullptr, *k_s = nullptr, *v_s = nullptr;
    int8_t *q8 = nullptr, *kc = nullptr, *vc = nullptr;
    int pos0 = 0, q_heads = 0, kv_heads = 0, max_pos = 0;
    // asymmetric activations (kDmaDequantAsym / kDmaSwigluAsym; optional for kDmaQkv, null = symmetric): zero point per
    // row, weight row sum (times its scale) per column
    const float *b_x = nullptr, *w_sum = nullptr;
};

// q/k/v from the dequantised tile [BM tokens][BN channels], pitch BN + 1: RoPE, static quantisation, the stores into q8 and the caches.
template <int BM, int BN, int NW>
__device__ __forceinline__ void qkv_tile_out(const float* tile, int row0, int col0, int m, int n, const QkvEpiArgs& qa) {
    constexpr int TP = BN + 1;
    const int t = threadIdx.x;
    // four waves at a time take a block of 64 tokens x one head
    constexpr int HM = BM / 64, HN = BN / 64, TEAMS = NW / 4;
    const int sel = t & 63, part = (t >> 6) & 3;
    for (int blk = t >> 8; blk < HM * HN; blk += TEAMS) {
        const int tr = (blk % HM) * 64, tc = (blk / HM) * 64, head = (col0 + tc) / kHd;      // 0..q_heads-1 q, then k heads, then v heads
        if (col0 + tc >= n) break;
        const float* sub = tile + tr * TP + tc;
        if (head < qa.q_heads + qa.kv_heads) {
            // RoPE + static quantisation: thread = (token sel, pairs 8*part .. 8*part+7)
            const int row = row0 + tr + sel, pos = qa.pos0 + row;
            if (row < m) {
                const bool is_q = head < qa.q_heads;
                const int hk = is_q ? head : head - qa.q_heads;
                const float div = is_q ? 8.0f * qa.q_s[hk] : 1.0f * qa.k_s[hk];     // sqrt(head_dim) folded into the Q scale
                const float* sn = qa.sin_t + (size_t)pos * 32 + part * 8;
                const float* cs = qa.cos_t + (size_t)pos * 32 + part * 8;
                uint32_t lo[2] = {0, 0}, hi[2] = {0, 0};
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float t0 = sub[sel * TP + part * 8 + j], t1 = sub[sel * TP + part * 8 + j + 32];
                    const float o0 = t0 * cs[j] - t1 * sn[j];
                    const float o1 = t0 * sn[j] + t1 * cs[j];
                    lo[j >> 2] |= (uint32_t)(static_q8(o0, div) & 0xff) << (8 * (j & 3));
                    hi[j >> 2] |= (uint32_t)(static_q8(o1, div) & 0xff) << (8 * (j & 3));
                }
                int8_t* dst = is_q ? qa.q8 + ((size_t)row * qa.q_heads + hk) * kHd : qa.kc + k_index(hk, pos, qa.max_pos);
                *reinterpret_cast<uint2*>(dst + part * 8) = make_uint2(lo[0], lo[1]);
                *reinterpret_cast<uint2*>(dst + part * 8 + 32) = make_uint2(hi[0], hi[1]);
            }
        } else {
            // V: thread = (channel sel, 16 consecutive positions 16*part ..): one 16-byte run of the transposed cache block
            const int hv = head - qa.q_heads - qa.kv_heads;
            const int rbase = row0 + tr + part * 16;
            if (rbase < m) {                               // m is a multiple of 32 (checked by the launcher)
                const float div = 1.0f * qa.v_s[hv];
                uint32_t wv4[4] = {0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < 16; i++)
                    wv4[i >> 2] |= (uint32_t)(static_q8(sub[(part * 16 + i) * TP + sel], div) & 0xff) << (8 * (i & 3));
                *reinterpret_cast<uint4*>(qa.vc + v_index(hv, qa.pos0 + rbase, sel, qa.max_pos)) = make_uint4(wv4[0], wv4[1], wv4[2], wv4[3]);
            }
        }
    }
}

__device__ __forceinline__ void gemm_dma_issue(const int8_t* base, unsigned voff, unsigned lds_dst) {
    unsigned saved_m0;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %3\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved_m0) : "v"(voff), "s"(base), "s"(lds_dst) : "memory");
}

template <int N>
__device__ __forceinline__ void gemm_wait_vmcnt() {            // s_waitcnt vmcnt(N) only; the count is a 6-bit split immediate
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// kDmaStages LDS stages; WPE = waves per SIMD the register allocation has to leave room for.
// BKB = k-bytes of a row per stage, 64 or 128.  A 64-byte segment is half a cache line, and the other half is asked
// for again one stage later: measured with the loads alone (no math, 128 x 256 tiles at K = 2048), the chip moves
// 23 TB/s into LDS in whole 128-byte lines and 14.5 TB/s in halves.  With 128-byte rows the slot rotation is
// s ^ ((r >> 1) & 7): two rows span the 64 banks, so 16 consecutive rows of one chunk fall on 16 different bank groups.
// NW = waves per workgroup, 4 (2x2 wave grid) or 8 (2x4).
template <int BM, int BN, int EPI, int kDmaStages, int WPE, int BKB, int NW>   // at most 4 stages (the wait below distinguishes up to 2 younger ones)
__global__ __launch_bounds__(NW * 64, WPE) void gemm_i8_dma_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ w,
                                                          int32_t* __restrict__ c_out, const float* __restrict__ s_x,
                                                          const float* __restrict__ w_s, const float* __restrict__ residual,
                                                          float* __restrict__ y, int m, int k, int n, int tiles_m, int tiles_n,
                                                          QkvEpiArgs qa) {
    static_assert(NW == 4 || NW == 8, "four or eight waves");
    constexpr int WGN = NW / 2;                               // waves along N
    constexpr int WM = BM / 2, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    static_assert(BKB == 64 || BKB == 128, "64 or 128 k-bytes per row and stage");
    constexpr int CPR = BKB / 16, RPI = 64 / CPR;             // 16-byte chunks per row; rows per direct load (1 KiB)
    constexpr int A_INSTR = BM / (NW * RPI), B_INSTR = BN / (NW * RPI);   // direct loads per wave per stage
    static_assert(A_INSTR >= 1 && B_INSTR >= 1 && TM >= 1 && TN >= 1, "tile too small for this wave count");
    constexpr int STAGE = (BM + BN) * BKB, KS = BKB / 32;     // KS MFMA k-steps per stage
    auto rot = [](int r) { return BKB == 64 ? (r >> 2) & 3 : (r >> 1) & 7; };
    extern __shared__ __attribute__((aligned(16))) int8_t gemm_smem[];

    int tm, tn;
    if ((tiles_n & 7) == 0) {                                  // see gemm_i8_kernel: one range of weight columns per XCD
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        tn = xcd * (tiles_n >> 3) + idx / tiles_m;
        tm = idx % tiles_m;
    } else {
        tm = blockIdx.x / tiles_n;
        tn = blockIdx.x % tiles_n;
    }
    int row0 = tm * BM, col0 = tn * BN;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
    int8_t* const ring = gemm_smem;

    // per-lane global offsets of this wave's direct loads (without the k offset, which is uniform)
    unsigned offa[A_INSTR], offb[B_INSTR];
#pragma unroll
    for (int j = 0; j < A_INSTR; j++) {
        const int r = (wave * A_INSTR + j) * RPI + lane / CPR;
        offa[j] = (unsigned)min(row0 + r, m - 1) * (unsigned)k + (unsigned)(((lane % CPR) ^ rot(r)) * 16);
    }
#pragma unroll
    for (int j = 0; j < B_INSTR; j++) {
        const int r = (wave * B_INSTR + j) * RPI + lane / CPR;
        offb[j] = (unsigned)min(col0 + r, n - 1) * (unsigned)k + (unsigned)(((lane % CPR) ^ rot(r)) * 16);
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)ring;
    auto issue_stage = [&](int kt) {
        const unsigned sb = lds0 + (unsigned)(kt % kDmaStages) * STAGE;
        const size_t koff = (size_t)kt * BKB;
#pragma unroll
        for (int j = 0; j < A_INSTR; j++) gemm_dma_issue(a + koff, offa[j], sb + (wave * A_INSTR + j) * 1024);
#pragma unroll
        for (int j = 0; j < B_INSTR; j++) gemm_dma_issue(w + koff, offb[j], sb + BM * BKB + (wave * B_INSTR + j) * 1024);
    };

    i32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

    const int nk = k / BKB;                                    // the launcher checks divisibility
    constexpr int PER = A_INSTR + B_INSTR;                     // direct loads per wave per stage
#pragma unroll
    for (int s0 = 0; s0 < kDmaStages - 1; s0++)
        if (s0 < nk) issue_stage(s0);
    // fragment addressing: lane l reads row (l % 32) of a 32-row tile, k-chunk 2*ks + l/32, from its rotated slot
    const int fr = lane & 31, fg = lane >> 5;
    auto read_frags = [&](int kt, int ks, i32x4 (&fa)[TM], i32x4 (&fb)[TN]) {
        const int8_t* sa = ring + (kt % kDmaStages) * STAGE;
        const int8_t* sb = sa + BM * BKB;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int r = wm + i * 32 + fr;
            fa[i] = *reinterpret_cast<const i32x4*>(sa + r * BKB + (((ks * 2 + fg) ^ rot(r)) * 16));
        }
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int r = wn + j * 32 + fr;
            fb[j] = *reinterpret_cast<const i32x4*>(sb + r * BKB + (((ks * 2 + fg) ^ rot(r)) * 16));
        }
    };
    auto mma = [&](const i32x4 (&fa)[TM], const i32x4 (&fb)[TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
    };
    static_assert(kDmaStages <= 4 && 2 * PER < 64, "the wait distinguishes up to two younger stages");
    // stage kt has landed once only the younger stages in flight remain outstanding
    auto wait_stage = [&](int kt) {
        const int younger = min(kDmaStages - 2, nk - 1 - kt);
        if (younger >= 2) gemm_wait_vmcnt<2 * PER>();
        else if (younger == 1) gemm_wait_vmcnt<PER>();
        else gemm_wait_vmcnt<0>();
    };

    // Software pipeline over k-steps of 32 bytes: the fragments of the next k-step are read from LDS before the
    // MFMAs of the current one are issued, so the LDS latency runs under matrix work.  The workgroup barrier
    // sits before the last k-step of a stage: after it stage kt+1 is complete in LDS and every wave has finished
    // reading stage kt, whose buffer the direct loads of the iteration after next overwrite.
    i32x4 fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    wait_stage(0);
    __syncthreads();
    read_frags(0, 0, fa0, fb0);
    // The last stage stands by itself, a branch less in the loop: 13 x 312 x 5888 14.5 -> 12.1 us, 451 x 280 x 11904 26.8 -> 21.9 us.
    auto stage = [&](int kt, auto more) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < KS; ks += 2) {
            read_frags(kt, ks + 1, fa1, fb1);
            if (more && ks == 0 && kt + kDmaStages - 1 < nk) issue_stage(kt + kDmaStages - 1);   // into the buffer that held stage kt-1
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

    // Epilogue.  In the accumulator layout a lane holds ONE column (l%32) and 16 rows of a 32x32 tile, so direct
    // stores would be 4 bytes per lane.  Each wave instead turns its tiles through a private LDS patch
    // (32 x 36 words) and then owns 4 consecutive columns of a row: 16-byte loads of the residual, 16-byte stores
    // (8 bytes for the SiLU*up pairs), 128 contiguous bytes per row.
    __syncthreads();                                           // all waves are done with the stage buffers
    if constexpr (EPI == kDmaQkv) {
        static_assert(BM % 64 == 0 && BN % 64 == 0 && NW % 4 == 0, "blocks of 64 tokens x one head");
        constexpr int TP = BN + 1;                             // odd pitch: a column walk hits every bank once
        float* tile = reinterpret_cast<float*>(gemm_smem);     // dequantised tile [BM tokens][BN channels]
        const bool asym = qa.b_x != nullptr;                  // asymmetric activations: + zero point x row sum of the dequantised weights
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int cl = wn + j * 32 + (lane & 31), col = min(col0 + cl, n - 1);
            const float ws = w_s[col];
            const float wq = asym ? qa.w_sum[col] : 0.0f;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int lr = wm + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                    const int row = min(row0 + lr, m - 1);
                    float v = (float)acc[i][j][r] * s_x[row] * ws;
                    if (asym) v = v + qa.b_x[row] * wq;
                    tile[lr * TP + cl] = v;
                }
        }
        __syncthreads();
        qkv_tile_out<BM, BN, NW>(tile, row0, col0, m, n, qa);
        return;
    }
    constexpr bool kAsym = EPI == kDmaDequantAsym || EPI == kDmaSwigluAsym;      // + zero point x row sum of the dequantised weights
    constexpr bool kPlain = EPI == kDmaDequant || EPI == kDmaDequantAsym;        // fp32 outputs (+ residual); else SiLU(gate) * up pairs
    constexpr int EP = 36;                                     // patch pitch in words (rows stay 16-byte aligned)
    int* patch = reinterpret_cast<int*>(gemm_smem) + wave * (32 * EP);
    const int pr = lane >> 3, pc = (lane & 7) * 4;             // row within a group of 8, first of this lane's 4 columns
    // Every scale this lane needs is loaded before the first tile: a load inside the tile loop would be waited for
    // together with the stores issued before it (one counter covers both), once per group of rows.
    float sxv[TM][4];
    float4 wsv[TN];
    float bxv[kAsym ? TM : 1][4];
    float4 wsumv[kAsym ? TN : 1];
    if constexpr (EPI != kDmaRaw) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int p = 0; p < 4; p++) sxv[i][p] = s_x[min(row0 + wm + i * 32 + p * 8 + pr, m - 1)];
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = col0 + wn + j * 32 + pc;
            wsv[j] = col < n ? *reinterpret_cast<const float4*>(w_s + col) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    if constexpr (kAsym) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int p = 0; p < 4; p++) bxv[i][p] = qa.b_x[min(row0 + wm + i * 32 + p * 8 + pr, m - 1)];
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = col0 + wn + j * 32 + pc;
            wsumv[j] = col < n ? *reinterpret_cast<const float4*>(qa.w_sum + col) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int col = col0 + wn + j * 32 + pc;               // n is a multiple of 4 (checked by the launcher)
        const bool col_ok = col < n;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            float4 rs[4];                                      // the tile's residual rows, in flight during the turn through LDS
            bool has_res = false;
            if constexpr (kPlain) {
                has_res = residual != nullptr;
                if (has_res) {
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        const int row = row0 + wm + i * 32 + p * 8 + pr;
                        rs[p] = col_ok && row < m ? *reinterpret_cast<const float4*>(residual + (size_t)row * n + col)
                                                  : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++)
                patch[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * EP + (lane & 31)] = acc[i][j][r];
            // the patch is private to the wave: the LDS operations of a wave complete in order, the compiler is kept from
            // moving them across this point
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // One explicit wait per tile, outside the guarded stores: the scales (first tile) and this tile's residual
            // rows have landed.  Left to the compiler the wait sits behind the store guards, is repeated for every group
            // of rows, and then also waits for the store issued just before it.
            if constexpr (EPI != kDmaRaw) { if ((i == 0 && j == 0) || has_res) gemm_wait_vmcnt<0>(); }
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const int lr = p * 8 + pr;
                const int row = row0 + wm + i * 32 + lr;
                const i32x4 v = *reinterpret_cast<const i32x4*>(patch + lr * EP + pc);
                // the arithmetic runs for every lane and only the store is guarded: a wait placed behind a branch
                // would be repeated at every later use, and there it would also wait for the stores in between
                const bool ok = col_ok && row < m;
                if constexpr (EPI == kDmaRaw) {
                    if (ok) *reinterpret_cast<i32x4*>(c_out + (size_t)row * n + col) = v;
                } else {
                    const float sx = sxv[i][p];
                    const float4 ws = wsv[j];
                    float4 o;
                    o.x = (float)v[0] * sx * ws.x; o.y = (float)v[1] * sx * ws.y;
                    o.z = (float)v[2] * sx * ws.z; o.w = (float)v[3] * sx * ws.w;
                    if constexpr (kAsym) {
                        const float bx = bxv[i][p];
                        const float4 wq = wsumv[j];
                        o.x = o.x + bx * wq.x; o.y = o.y + bx * wq.y; o.z = o.z + bx * wq.z; o.w = o.w + bx * wq.w;
                    }
                    if constexpr (kPlain) {
                        if (has_res) { o.x = o.x + rs[p].x; o.y = o.y + rs[p].y; o.z = o.z + rs[p].z; o.w = o.w + rs[p].w; }
                        if (ok) *reinterpret_cast<float4*>(y + (size_t)row * n + col) = o;
                    } else {
                        // weight rows are interleaved (2c gate, 2c+1 up): columns (col, col+1) and (col+2, col+3) are pairs
                        float2 h;
                        h.x = o.y * silu_f(o.x);
                        h.y = o.w * silu_f(o.z);
                        if (ok) *reinterpret_cast<float2*>(y + (size_t)row * (n >> 1) + (col >> 1)) = h;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();               // reads of this tile before the next tile's writes
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}

template <int BM, int BN, int EPI, int STAGES, int WPE, int BKB, int NW = 4>
inline int launch_gemm_dma(const int8_t* a, const int8_t* w, int32_t* c, const float* s_x, const float* w_s,
                           const float* residual, float* y, int m, int k, int n, hipStream_t st, QkvEpiArgs qa = QkvEpiArgs()) {
    static std::atomic<bool> opted_in{false};             // more than the default 64 KiB of LDS per workgroup
    if (!opted_in.load(std::memory_order_acquire)) {   // idempotent: two threads racing here both set the same attribute
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_i8_dma_kernel<BM, BN, EPI, STAGES, WPE, BKB, NW>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, gemm_dma_lds_bytes(BM, BN, STAGES, BKB, NW, EPI)));
        opted_in.store(true, std::memory_order_release);
    }
    const int tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
    gemm_i8_dma_kernel<BM, BN, EPI, STAGES, WPE, BKB, NW><<<tm * tn, NW * 64, gemm_dma_lds_bytes(BM, BN, STAGES, BKB, NW, EPI), st>>>(a, w, c, s_x, w_s, residual, y, m, k, n, tm, tn, qa);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// static_q8 (attn_decode_kernels.h) of four values that share a divisor, without a division each, packed.  quant_vector rounds as the quotient does up to
// 255; what is beyond is clamped either way.
__device__ __forceinline__ uint32_t static_q8x4(const float (&v)[4], float div) {
    int n[4];
    quant_vector<4>(v, div, n);
#pragma unroll
    for (int e = 0; e < 4; e++) n[e] = max(min(n[e], 127), -128);
    return pack4_i8(n[0], n[1], n[2], n[3]);
}

// Tiles of 256 columns, 128-byte rows: the walk of gemm_walk.h.  Before (gemm_i8_dma_kernel, eight waves of 32 x 32 instructions) and now, us:
// 2528 x 16384 x 2048 (m, n, k) 110 and 101, 1531 x 16384 x 2048 69 and 64, 2528 x 2048 x 8192 58.2 and 53.8, 4096 x 2048 x 8192 74 and 62,
// 1024 x 16384 x 2048 with the gated unit 43.8 and 38.  A product of a short k is bound by what stands around the walk: of
// 2528 x 16384 x 2048's 100 us three rounds take 19 us of walk each (16 stages of 0.8 us), the rest are the first stages' trips and the
// outputs.  Smaller tiles stay on the other kernel, whose eight waves hide more of each other's trips (1024 x 2048 x 8192 on
// 64 x 128 28.5 us, 28.6 here; on 128 x 128 34.6 and 38.3).
template <int MI> using WideI8 = GemmWalk<int8_t, 2, MI, 8, MI == 4 ? 4 : 3, MI == 4 ? 3 : 2>;      // 32 * MI rows

template <int EPI, int MI>
__global__ __launch_bounds__(256, WideI8<MI>::per_cu()) void gemm_i8_walk_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ w, int32_t* __restrict__ c_out,
                                                                                 const float* __restrict__ s_x, const float* __restrict__ w_s, const float* __restrict__ residual,
                                                                                 float* __restrict__ y, int m, int k, int n, int tiles_m, int tiles_n, QkvEpiArgs qa) {
    using W = WideI8<MI>;
    constexpr int NI = 8;
    extern __shared__ __attribute__((aligned(16))) int8_t gemm_smem[];
    int tm, tn;
    gemm_tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int row0 = tm * W::BM, col0 = tn * W::BN;
    unsigned offa[W::AI], offb[W::BI];
#pragma unroll
    for (int j = 0; j < W::AI; j++) {
        const int r = W::load_row_a(j);
        offa[j] = (unsigned)min(row0 + r, m - 1) * (unsigned)k + W::load_byte(r);
    }
#pragma unroll
    for (int j = 0; j < W::BI; j++) {
        const int r = W::load_row_b(j);
        offb[j] = (unsigned)min(col0 + r, n - 1) * (unsigned)k + W::load_byte(r);
    }
    i32x4 acc[MI][NI];
    W::run(a, w, offa, offb, k / 128, gemm_smem, acc, OneTile());
    const int lane = threadIdx.x & 63, fr = lane & 15, fg = lane >> 4;
    const int wr = W::row_of_wave(), wc = W::col_of_wave();
    if constexpr (EPI == kDmaQkv) {
        // A wave has 64 tokens x two heads.  Channels c and c + 32 of a token are in blocks j and j + 2 of one lane, so RoPE stays in registers, and
        // the quantised head of a token leaves in 16-byte pieces.  Everything that has to be read is asked for at once: one wave per SIMD
        // waits for each trip (2528 x 3072 x 2048, asked for token by token 34.4 us, 32.0 so).
        static_assert(MI == 4 && NI == 8, "64 tokens x two heads per wave");
        constexpr int TP = 64 + 16, HEADS = 2;                 // TP: V only, a head's bytes [channel][token], turned through LDS
        int8_t* const turn = gemm_smem + W::wave() * (64 * TP);
        const bool asym = qa.b_x != nullptr;                   // asymmetric activations: + zero point x row sum of the dequantised weights
        f32x4 sn[MI][2], cs[MI][2], ws[HEADS][4], wq[HEADS][4];
        float sx[MI], bx[MI];
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const int r = min(row0 + wr + i * 16 + fr, m - 1);
            sx[i] = s_x[r];
            bx[i] = asym ? qa.b_x[r] : 0.0f;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                sn[i][j] = *reinterpret_cast<const f32x4*>(qa.sin_t + (size_t)(qa.pos0 + r) * 32 + j * 16 + fg * 4);
                cs[i][j] = *reinterpret_cast<const f32x4*>(qa.cos_t + (size_t)(qa.pos0 + r) * 32 + j * 16 + fg * 4);
            }
        }
#pragma unroll
        for (int hh = 0; hh < HEADS; hh++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int c = min(col0 + wc + hh * 64 + j * 16 + fg * 4, n - 4);
                ws[hh][j] = *reinterpret_cast<const f32x4*>(w_s + c);
                wq[hh][j] = asym ? *reinterpret_cast<const f32x4*>(qa.w_sum + c) : f32x4{};
            }
        __syncthreads();                                       // all waves are done with the stage buffers
#pragma unroll
        for (int hh = 0; hh < HEADS; hh++) {
            const int c0 = col0 + wc + hh * 64, head = c0 / kHd;      // 0..q_heads-1 q, then k heads, then v heads
            if (c0 >= n) break;
            const bool is_q = head < qa.q_heads, is_v = head >= qa.q_heads + qa.kv_heads;
            const int hk = is_q ? head : is_v ? head - qa.q_heads - qa.kv_heads : head - qa.q_heads;
            const float div = is_q ? 8.0f * qa.q_s[hk] : is_v ? 1.0f * qa.v_s[hk] : 1.0f * qa.k_s[hk];     // sqrt(head_dim) folded into the Q scale
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int row = row0 + wr + i * 16 + fr, pos = qa.pos0 + row;
                f32x4 v[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[j][e] = (float)acc[i][hh * 4 + j][e] * sx[i] * ws[hh][j][e];
                    if (asym) v[j] = v[j] + bx[i] * wq[hh][j];
                }
                if (is_v) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float x[4] = {v[j][0], v[j][1], v[j][2], v[j][3]};
                        const uint32_t q = static_q8x4(x, div);
#pragma unroll
                        for (int e = 0; e < 4; e++) turn[(j * 16 + fg * 4 + e) * TP + i * 16 + fr] = (int8_t)(q >> (8 * e));
                    }
                    continue;
                }
                uint32_t o[4][1];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    float lo[4], hi[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        lo[e] = v[j][e] * cs[i][j][e] - v[j + 2][e] * sn[i][j][e];
                        hi[e] = v[j][e] * sn[i][j][e] + v[j + 2][e] * cs[i][j][e];
                    }
                    o[j][0] = static_q8x4(lo, div);
                    o[j + 2][0] = static_q8x4(hi, div);
                }
                join_blocks<1>(o);
                int8_t* dst = is_q ? qa.q8 + ((size_t)row * qa.q_heads + hk) * kHd : qa.kc + k_index(hk, pos, qa.max_pos);
                if (row < m) *reinterpret_cast<uint4*>(dst + fg * 16) = make_uint4(o[0][0], o[1][0], o[2][0], o[3][0]);
            }
            if (is_v) {
                // the patch is private to the wave, whose LDS operations complete in order
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                // lane = channel; 16 consecutive positions are one run of the transposed cache block
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const int row = row0 + wr + p * 16;            // m is a multiple of 32 (checked by the launcher)
                    const uint4 run = *reinterpret_cast<const uint4*>(turn + lane * TP + p * 16);
                    if (row < m) *reinterpret_cast<uint4*>(qa.vc + v_index(hk, qa.pos0 + row, lane, qa.max_pos)) = run;
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
        return;
    } else {
        constexpr bool kAsym = EPI == kDmaDequantAsym || EPI == kDmaSwigluAsym, kUnit = EPI == kDmaSwiglu || EPI == kDmaSwigluAsym;
        constexpr int J = kUnit ? 2 : 1;                       // blocks of 16 columns whose outputs leave together, 64 bytes of a row
        const int rows = m - row0 - wr, ld = kUnit ? n >> 1 : n;
        const TileRows out(EPI == kDmaRaw ? reinterpret_cast<float*>(c_out) + (size_t)(row0 + wr) * ld : y + (size_t)(row0 + wr) * ld, rows, MI * 16, ld * 4);
        const bool has_res = !kUnit && EPI != kDmaRaw && residual != nullptr;
        const TileRows res(const_cast<float*>(has_res ? residual + (size_t)(row0 + wr) * n : y), has_res ? rows : 0, MI * 16, n * 4);
        float sx[MI], bx[MI];
        if constexpr (EPI != kDmaRaw) {
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int row = min(row0 + wr + i * 16 + fr, m - 1);
                sx[i] = s_x[row];
                if constexpr (kAsym) bx[i] = qa.b_x[row];
            }
        }
        // byte of the lane's 16 in the tile's first row.  They lie inside or behind the row as a whole, or (a unit whose rows end in the middle: it
        // makes them of eight columns, and n is a multiple of 4) their first half does: that leaves by itself.
        constexpr int PC = kUnit ? 8 : 4;                      // columns that 16 bytes of output are made of
        auto place = [&](int j0, int cols) __attribute__((always_inline)) {
            const int col = col0 + wc + j0 * 16 + fg * PC;
            return col + cols <= n ? (kUnit ? col * 2 : col * 4) + fr * ld * 4 : kNowhere;
        };
        // residuals of the next columns are asked for ahead of the stores of these: a wait for loads is one for the stores before them, too
        f32x4 rs[2][MI];
        auto residuals = [&](int j0) __attribute__((always_inline)) {
            const int at = place(j0, PC);
#pragma unroll
            for (int i = 0; i < MI; i++) rs[(j0 / J) & 1][i] = res.get(at == kNowhere ? kNowhere : at + i * 16 * ld * 4);
        };
        auto columns = [&](int j0, auto ends) __attribute__((always_inline)) {      // ends: the first halves of those 16 bytes that the row ends in
            constexpr bool kEnds = decltype(ends)::value;
            f32x4 ws[J], wq[J];
            const int at = kEnds && place(j0, PC) != kNowhere ? kNowhere : place(j0, kEnds ? 4 : PC);
#pragma unroll
            for (int j = 0; j < J; j++) {
                const int c = min(col0 + wc + (j0 + j) * 16 + fg * 4, n - 4);
                if constexpr (EPI != kDmaRaw) ws[j] = *reinterpret_cast<const f32x4*>(w_s + c);
                if constexpr (kAsym) wq[j] = *reinterpret_cast<const f32x4*>(qa.w_sum + c);
            }
            if (has_res && j0 + J < NI) residuals(j0 + J);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MI; i++) {
                uint32_t o[J][4 / J];
#pragma unroll
                for (int j = 0; j < J; j++) {
                    const i32x4 q = acc[i][j0 + j];
                    if constexpr (EPI == kDmaRaw) {
                        __builtin_memcpy(o[j], &q, 16);
                    } else {
                        f32x4 v;
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = (float)q[e] * sx[i] * ws[j][e];
                        if constexpr (kAsym) v = v + bx[i] * wq[j];
                        if constexpr (kUnit) {
                            // weight rows are interleaved (2c gate, 2c+1 up)
                            const float h[2] = {v[1] * silu_f(v[0]), v[3] * silu_f(v[2])};
                            __builtin_memcpy(o[j], h, 8);
                        } else {
                            if (has_res) v = v + rs[(j0 / J) & 1][i];
                            __builtin_memcpy(o[j], &v, 16);
                        }
                    }
                }
                join_blocks<4 / J>(o);
                const int to = at == kNowhere ? kNowhere : at + i * 16 * ld * 4;
                if constexpr (kEnds) out.put_half(&o[0][0], to); else out.put(&o[0][0], to);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (has_res) residuals(0);
#pragma unroll
        for (int j0 = 0; j0 < NI; j0 += J) columns(j0, std::false_type());
        if constexpr (kUnit) {
            const int left = n - (col0 + wc);
            if ((left & 4) && left > 0 && left < NI * 16) {
#pragma unroll
                for (int j0 = 0; j0 < NI; j0 += J)
                    if (left / (J * 16) == j0 / J) columns(j0, std::true_type());
            }
        }
    }
}

template <int EPI, int MI>
inline int launch_gemm_walk(const int8_t* a, const int8_t* w, int32_t* c, const float* s_x, const float* w_s, const float* residual, float* y, int m, int k, int n,
                            hipStream_t st, QkvEpiArgs qa) {
    using W = WideI8<MI>;
    static std::atomic<bool> opted_in{false};
    if (!opted_in.load(std::memory_order_acquire)) {
        FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_i8_walk_kernel<EPI, MI>), hipFuncAttributeMaxDynamicSharedMemorySize, W::kLds));
        opted_in.store(true, std::memory_order_release);
    }
    const int tm = (m + W::BM - 1) / W::BM, tn = (n + W::BN - 1) / W::BN;
    gemm_i8_walk_kernel<EPI, MI><<<tm * tn, 256, W::kLds, st>>>(a, w, c, s_x, w_s, residual, y, m, k, n, tm, tn, qa);
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// The direct-load kernel runs on the tile whose rounds over the 256 CUs (per_cu at a time) cost least, in about 0.01 us: per stage, and
// once per round for what lies around them (first loads, epilogue).  Rows of a stage are whole 128-byte lines where k
// allows, 64 bytes where it is a multiple of 64 alone.
// 128-byte rows, measured against the fixed choices before (us): 512 x 16384 x 2048 43.8 -> 24.8 (128 x 256), 2048 x 2048 x 8192 62.7 -> 45.8
// (128 x 128), 2528 x 2048 x 8192 85.1 -> 65.1 (128 x 256), 1536 x 2048 x 8192 53.4 -> 41.3 (128 x 128), 4096 x 2048 x 8192 91.0 -> 80.4
// (128 x 256), 1024 x 2048 x 2048 12.1 -> 11.3 (64 x 128); 1024 x 16384 x 2048 stays on 256 x 256, 41.5.
// 64-byte rows, against 64 x 64 everywhere (us): 1024 x 8192 x 2112 41.6 -> 25.3 (128 x 256), 1024 x 16384 x 2112 85.2 -> 40.3 and
// 4096 x 16384 x 2112 427 -> 192 (256 x 256), 1024 x 2048 x 8256 42.1 -> 32.3 (64 x 128), 2048 x 2048 x 8256 95.9 -> 47.6 (128 x 128).
// A product of a short k is bound by the stores of its output: 917 x 19348 x 704 40.7 us on 128 x 256, 29.8 on 128 x 128; 3575 x 2548 x 192
// 26.2 us on 256 x 256, 17.1 on 64 x 64.
// 128 x 128 in four waves with two stages fits twice into a CU (per_cu): 3700 x 2064 x 8576, 493 tiles, 74.6 us in one round of it, 86.2 in
// two of the one with four stages.  64 x 64 with three stages fits three times: 1536 x 2048 x 2048, 768 tiles, 14.4 us in one
// round of it, 15.8 on 128 x 128; 393 x 9536 x 128 7.5 us, 9.5 on 128 x 128 twice per CU.  The q/k/v
// epilogue turns whole heads, for which small tiles are no better: 1024 x 3072 x 2048 stays on 128 x 128.
// The costs are the ones that lost least over 384 sizes (128-byte rows) and 136 sizes (64-byte rows) of 1 to 4096 rows and 64 to 14336 k with
// every tile on this kernel (0.6 and 0.2 % from the best ones on average); with the wide ones on the walk it is 3.4 % over 44 sizes, most of it
// at k below 1152.
struct GemmI8Tile { int bm, bn, stage, round, per_cu; };
constexpr GemmI8Tile kGemmI8Tiles[2][7] = {
    {{256, 256, 126, 2000, 1}, {128, 256, 81, 1140, 1}, {128, 128, 74, 400, 1}, {64, 128, 60, 410, 1}, {64, 64, 27, 450, 1}, {64, 64, 77, 350, 3}, {128, 128, 112, 950, 2}},
    {{256, 256, 40, 1640, 1}, {128, 256, 29, 1180, 1}, {128, 128, 25, 260, 1}, {64, 128, 18, 390, 1}, {64, 64, 13, 70, 1}, {}, {}}};
inline int gemm_i8_tile(int m, int k, int n, bool qkv) {
    const bool half = k % 128 != 0;
    long best = 0;
    int pick = -1;
    for (int i = qkv ? 1 : 0; i < (half || qkv ? 5 : 7); i++) {     // the q/k/v epilogue's tile has to fit in LDS, with per_cu of them
        const GemmI8Tile& t = kGemmI8Tiles[half][i];
        const long wgs = (long)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn), slots = 256 * t.per_cu;
        const long cost = (wgs + slots - 1) / slots * (t.stage * (k / (half ? 64 : 128)) + t.round);
        if (pick < 0 || cost < best) { best = cost; pick = i; }
    }
    return pick;
}

// Products on 128-byte rows whose tile has 256 columns share their rows out anew, as bfloat16 ones do (gemm_float.hip); costs in 0.01 us.
// 96 rows, which bfloat16 has too, make 2528 x 2048 x 8192 alone 8 % faster and the w4a4 prompt of 2528 around it 1.5 % slower (4350, 4415 us).
struct GemmI8Rows { int rows, stage, round; };
constexpr GemmI8Rows kGemmI8Rows[] = {{256, 110, 1500}, {224, 99, 1350}, {192, 88, 1200}, {160, 80, 1050}, {128, 70, 900}};
inline int gemm_i8_rows(int m, int k, int n, bool qkv) {
    if (qkv) return 128;                                       // blocks of 64 tokens
    long best = 0;
    int rows = 0;
    for (const GemmI8Rows& t : kGemmI8Rows) {
        const long tiles = (long)((m + t.rows - 1) / t.rows) * ((n + 255) / 256), cost = (tiles + 255) / 256 * (t.stage * (k / 128) + t.round);
        if (!rows || cost < best) { best = cost; rows = t.rows; }
    }
    return rows;
}

template <int EPI>
inline int launch_gemm_tiles(const int8_t* a, const int8_t* w, int32_t* c, const float* s_x, const float* w_s, const float* residual, float* y,
                             int m, int k, int n, hipStream_t st, QkvEpiArgs qa = QkvEpiArgs()) {
    const int pick = gemm_i8_tile(m, k, n, EPI == kDmaQkv);
#define FX_GEMM_TILE(BM, BN, ...) launch_gemm_dma<BM, BN, EPI, __VA_ARGS__>(a, w, c, s_x, w_s, residual, y, m, k, n, st, qa)
    if (k % 128 != 0) {
        if constexpr (EPI != kDmaQkv)
            if (pick == 0) return FX_GEMM_TILE(256, 256, 4, 2, 64, 8);
        if (pick == 1) return FX_GEMM_TILE(128, 256, 4, 2, 64, 8);
        if (pick == 2) return FX_GEMM_TILE(128, 128, 4, 2, 64, 8);
        if (pick == 3) return FX_GEMM_TILE(64, 128, 4, 2, 64);
        return FX_GEMM_TILE(64, 64, 4, 2, 64);
    }
    // (a head's 64 bytes leave in 16-byte pieces, and the scales and tables are read in such)
    if constexpr (EPI == kDmaQkv) {
        const auto bits = [](auto... p) { return (reinterpret_cast<uintptr_t>(p) | ...); };
        // (on 128 x 128 the eight waves of the other kernel hide more of it: 1024 x 3072 x 2048 19.1 us, 20.4 as a walk)
        if (pick == 1 && !(bits(qa.q8, qa.kc, qa.vc, qa.sin_t, qa.cos_t, w_s, qa.w_sum) & 15)) return launch_gemm_walk<EPI, 4>(a, w, c, s_x, w_s, residual, y, m, k, n, st, qa);
    }
    // (Units whose rows end inside 16 bytes went to 128 x 128 for a while: 1531 x 16388 x 2048 70 us ahead of the walk, 92 there, 64 here.)
    if (pick < 2 && EPI != kDmaQkv && rows_fit(n, 4)) {
#define FX_GEMM_ROWS(MI) launch_gemm_walk<EPI, MI>(a, w, c, s_x, w_s, residual, y, m, k, n, st, qa)
        if constexpr (EPI != kDmaQkv) switch (gemm_i8_rows(m, k, n, false)) {
            case 256: return FX_GEMM_ROWS(8);
            case 224: return FX_GEMM_ROWS(7);
            case 192: return FX_GEMM_ROWS(6);
            case 160: return FX_GEMM_ROWS(5);
            default: return FX_GEMM_ROWS(4);
        }
#undef FX_GEMM_ROWS
    }
    if constexpr (EPI != kDmaQkv) {
        if (pick == 5) return FX_GEMM_TILE(64, 64, 3, 3, 128);
        if (pick == 6) return FX_GEMM_TILE(128, 128, 2, 2, 128);
    }
    if (pick <= 2) return FX_GEMM_TILE(128, 128, 4, 2, 128, 8);
    if (pick == 3) return FX_GEMM_TILE(64, 128, 4, 2, 128, 8);
    return FX_GEMM_TILE(64, 64, 4, 2, 128);
#undef FX_GEMM_TILE
}

template <int EPI>
inline int launch_gemm(const int8_t* a, const int8_t* w, int32_t* c, const float* s_x, const float* w_s,
                       const float* residual, float* y, int m, int k, int n, hipStream_t st) {
    // the direct-load kernel needs 32-bit element offsets into both operands and 16-byte aligned output rows
    if ((size_t)m * k < (1ull << 31) && (size_t)n * k < (1ull << 31) && n % 4 == 0)
        return launch_gemm_tiles<EPI == kGemmDequant ? kDmaDequant : kDmaRaw>(a, w, c, s_x, w_s, residual, y, m, k, n, st);
    const int mode = ((m + 127) / 128) * ((n + 127) / 128) >= 1024 ? 0 : 2;
    const int nk = k / kGemmBK;
#define FX_GEMM_LAUNCH(BM, BN, DD)                                                                                \
    do {                                                                                                          \
        const int tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;                                                 \
        gemm_i8_kernel<BM, BN, EPI, DD><<<tm * tn, 256, 0, st>>>(a, w, c, s_x, w_s, residual, y, m, k, n, tm, tn); \
    } while (0)
    const bool deep = nk % 4 == 0;      // prefetch depth 4 needs the k-steps in groups of 4 (K % 256 == 0)
    if (mode == 0) { if (deep) FX_GEMM_LAUNCH(128, 128, 4); else FX_GEMM_LAUNCH(128, 128, 1); }
    else { if (deep) FX_GEMM_LAUNCH(64, 64, 4); else FX_GEMM_LAUNCH(64, 64, 1); }
#undef FX_GEMM_LAUNCH
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// Asymmetric activations held one value per byte (0..127, e.g. the uint4 values of the W4A4 path before packing) times
// int8 weights on the direct-load kernel: y = (float(acc) * s_x) * w_s + b_x * w_sum (+ residual).
inline int launch_gemm_asym(const int8_t* a, const int8_t* w, const float* s_x, const float* b_x, const float* w_s,
                            const float* w_sum, const float* residual, float* y, int m, int k, int n, hipStream_t st) {
    FX_REQUIRE((size_t)m * k < (1ull << 31) && (size_t)n * k < (1ull << 31) && n % 4 == 0,
               "linear_i8_gemm_dequant_asym: m=%d k=%d n=%d outside the direct-load kernel's range", m, k, n);
    QkvEpiArgs qa = QkvEpiArgs();
    qa.b_x = b_x; qa.w_sum = w_sum;
    return launch_gemm_tiles<kDmaDequantAsym>(a, w, nullptr, s_x, w_s, residual, y, m, k, n, st, qa);
}

// The gate/up projection of the W4A4 graph (interleaved rows, asymmetric activations held one value per byte) with
// SiLU(gate)*up in the epilogue: the asymmetric dequantisation of launch_gemm_asym followed by the product that the
// Hadamard kernel would otherwise form from the interleaved fp32 columns - the same arithmetic, half the output.
inline int launch_gemm_swiglu_asym(const int8_t* a, const int8_t* w_gu, const float* s_x, const float* b_x, const float* w_s_gu,
                                   const float* w_sum_gu, float* h, int m, int k, int n2, hipStream_t st) {
    FX_REQUIRE((size_t)m * k < (1ull << 31) && (size_t)n2 * k < (1ull << 31) && n2 % 4 == 0,
               "linear_i8_gemm_swiglu_asym: m=%d k=%d n=%d outside the direct-load kernel's range", m, k, n2 / 2);
    QkvEpiArgs qa = QkvEpiArgs();
    qa.b_x = b_x; qa.w_sum = w_sum_gu;
    return launch_gemm_tiles<kDmaSwigluAsym>(a, w_gu, nullptr, s_x, w_s_gu, nullptr, h, m, k, n2, st, qa);
}

// W4A4 prefill GEMM on nibble-packed operands (register-staged kernel, nibbles widened on the way to LDS).
template <int EPI>
inline int launch_gemm_u4i4(const uint8_t* a4, const uint8_t* w4, int32_t* c, const float* s_x, const float* b_x,
                            const float* w_s, const float* w_sum, const float* residual, float* y, int m, int k, int n, hipStream_t st) {
    const int8_t* a = reinterpret_cast<const int8_t*>(a4);
    const int8_t* w = reinterpret_cast<const int8_t*>(w4);
    const bool big = ((m + 127) / 128) * ((n + 127) / 128) >= 768;
    if (big) {
        const int tm = (m + 127) / 128, tn = (n + 127) / 128;
        gemm_i8_kernel<128, 128, EPI, 1, true><<<tm * tn, 256, 0, st>>>(a, w, c, s_x, w_s, residual, y, m, k, n, tm, tn, b_x, w_sum);
    } else {
        const int tm = (m + 63) / 64, tn = (n + 63) / 64;
        gemm_i8_kernel<64, 64, EPI, 1, true><<<tm * tn, 256, 0, st>>>(a, w, c, s_x, w_s, residual, y, m, k, n, tm, tn, b_x, w_sum);
    }
    FX_LAUNCH_CHECK();
    return FLEXLLM_OK;
}

// Gate/up projection with the SiLU(gate)*up product in the epilogue; n2 = 2 * intermediate size (interleaved rows).
inline int launch_gemm_swiglu(const int8_t* a, const int8_t* w_gu, const float* s_x, const float* w_s_gu, float* h, int m,
                              int k, int n2, hipStream_t st) {
    FX_REQUIRE((size_t)m * k < (1ull << 31) && (size_t)n2 * k < (1ull << 31) && n2 % 4 == 0,
               "linear_i8_gemm_swiglu: m=%d k=%d n=%d outside the direct-load kernel's range", m, k, n2 / 2);
    return launch_gemm_tiles<kDmaSwiglu>(a, w_gu, nullptr, s_x, w_s_gu, nullptr, h, m, k, n2, st);
}

// Fused q/k/v projection: GEMM over the concatenated [q | k | v] weight rows with RoPE, static int8 quantisation and
// the stores into q8 [tokens][q_heads][64], the K cache and the V cache in the epilogue.  Token i sits at position
// pos0 + i; pos0 % 64 == 0 and m % 32 == 0 so that a tile of 64 tokens is one block of the transposed V cache.
inline int launch_gemm_qkv(const int8_t* a, const int8_t* w_qkv, const float* s_x, const float* w_s, int m, int k,
                           const QkvEpiArgs& qa, hipStream_t st) {
    const int n = (qa.q_heads + 2 * qa.kv_heads) * kHd;
    FX_REQUIRE(m % 32 == 0 && qa.pos0 % 64 == 0 && qa.pos0 + m <= qa.max_pos, "gemm_qkv: m=%d pos0=%d max_pos=%d", m, qa.pos0, qa.max_pos);
    FX_REQUIRE((size_t)m * k < (1ull << 31) && (size_t)n * k < (1ull << 31), "gemm_qkv: m=%d k=%d outside the direct-load kernel's range", m, k);
    return launch_gemm_tiles<kDmaQkv>(a, w_qkv, nullptr, s_x, w_s, nullptr, nullptr, m, k, n, st, qa);
}

}  // namespace fx
