// The walk over k that the GEMMs of many rows share (int8, bfloat16 and float32): C[m][n] = sum_k A[m][k] * W[n][k], both operands
// K-contiguous, on 16 x 16 matrix instructions.
//
// Four waves per workgroup, one per SIMD, as a grid of two by two; a wave's tile is MI x NI blocks of 16 x 16.  Rows go global -> LDS by
// direct loads in stages of 128 bytes of k (whole lines; halves of them reach 14.5 TB/s where lines reach 23), through a ring of NA
// stages of A and one of NB stages of W.  A lane's 16 bytes of a row are one operand, so nothing is transposed; the 16-byte chunks of
// row r are stored rotated by (r >> 1) & 7, which is applied on the global side of the load, and the operand reads are free of conflicts.
//
// What bounds it.  A 256 x 256 tile reads 32 KiB of operands from LDS per 16 KiB that arrive, against 48 with eight waves of 128 x 64: with
// those, LDS was busy all the time and the matrix cores 55 % of it.  Now they are busy for 73 to 78 % of the cycles of a long walk, and the chip's
// power holds the clock at 1.76 to 1.85 GHz (counters of 4096 x 28672 x 4096, 4096 x 4096 x 4096 and 4096 x 16384 x 4096; 16 x 16 instructions take less of
// it than 32 x 32 ones, which took 4 to 6 % more time).  What it took: each matrix instruction has at most an operand read and one half of a direct load behind it; the
// loads of a stage are spread over one and a half k-steps (in a burst they queue up and the matrix instructions behind them
// wait), and A is a stage further ahead than W, which is what fits into 160 KiB.
// bfloat16, before (eight waves, 32 x 32 instructions) and now, us: 4096 x 4096 x 14336 (m, n, k) 407 and 320, 1504 TFLOP/s; 4096 x 28672 x 4096 879
// and 706; 4096 x 4096 x 4096 127 and 98; 777 x 4096 x 14336 on 128 x 128 113 and 99; 1024 x 2048 x 2048 on 64 x 128 16.6 and 16.0.
// float32: 333 x 16384 x 2048 205 and 182, 333 x 2048 x 8192 150 and 135.
//
// The operands of the matrix instruction are exchanged: W's rows are its rows, A's rows its columns.  A lane then holds four
// consecutive columns n of one row m, and the outputs leave without a turn through LDS.
#pragma once
#include "elem.h"

namespace fx {

template <typename ET> struct MatrixOp;
template <> struct MatrixOp<int8_t> {
    using Frag = i32x4; using Acc = i32x4;
    static __device__ __forceinline__ void mma(const Frag& w, const Frag& a, Acc& c) { c = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, a, c, 0, 0, 0); }
};
template <> struct MatrixOp<bf16_t> {
    using Frag = bf16x8; using Acc = f32x4;
    static __device__ __forceinline__ void mma(const Frag& w, const Frag& a, Acc& c) { c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, c, 0, 0, 0); }
};
template <> struct MatrixOp<float> {     // 16 bytes are four k of a row; an instruction takes the same one of every lane, in both operands
    using Frag = f32x4; using Acc = f32x4;
    static __device__ __forceinline__ void mma(const Frag& w, const Frag& a, Acc& c) {
#pragma unroll
        for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e ^ 1], a[e ^ 1], c, 0, 0, 0);   // any order will do
    }
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {                 // s_waitcnt vmcnt(N) only; the count is a 6-bit split immediate
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// The tile of workgroup `id`.  Ids go to the eight dies in turn, each with an L2 of its own: of every 256 tiles (a round over the chip) a
// die takes 32 in a row, which are eight row tiles by four column tiles.  They read 12 stages of rows per stage where 32 row
// tiles by one column tile read 33.
// Quotients stand ahead of the first load, so they are float ones put right by the remainder (exact: a quotient of tiles is below 2^20, and the
// float one below half off); a division of integers takes three times the instructions.
__device__ __forceinline__ int quotient_of_lane(int a, int d) {
    const int q = (int)((float)a * __builtin_amdgcn_rcpf((float)d)), r = a - q * d;
    return q + (r >= d) - (r < 0);
}
__device__ __forceinline__ int quotient(int a, int d) { return __builtin_amdgcn_readfirstlane(quotient_of_lane(a, d)); }
// Groups of rows that have a W each: one row tile by all column tiles, which share its rows (ROWS 1).
template <int ROWS = 8, class Q>
__device__ __forceinline__ void gemm_tile_by(Q quotient, int id, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n, round = id & ~255, in = id & 255, left = min(total - round, 256), die = in & 7;
    const int t = round + die * (left >> 3) + min(die, left & 7) + (in >> 3);
    constexpr int G = ROWS;
    const int group = tiles_m <= G ? 0 : quotient(t, G * tiles_n), rows = min(G, tiles_m - group * G), o = t - group * G * tiles_n;
    tn = rows == G ? o / G : quotient(o, rows);
    tm = group * G + o - tn * rows;
}

template <int ROWS = 8>
__device__ __forceinline__ void gemm_tile_of(int id, int tiles_m, int tiles_n, int& tm, int& tn) { gemm_tile_by<ROWS>(quotient, id, tiles_m, tiles_n, tm, tn); }
template <int ROWS = 8>                                        // an id of every lane's own
__device__ __forceinline__ void gemm_tile_of_lane(int id, int tiles_m, int tiles_n, int& tm, int& tn) { gemm_tile_by<ROWS>(quotient_of_lane, id, tiles_m, tiles_n, tm, tn); }

// R words of each of 4/R blocks, as lanes hold them (lane group g of 16 lanes has words g*R .. g*R + R - 1 of a block's row), become four
// consecutive words per lane: group g then has words 4g .. 4g + 3 of the row through all the blocks, in the order w[0][0], w[0][1] ...
template <int R>
__device__ __forceinline__ void join_blocks(uint32_t (&w)[4 / R][R]) {
    auto swap32 = [](uint32_t& a, uint32_t& b) { const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false); a = r[0]; b = r[1]; };
    auto swap16 = [](uint32_t& a, uint32_t& b) { const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false); a = r[0]; b = r[1]; };
    if constexpr (R == 2) {
#pragma unroll
        for (int r = 0; r < 2; r++) { swap32(w[0][r], w[1][r]); swap16(w[0][r], w[1][r]); }
    } else if constexpr (R == 1) {
        swap32(w[0][0], w[2][0]); swap32(w[1][0], w[3][0]);
        swap16(w[0][0], w[1][0]); swap16(w[2][0], w[3][0]);
    }
}

// Rows of an output (or a residual) as a tile sees them: 16-byte accesses at byte offsets (of whole words) behind its first row.  What lies behind the last
// row is neither written nor read (zeros come back), and neither is offset kNowhere: no branch stands around a store, so that
// loads issued ahead of stores are not waited for together with them.  A tile's rows have to stay below 2 GiB (rows_fit): of the rows that are
// left of the matrix only the tile's own `most` count, all of them can be more bytes than 32 bits say.
constexpr int kNowhere = -1;
inline bool rows_fit(int ld, int bytes) { return (size_t)256 * ld * bytes < (1ull << 31); }
struct TileRows {
    __amdgpu_buffer_rsrc_t r;
    static __host__ __device__ constexpr int bytes(int left, int most, int row_bytes) { return left <= 0 ? 0 : (left < most ? left : most) * row_bytes; }
    __device__ __forceinline__ TileRows(void* first_row, int left, int most, int row_bytes)
        : r(__builtin_amdgcn_make_buffer_rsrc(first_row, 0, bytes(left, most, row_bytes), 0x00027000)) {}
    __device__ __forceinline__ void put(const uint32_t* w, int at) const {
        const i32x4 v = {(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        __builtin_amdgcn_raw_buffer_store_b128(v, r, at, 0, 0);
    }
    __device__ __forceinline__ void put_half(const uint32_t* w, int at) const {      // the first 8 of the 16 bytes
        using i32x2 = int __attribute__((ext_vector_type(2)));
        const i32x2 v = {(int)w[0], (int)w[1]};
        __builtin_amdgcn_raw_buffer_store_b64(v, r, at, 0, 0);
    }
    __device__ __forceinline__ f32x4 get(int at) const {
        const i32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0);
        return {__int_as_float(v[0]), __int_as_float(v[1]), __int_as_float(v[2]), __int_as_float(v[3])};
    }
};

static_assert(TileRows::bytes(65536, 128, 65536) == 128 * 65536 && TileRows::bytes(5, 128, 65536) == 5 * 65536 && TileRows::bytes(-3, 128, 65536) == 0, "bytes of a tile's rows");

// A kernel's arguments come from memory, and each group of them that is asked for behind a branch or an index is a trip of its own ahead of
// the first load.  Values that stand here are in scalar registers from here on, so that they are asked for together at the start
// (three trips one after the other before, us: 24 x 8192 x 512 5.81 and 5.48, 41 x 2560 x 2048 9.41 and 9.11; the two trips of the wide tiles stay, with the
// arguments in registers their sums do not fit).
template <typename... T>
__device__ __forceinline__ void arguments(const T&... v) {
    auto one = [](const auto& x) __attribute__((always_inline)) { asm volatile("" :: "s"(x)); };
    (one(v), ...);
}

// The workgroup's barrier alone: what has to be waited for is waited for explicitly ahead of it.  No memory access moves across it.
__device__ __forceinline__ void barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

// A direct load, global -> LDS: 16 bytes per lane from byte `off` behind base, to 16 bytes per lane from LDS address `to` on, which the
// instruction takes from m0 (one wait state after it was written).  m0 is an output, so that the compiler knows that what it may have there itself
// is gone.  ONCE: read once on this chip.
template <bool ONCE = false>
__device__ __forceinline__ void load_to_lds(const void* base, unsigned off, unsigned to) {
    unsigned m0;
    if constexpr (ONCE) asm volatile("s_mov_b32 %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3 nt" : "=&{m0}"(m0) : "s"(to), "v"(off), "s"(base) : "memory");
    else asm volatile("s_mov_b32 %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3" : "=&{m0}"(m0) : "s"(to), "v"(off), "s"(base) : "memory");
}

// The tile of a workgroup that walks one.  A workgroup that walks several (kMany) says besides: more(), whether another tile follows; rows() and cols(),
// which put the offsets of that one's loads in the place of this one's; out(), this one's outputs, behind which the other one is this one.
// Every tile walks k from its beginning: a sum's order does not hang on where its tile lies or on how many rows there are.  (Workgroups that read W once and begin
// together ask for the same bytes of rows a power of two apart.  Begun at different stages of k, products of up to 128 rows were 2 to 5 % faster, but a row's sums
// were then others than on the tiles of longer prompts, and what is rounded to bfloat16 behind them as well.)
struct OneTile {
    static constexpr bool kMany = false;
    template <class... X> __device__ void rows(X&...) const {}
    template <class... X> __device__ void cols(X&...) const {}
};

// ONCE: W is read by one row tile alone, and does not take the place of what is read again in the caches.
template <typename ET, int WM, int MI, int NI, int NA, int NB, bool ONCE = false>
struct GemmWalk {
    static constexpr bool kOnce = ONCE;
    using Op = MatrixOp<ET>;
    using Frag = typename Op::Frag;
    using Acc = typename Op::Acc;
    static constexpr int WN = 4 / WM, BM = WM * MI * 16, BN = WN * NI * 16;
    static constexpr int RA = (BM + 31) / 32 * 32, RB = BN;    // rows in LDS: every wave issues the same number of loads, of eight rows each
    static constexpr int AI = RA / 32, BI = RB / 32, PER = AI + BI;
    static constexpr int ASZ = RA * 128, BSZ = RB * 128, kLds = NA * ASZ + NB * BSZ;
    static_assert(WM == 2, "waves along the rows");
    static_assert(RB % 32 == 0 && (NA == NB || NA == NB + 1) && NB >= 2 && NB <= 4 && kLds <= 160 * 1024, "ring");
    // waves per SIMD that registers have to leave room for: as many workgroups as LDS does, two waves' worth of registers where that is enough
    static constexpr int per_cu() { return kSumsApart ? 1 : 160 * 1024 / kLds < 2 ? 2 : 160 * 1024 / kLds < 3 ? 2 : 3; }
    // a wave's loads in flight behind those of the stage that a wait is for, `younger` stages behind it
    static constexpr int in_flight(int younger) {
        const int a = younger < NA - 1 ? younger : NA - 1, b = younger < NB - 1 ? younger : NB - 1;
        // loads of stage s go out behind the barrier of stage s - NB (W) and s - NA (A), W ahead of A
        return NA == NB ? (a < NB - 2 ? a : NB - 2) * PER : (a < NB - 1 ? a : NB - 1) * AI + (b < NB - 2 ? b : NB - 2) * BI;
    }
    static_assert((NB - 1) * PER < 64, "wait count");
    // Beyond a wave's 256 vector registers the sums live in the accumulation registers.
    static constexpr bool kSumsApart = (MI * NI + 2 * (MI + NI)) * 4 > 210;

    // Place, counted in matrix instructions behind a barrier, at which the j-th load of W (A) is aimed; it goes out behind the next matrix
    // instruction, in the same stage.
    static constexpr int NM = MI * NI, NR = MI + NI, KS = 2;
    static constexpr int SB = NM / 2 > BI ? NM / 2 : BI, SA = KS * NM - SB < NM ? KS * NM - SB : NM;
    static constexpr int slot_b(int j) { return j * SB / BI; }
    static constexpr int slot_a(int j) { return SB + j * SA / AI + (SB + j * SA / AI == NM - 1); }
    static constexpr int early() {                             // A's loads inside the last k-step
        int n = 0;
        for (int j = 0; j < AI; j++) n += slot_a(j) + 1 < NM;
        return n;
    }
    static_assert(SB < NM && SA >= 2 * AI && slot_b(BI - 1) + 1 <= SB && slot_a(AI - 1) + 1 < KS * NM, "places of the loads");
    static_assert(NR <= NM, "an operand read behind a matrix instruction");

    static __device__ __forceinline__ int rot(int r) { return (r >> 1) & 7; }
    static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }
    static __device__ __forceinline__ int row_of_wave() { return (wave() / WN) * (MI * 16); }
    static __device__ __forceinline__ int col_of_wave() { return (wave() % WN) * (NI * 16); }
    // row of the tile that this lane's j-th load of A (W) is for, and the lane's byte within the 128 of the stage
    static __device__ __forceinline__ int load_row_a(int j) { return (wave() * AI + j) * 8 + ((int)threadIdx.x & 63) / 8; }
    static __device__ __forceinline__ int load_row_b(int j) { return (wave() * BI + j) * 8 + ((int)threadIdx.x & 63) / 8; }
    static __device__ __forceinline__ unsigned load_byte(int r) { return (unsigned)((((int)threadIdx.x & 7) ^ rot(r)) * 16); }

    // a, w: first byte of k of the operands; offa, offb: byte offsets of this lane's loads behind them; nk: stages.  Nothing else of the
    // workgroup may be on its way to LDS.  Ends with every wave's loads and reads of LDS complete, without a barrier.
    // Of several tiles (nk >= NA) the ring goes on from one to the next: the last stages of a tile ask for the first ones of the tile behind it, which are on
    // their way while the outputs leave, and the place of a tile takes neither the trips ahead of its first stage nor the drain behind its last.
    template <class T>
    static __device__ __forceinline__ void run(const int8_t* a, const int8_t* w, unsigned (&offa)[AI], unsigned (&offb)[BI], int nk, int8_t* smem,
                                               Acc (&acc)[MI][NI], T tiles) {
        const int lane = threadIdx.x & 63, wv = wave();
        const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
        const unsigned lds_a = lds0 + wv * (AI * 1024), lds_b = lds0 + NA * ASZ + wv * (BI * 1024);
        // A direct load in two halves, with a matrix instruction between them: the address has to be in m0 one wait state ahead of the load.
        // What `aim` leaves in m0 is an operand of `load_a` and `load_w`, so that the compiler puts nothing of its own there between them.
        unsigned m0 = 0;
        auto aim = [&](unsigned base, int j) __attribute__((always_inline)) {
            asm volatile("s_add_u32 %0, %1, %2" : "={m0}"(m0) : "s"(__builtin_amdgcn_readfirstlane(base)), "i"(j * 1024) : "scc");
        };
        auto load_a = [&](unsigned off, int stage) __attribute__((always_inline)) {
            asm volatile("global_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(a + (size_t)stage * 128), "{m0}"(m0) : "memory");
        };
        auto load_w = [&](unsigned off, int stage) __attribute__((always_inline)) {
            if constexpr (ONCE) asm volatile("global_load_lds_dwordx4 %0, %1 nt" :: "v"(off), "s"(w + (size_t)stage * 128), "{m0}"(m0) : "memory");
            else asm volatile("global_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(w + (size_t)stage * 128), "{m0}"(m0) : "memory");
        };
        auto settle = [] __attribute__((always_inline)) { asm volatile("s_nop 0" ::: "memory"); };
        auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NI; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] = 0;
            // Zeros of its own for every block: from one shared zero the compiler cannot keep the sums in place, and the loop is full of moves.
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NI; j++) {
                    if constexpr (kSumsApart) asm volatile("" : "+a"(acc[i][j])); else asm volatile("" : "+v"(acc[i][j]));
                }
        };
        clear();
        wait_vmcnt<0>();                                        // what the compiler loaded itself stays out of the counts
        // Behind the barrier of stage e: W's loads of stage e + NB over the first half of the last k-step, then A's of e + NA over
        // as many matrix instructions as a k-step has.
        constexpr int early_a = early();
#pragma unroll
        for (int s = 0; s < NA; s++) {
#pragma unroll
            for (int j = 0; j < BI; j++)
                if (s < NB && s < nk) { aim(lds_b + s * BSZ, j); settle(); load_w(offb[j], s); }
#pragma unroll
            for (int j = 0; j < AI; j++)
                if ((s < NA - 1 || j < early_a) && s < nk) { aim(lds_a + s * ASZ, j); settle(); load_a(offa[j], s); }
        }
        const int fr = lane & 15, fg = lane >> 4;
        int at[KS];
#pragma unroll
        for (int s = 0; s < KS; s++) at[s] = fr * 128 + (((s * 4 + fg) ^ rot(fr)) * 16);
        const int8_t* const read_a = smem + row_of_wave() * 128;
        const int8_t* const read_b = smem + NA * ASZ + col_of_wave() * 128;
        Frag fa[2][MI], fb[2][NI];
        auto read = [&](unsigned sa, unsigned sb, int ks, int set, int q) __attribute__((always_inline)) {       // q-th of the reads of a k-step
            if (q == 0) fa[set][0] = *reinterpret_cast<const Frag*>(read_a + sa + at[ks]);
            else if (q <= NI) fb[set][q - 1] = *reinterpret_cast<const Frag*>(read_b + sb + at[ks] + (q - 1) * 2048);
            else fa[set][q - NI] = *reinterpret_cast<const Frag*>(read_a + sa + at[ks] + (q - NI) * 2048);
        };
        auto wait_stage = [&](int younger) __attribute__((always_inline)) {
            if (younger >= NB) wait_vmcnt<in_flight(NB)>();
            else if (NB > 3 && younger == 3) wait_vmcnt<in_flight(3)>();
            else if (NB > 2 && younger == 2) wait_vmcnt<in_flight(2)>();
            else if (younger == 1) wait_vmcnt<in_flight(1)>();
            else wait_vmcnt<0>();
        };
        // Stage 0 is in when what was asked for behind it is out: all of the stages 1 .. NA - 1 that there are, as far as they are asked for.
        {
            constexpr int full = (NB - 1) * BI + (NA - 2) * AI + early_a;
            if (nk >= NA) wait_vmcnt<(full < 63 ? full : 63)>();
            else wait_vmcnt<0>();
        }
        barrier();
#pragma unroll
        for (int q = 0; q < NR; q++) read(0, 0, 0, 0, q);
        // ring slots of the last, this and the next stage; the last one's are refilled
        unsigned a0 = (NA - 1) * ASZ, a1 = 0, a2 = ASZ, b0 = (NB - 1) * BSZ, b1 = 0, b2 = BSZ;
        int ka = NA - 1, kb = NB - 1;                            // stages kt - 1 + NA and kt - 1 + NB (as numbers: pointers cost the wide tiles spills)
        // left: stages behind this one.  loads: 2 all, 1 what is left for the last stages (the rest of the last barrier's, and W's where it is a stage
        // behind A), 0 none.  No branches among them: those cost a short walk 2 % (250 x 2560 x 2048 in four parts, eight stages on 128 x 128, 11.4 us and 11.2).
        // turn, where another tile follows: 1 from the last k-step on the loads are that one's, 2 the next stage is that one's and is read behind the outputs.
        auto turning = [&](int left, auto next, auto loads, auto turn) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < KS; s++) {
                constexpr bool kNext = decltype(next)::value;
                constexpr int kLoads = decltype(loads)::value;
                constexpr int kTurn = decltype(turn)::value;
                const bool last = s == KS - 1;
                if constexpr (kTurn & 1) {
                    if (last) {
                        tiles.rows(offa);
                        tiles.cols(offb, w);
                        ka = kb = -1;
                    }
                }
                if (last && kNext) {
                    if constexpr (kLoads > 0) wait_vmcnt<in_flight(NA - 2)>(); else wait_stage(left - 1);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    barrier();
                }
#pragma unroll
                for (int x = 0; x < NM; x++) {
                    Op::mma(fb[s & 1][x % NI], fa[s & 1][x / NI], acc[x / NI][x % NI]);
                    // operands of the next k-step, evenly over the first half of the matrix instructions
                    constexpr int RS = NM / 2 / NR > 0 ? NM / 2 / NR : 1;
                    if (x % RS == 0 && x / RS < NR) {
                        if (!last) read(a1, b1, s + 1, (s + 1) & 1, x / RS);
                        else if (kNext && !(kTurn & 2)) read(a2, b2, 0, (s + 1) & 1, x / RS);
                    }
                    // place behind the barrier of this stage (last k-step) or of the one before
                    const int p = last ? x : (s + 1) * NM + x;
                    const unsigned sa = last ? a1 : a0, sb = last ? b1 : b0;
                    const bool there_a = kLoads == 2 || (kLoads == 1 && !last), there_b = kLoads == 2 || (kLoads == 1 && NA > NB && last);
#pragma unroll
                    for (int j = 0; j < BI; j++) {
                        if (p == slot_b(j) + 1 && there_b) load_w(offb[j], last ? kb + 1 : kb);
                        if (p == slot_b(j) && there_b) aim(lds_b + sb, j);
                    }
#pragma unroll
                    for (int j = 0; j < AI; j++) {
                        if (p == slot_a(j) + 1 && there_a) load_a(offa[j], last ? ka + 1 : ka);
                        if (p == slot_a(j) && there_a) aim(lds_a + sa, j);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            ka++; kb++;
            a0 = a1; a1 = a2; a2 = a2 == (NA - 1) * ASZ ? 0 : a2 + ASZ;
            b0 = b1; b1 = b2; b2 = b2 == (NB - 1) * BSZ ? 0 : b2 + BSZ;
        };
        auto stage = [&](int left, auto next, auto loads) __attribute__((always_inline)) { turning(left, next, loads, std::integral_constant<int, 0>()); };
        int left = nk - 1;
        if constexpr (T::kMany) {
            static_assert(NA == NB, "rows and columns turn to the next tile in the same stage");
            using All = std::integral_constant<int, 2>;
            while (tiles.more()) {
                for (; left >= NA; left--) stage(left, std::true_type(), All());
                turning(left--, std::true_type(), All(), std::integral_constant<int, 1>());
                for (; left >= 1; left--) stage(left, std::true_type(), All());
                turning(0, std::true_type(), All(), std::integral_constant<int, 2>());
                tiles.out(acc);
                clear();
#pragma unroll
                for (int q = 0; q < NR; q++) read(a1, b1, 0, 0, q);
                left = nk - 1;
            }
        }
        if (nk >= NA) {
            for (; left >= NA; left--) stage(left, std::true_type(), std::integral_constant<int, 2>());
            stage(left--, std::true_type(), std::integral_constant<int, 1>());
        }
        for (; left >= 1; left--) stage(left, std::true_type(), std::integral_constant<int, 0>());     // everything is on its way
        stage(0, std::false_type(), std::integral_constant<int, 0>());
        if constexpr (T::kMany) tiles.out(acc);
    }
};

}  // namespace fx
