// Whole decode steps of one token in one kernel: 256 workgroups, one per CU, stay resident and walk through the linears and
// the attention of all layers, the head and the choice of the next token.
//
// What bounds a step of one token: a layer is a chain of five linears and attentions, each of which needs all of the one before.  As
// kernels of their own every link costs 3.5 us of launch and ramp beside its stream of weights: 16 layers of 2048, feed-forward 8192, bfloat16, 1531
// tokens held, take 43 us each for 122 MB (17 us at the rate of a read stream).  Here a link costs an exchange between resident
// workgroups, 1.3 us behind the slowest of them, and the weights, which do not hang on the activations, are asked for ahead of it: 33 us per
// layer, 771 -> 595 us per token (four layers of 4096: 535 -> 466; ten layers, six of them twice, float32: 1098 -> 903).
// bfloat16 products on the matrix cores, the vector as three parts: 595 -> 566 us per token, with latent and recurrent layers in turn 713 -> 692, with mixtures
// 520 -> 516; four layers of 4096, whose quads are the weights' stream, 462 and 461, 522 and 525.
// Eight of a workgroup's twelve waves ("stream waves") do nothing but walk through the workgroup's rows of all linears.  The other four ("service
// waves") wait for the vectors, norm them, attend, finish the sums.  Answers of vector memory return to a wave in order, so a wave that streams could not see a word of
// another workgroup before its weights.
// The two kinds meet twice in every linear, by counts in LDS that are added to with release and read with acquire (kFree), in models with mixtures at workgroup barriers in
// the same two places:
//   L.ready, one from each service wave: its share of the vector is in LDS, and it has read the sums of the linear before.  Behind all four the stream waves read the
//     vector and write sums.
//   L.done, one from each stream wave: its sums are in LDS, and it has read the vector for the last time.  Behind all eight the service waves read the sums, and the vector's
//     place is theirs: the mixers' values lie over it, until all service waves have met (take, norm) and put the next vector there.  The head's sums, which may lie
//     behind its vector where a longer one would, are read before the service waves meet in the next token's first norm.
//   L.sent guards nothing: stream waves ask for more once the sums have left, so that the words stand ahead of their requests.
// Words between workgroups: a float32 goes past the L2 caches (which do not see each other's lines) to a place of its own per layer run,
// which holds kUnset until then; readers poll the places themselves, 16 bytes per lane.  There are two sets of places, for tokens in
// turn: who writes a word of one set puts kUnset back in the other one, whose readers were done a token ago (a token ends with an exchange that all
// workgroups take part in, or with the kernel).  A result that happens to have kUnset's bits leaves as another NaN.
// All waits are bounded: a wait that times out raises a flag, everybody then runs to the end without waiting.  The host has a copy of the
// flag, and refuses further steps until it has been asked for.
#include "decode_float.h"
#include "route.h"
#include <atomic>

namespace fx {

constexpr int kSvcWaves = 4, kSvcT = kSvcWaves * 64, kStrWaves = 8, kWalkT = kSvcT + kStrWaves * 64;
constexpr unsigned kUnset = 0xFFFFFFFFu;
constexpr int kWalkErrPeriod = 64;
constexpr int kQuad = 4096;                               // bytes that a stream wave asks for at a time: 4 x 16 per lane

// Pointers out of tables are global ones: as the generic ones that the compiler takes them for, their loads would count as LDS accesses
// too, and every wait for LDS would wait for all of them.
template <typename T> using Global = T __attribute__((address_space(1)));
template <typename T> __device__ __forceinline__ const Global<T>* global(const T* p) { return (const Global<T>*)p; }
using RunPtr = const WalkRun __attribute__((address_space(4)))*;       // read-only for the whole launch: scalar loads

__device__ __forceinline__ bool unset(float v) { return (unsigned)__float_as_int(v) == kUnset; }

struct Wait {
    const WalkArgs& a;
    bool dead;
    __device__ __forceinline__ bool give_up(int it) {
        if (it % kWalkErrPeriod != 0 && it < a.polls) return false;
        if (__hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            dead = true;
        } else if (it >= a.polls) {
            __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.told, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            dead = true;
        }
        return dead;
    }
};
// N x 16 bytes per lane from base + off[i] (bytes), past the L2
template <int N>
__device__ __forceinline__ void load_words(const float* base, const unsigned (&off)[N], f32x4 (&v)[N]) {
    if constexpr (N == 1) {
        asm volatile("global_load_dwordx4 %0, %1, %2 sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v[0]) : "v"(off[0]), "s"(base) : "memory");
    } else if constexpr (N == 2) {
        asm volatile("global_load_dwordx4 %0, %2, %4 sc1\n\tglobal_load_dwordx4 %1, %3, %4 sc1\n\ts_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]) : "v"(off[0]), "v"(off[1]), "s"(base) : "memory");
    } else if constexpr (N == 4) {
        asm volatile("global_load_dwordx4 %0, %4, %8 sc1\n\tglobal_load_dwordx4 %1, %5, %8 sc1\n\tglobal_load_dwordx4 %2, %6, %8 sc1\n\t"
                     "global_load_dwordx4 %3, %7, %8 sc1\n\ts_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base) : "memory");
    } else {
        static_assert(N == 8, "words at a time");
        asm volatile("global_load_dwordx4 %0, %8, %16 sc1\n\tglobal_load_dwordx4 %1, %9, %16 sc1\n\tglobal_load_dwordx4 %2, %10, %16 sc1\n\t"
                     "global_load_dwordx4 %3, %11, %16 sc1\n\tglobal_load_dwordx4 %4, %12, %16 sc1\n\tglobal_load_dwordx4 %5, %13, %16 sc1\n\t"
                     "global_load_dwordx4 %6, %14, %16 sc1\n\tglobal_load_dwordx4 %7, %15, %16 sc1\n\ts_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
                     : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "v"(off[5]), "v"(off[6]), "v"(off[7]), "s"(base) : "memory");
    }
}
// The same, until none of the words is unset; of the last 16 bytes the first LAST words count.
template <int N, int LAST = 4>
__device__ __forceinline__ void poll_words(const float* base, const unsigned (&off)[N], bool need, f32x4 (&v)[N], Wait& w) {
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bool ok = !need || w.dead;
    int it = 0;
    for (;;) {
        if (!ok) {
            load_words<N>(base, off, v);
            ok = true;
#pragma unroll
            for (int i = 0; i < N; i++)
#pragma unroll
                for (int e = 0; e < (i == N - 1 ? LAST : 4); e++) ok = ok && !unset(v[i][e]);
        }
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) break;
        if (w.give_up(++it)) break;
    }
}

template <int N>
__device__ __forceinline__ float lanes_sum(float v) {     // over groups of N neighbouring lanes
    if constexpr (N > 1) v += lane_xor_f<1>(v);
    if constexpr (N > 2) v += lane_xor_f<2>(v);
    if constexpr (N > 4) v += lane_xor_f<4>(v);
    if constexpr (N > 8) v += lane_xor_f<8>(v);
    if constexpr (N > 16) v += lane_xor_f<16>(v);
    return v;
}
// f for the masks of a butterfly over groups of n neighbouring lanes, n a power of two up to 16
template <class F>
__device__ __forceinline__ void group(int n, F f) {
    f(std::integral_constant<int, 1>());
    f(std::integral_constant<int, 2>());
    if (n > 4) f(std::integral_constant<int, 4>());
    if (n > 8) f(std::integral_constant<int, 8>());
}

constexpr float kWalkLog2e = 1.44269504088896340736f;

// A linear of the workgroup.  phase: address of its rows; quads and quads per row (0: half a one), with parts rows and blocks of k.  group, for mixtures: the vector's and the
// sums' places; number of the group; [last << 31 | first << 30 | wave that begins << 16 | mixture].
struct WalkTables { int4 *phase, *group; };
struct MixerLds {                                         // where the vector lies otherwise: nobody needs that while the mixers are at work
    __attribute__((aligned(16))) float q[kWalkRow2];      // query; of gated linear attention query, key, decay, and what is short
    __attribute__((aligned(16))) float kx[kWalkRow2];     // the row of this step
    __attribute__((aligned(16))) float ql[kWalkRow2];     // latent query
    __attribute__((aligned(16))) float sums[kSvcWaves][kWalkRank];
};
static_assert(sizeof(MixerLds) <= kWalkMixerLds, "room for the mixers");
struct WalkLds {                                          // ahead of the tables, the vector and the sums
    __attribute__((aligned(16))) float of_head[32];
    float z[kWalkExperts + 1], choice_w[kWalkTop + 1];
    float m[kSvcWaves], l[kSvcWaves];
    int met, ready, done, sent, chosen;                   // service waves' barrier; linears (free: shares) whose vector is there, shares whose sums are; linears whose sums have left; mixtures that have chosen
    float norm[2][kSvcWaves];
    float bestv[2][kSvcWaves];
    int besti[2][kSvcWaves];
};

// ---- stream waves ---------------------------------------------------------------------------------------------------
// A workgroup's rows of a linear are one stretch of memory, dealt to the stream waves in turn in quads of 4 KiB, of which a row is a whole
// number.  Each wave has a ring of `slots` quads in LDS.  The trip is direct (the compiler does not see it: a wait names how many
// younger quads are on their way), so a request holds no register and may be made at any time.  When it is made matters: a CU takes
// 32 KiB of requests or so, then the wave that asks stands still until bytes arrive.  Freed slots are therefore filled at once only from the same
// linear; what belongs to the next ones is asked for behind the sums, beside the exchange.  (With register buffers that the
// compiler waits for, refilled on the spot, the last products of a linear wait until the next one's first quads are asked for: gate/up of
// 16384 x 2048 8.7 us behind a full ring, 7.1 so.  Eight waves: with four, one per SIMD, a quad's 100 instructions are not hidden, 13 us.)
__device__ __forceinline__ void quad_to_lds(const char* base, unsigned voff, unsigned dst) {
    unsigned saved_m0;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %3\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2 nt\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:1024 nt\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:2048 nt\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:3072 nt\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved_m0) : "v"(voff), "s"(base), "s"(dst) : "memory");
}
// Until all but the youngest n quads have arrived; n at most 3, since a ring has at most four.
__device__ __forceinline__ void wait_quads(int n) {
    switch (n) {
        case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
        case 1: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
        case 2: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
    }
}
// A wave's part in a count that others wait for: what it has written to LDS before is there.
__device__ __forceinline__ void add(int& f) {
    if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(&f, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int flag(const int& f) { return __builtin_amdgcn_readfirstlane(__hip_atomic_load(&f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)); }
// Between linears the waves ask and look for the vector in turn.  FREE: they do not stand still until a quad is there, and the two kinds of waves meet by counts;
// otherwise a wave has one quad at a time on its way, and they meet at barriers, for which all have to be there.  16 layers of 2048, 24 tokens behind 1531 rows:
// 19170 us with barriers, 18500 free; latent rows and gated linear attention 19390 and 19110; with mixtures 15200 and 15470, whose choice is one more chain of words
// that requests stand in the way of.
template <int KIND> constexpr bool kFree = KIND != kWalkMixture;
// MOE: with groups of linears and rows of half a quad (the other models are 2 to 3 % faster without).
template <typename ET, bool MOE, bool FREE>
__device__ __forceinline__ void stream_waves(WalkLds& L, WalkTables T, const float* xs, float* red, const char* ring, int slots, int phases, int tokens, int routed, int head, int head_off) {
    constexpr int CE = Chunk<ET>::N, PL = CE / 4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) - kSvcWaves;
    auto word = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const char* mine = ring + (size_t)wave * slots * kQuad;
    const unsigned dst = word((int)(unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)mine);
    // what is asked for next: quad iq of linear ip of token it
    int ip = 0, it = 0, iq = wave, itotal = word(T.phase[0].z), iorder = 0, igroup = 0, islot = 0, ahead = 0;      // ahead: quads asked for and not taken in
    auto base_of = [&](int p) { return reinterpret_cast<const char*>(((unsigned long long)(unsigned)word(T.phase[p].y) << 32) | (unsigned)word(T.phase[p].x)); };
    auto begins = [&](int flags) { return (wave + (flags >> 16 & 7)) & (kStrWaves - 1); };      // this wave's first quad
    const char* ibase = base_of(0);
    auto settle = [&] {                                   // on to a linear of which this wave has a quad
        while (iq >= itotal && it < tokens) {
            if (++ip == phases) { ip = 0; it++; }
            const int4 ph = T.phase[ip];
            itotal = word(ph.z);
            ibase = reinterpret_cast<const char*>(((unsigned long long)(unsigned)word(ph.y) << 32) | (unsigned)word(ph.x));
            if constexpr (MOE) {
                const int4 gr = T.group[ip];
                const int flags = word(gr.w);
                iq = begins(flags);
                iorder = flags & 0xFFFF;
                igroup = word(gr.z);
            } else {
                iq = wave;
                igroup = ip;
            }
        }
    };
    auto known = [&] {                                    // an expert's weights have no address before the choice
        if (it >= tokens) return false;
        if (!MOE || iorder == 0) return true;
        const bool yes = flag(L.chosen) >= it * routed + iorder;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");         // the addresses are read behind the flag
        return yes;
    };
    auto ask = [&] {
        if (MOE && iorder) ibase = base_of(ip);
        quad_to_lds(ibase, (unsigned)iq * kQuad + lane * 16, dst + islot * kQuad);
        islot = islot + 1 == slots ? 0 : islot + 1;
        ahead++;
        iq += kStrWaves;
        settle();
    };
    settle();
    int slot = 0, n = 0;
    float xr[4][CE];
    for (int ct = 0; ct < tokens; ct++)
        for (int cp = 0; cp < phases; cp++) {
            const int4 ph = T.phase[cp];
            int4 gr = make_int4(0, 0, cp, (int)(3u << 30));
            if constexpr (MOE) gr = T.group[cp];
            const int total = word(ph.z), rq = word(ph.w), flags = word(gr.w), cgroup = MOE ? word(gr.z) : cp;
            const bool half = MOE && rq == 0, first = !MOE || (flags >> 30 & 1), last = !MOE || flags < 0;
            const int segs = half ? 2 : 4 * rq, from = MOE ? begins(flags) : wave;
            if (!first && !last && from >= total) continue;
            const float* x0 = MOE ? xs + word(gr.x) : xs;
            float* sums = red + (MOE ? word(gr.y) : cp == head ? head_off : 0);
            int at = from;                                // place of the quad in its row
            while (!half && at >= rq) at -= rq;
            const bool held = half || kStrWaves % rq == 0;             // the same in all rows
            auto vector = [&](float (&x)[4][CE], int at) {
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int q = 0; q < PL; q++) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(x0 + ((q * segs + (half ? i & 1 : 4 * at + i)) * 64 + lane) * 4);
#pragma unroll
                        for (int e = 0; e < 4; e++) x[i][q * 4 + e] = v[e];
                    }
            };
            auto read = [&](i32x4 (&u)[4]) {
#pragma unroll
                for (int i = 0; i < 4; i++) u[i] = *reinterpret_cast<const i32x4*>(mine + slot * kQuad + i * 1024 + lane * 16);
                slot = slot + 1 == slots ? 0 : slot + 1;
                ahead--;
            };
            auto dots = [&](const i32x4 (&u)[4], const float (&x)[4][CE], float (&s)[4]) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float wv[CE];
                    Chunk<ET>::unpack(make_uint4(u[i][0], u[i][1], u[i][2], u[i][3]), wv);
                    s[i] = 0.0f;
#pragma unroll
                    for (int e = 0; e < CE; e++) s[i] = fma_f(wv[e], x[i][e], s[i]);
                }
            };
            auto dot = [&](const i32x4 (&u)[4], const float (&x)[4][CE]) {
                float s[4];
                dots(u, x, s);
                return (s[0] + s[1]) + (s[2] + s[3]);
            };
            auto next = [&] {
                at += kStrWaves;
                while (at >= rq) at -= rq;
            };
            auto same = [&] { return igroup == cgroup && it == ct; };
            // When the ring is full, the linear's first quads move into registers.
            i32x4 u[2][4];
            bool taken = false;
            if (first) {
                n++;
                while (flag(L.ready) < (FREE ? kSvcWaves * n : n)) {
                    if (ahead < slots && known()) {
                        ask();
                        if constexpr (!FREE) wait_quads(0);
                    } else if (!taken && ahead == slots && ahead >= 2 && !half && from + kStrWaves < total) {
                        wait_quads(ahead - 2);
                        read(u[0]);
                        read(u[1]);
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the slots have been read
                        taken = true;
                    } else {
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                if constexpr (FREE) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                else __syncthreads();                     // the vector is there
                while (ahead < slots && same()) ask();
            }
            // experts' gate/up: all on the one vector, which is still there
            if (from < total && (first || !held || half || word(gr.x) != 0 || from != wave)) vector(xr, at);
            int q = from;
            for (; !half && q + kStrWaves < total; q += 2 * kStrWaves) {       // two at a time, which hide each other's latencies
                if (!taken) {
                    wait_quads(ahead - 2);
                    read(u[0]);
                    read(u[1]);
                }
                float v[2];
                if (held) {
                    v[0] = dot(u[0], xr);
                    v[1] = dot(u[1], xr);
                } else {
                    float x2[4][CE];
                    if (q > from) vector(xr, at);
                    next();
                    vector(x2, at);
                    next();
                    v[0] = dot(u[0], xr);
                    v[1] = dot(u[1], x2);
                }
                if (!taken) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the slots have been read
                    if (same()) ask();
                    if (same()) ask();
                }
                taken = false;
                multi_sum_step<2, 1>(v, lane);
                if (lane < 2) sums[q + kStrWaves * lane] = v[0];
            }
            for (; q < total; q += kStrWaves) {           // the last one, or all halves
                wait_quads(ahead - 1);
                read(u[0]);
                if (!held && q > from) vector(xr, at);
                float s[4];
                dots(u[0], xr, s);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (same()) ask();
                float v[2] = {s[0] + s[1], s[2] + s[3]};
                if (half) {
                    multi_sum_step<2, 1>(v, lane);
                    if (lane < 2) sums[2 * q + lane] = v[0];
                } else {
                    const float o = wave_sum(v[0] + v[1]);
                    if (lane == 0) sums[q] = o;
                }
            }
            if (last) {
                if constexpr (FREE) add(L.done);
                else __syncthreads();                     // the sums are there
                while (flag(L.sent) < n) __builtin_amdgcn_s_sleep(1);      // they leave first: a store, too, stands in line
            }
        }
}

// bfloat16 weights on the matrix cores.  A quad is 1 KiB, 512 of k, of four neighbouring rows (a block); a float32 vector is the sum of three
// bfloat16 parts to 24 bits, and their products with the weights are exact in float32.  An instruction (16 x 16 x 32) takes 256 bytes of each row: its rows
// are 4 weight rows x 4 pieces of k, its columns 3 parts x the same 4 pieces, and where the pieces meet are the sums.  So 512 weights take one
// instruction for 20 of a lane's own, operands come in requests of 1 KiB of one row, and a wave that stays in a block of k keeps the vector in 16 registers.
// In LDS 16 bytes c of row r lie at place c ^ 2r, of part p at c ^ 2p: eight neighbouring lanes that read 16 bytes each are on different banks.  (Counted: a quad takes 86
// cycles of its CU's LDS, 23 of them conflicts; the matrix cores are busy for 3 % of a token.)
__device__ __forceinline__ void block_to_lds(const char* base, const unsigned (&voff)[4], unsigned dst) {
    unsigned saved_m0;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %6\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %5 nt\n\t"
                 "s_add_u32 m0, m0, 0x400\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %2, %5 nt\n\t"
                 "s_add_u32 m0, m0, 0x400\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %3, %5 nt\n\t"
                 "s_add_u32 m0, m0, 0x400\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %4, %5 nt\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved_m0) : "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(base), "s"(dst) : "memory", "scc");
}
template <bool MOE, bool FREE>
__device__ __forceinline__ void stream_parts(WalkLds& L, WalkTables T, const float* xs, float* red, const char* ring, int slots, int phases, int tokens, int routed, int head, int head_off) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) - kSvcWaves;
    auto word = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const char* mine = ring + (size_t)wave * slots * kQuad;
    const unsigned dst = word((int)(unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)mine);
    // as an operand's row lane & 15 is row or part lane & 3 of piece lane >> 2 & 3, of which this lane has 16 bytes
    const int row = lane & 3, part = min(row, 2), piece = lane >> 4 << 2 | (lane >> 2 & 3);
    const bool meets = row < 3 && (lane >> 2 & 3) == lane >> 4;
    const char* get = mine + row * 1024 + (piece ^ 2 * row) * 16;
    // what is asked for next: block ikb of rows 4 irg .. of linear ip of token it
    int ip = 0, it = 0, irg = 0, ikb = wave, irows = 0, inkb = 1, iorder = 0, igroup = 0, islot = 0, ahead = 0;      // ahead: quads asked for and not taken in
    auto address = [&](const int4& ph) { return reinterpret_cast<const char*>(((unsigned long long)(unsigned)word(ph.y) << 32) | (unsigned)word(ph.x)); };
    auto begins = [&](int flags) { return (wave + (flags >> 16 & 7)) & (kStrWaves - 1); };      // this wave's first quad
    const char* ibase = nullptr;
    auto start = [&] {
        const int4 ph = T.phase[ip];
        irows = word(ph.z);
        inkb = word(ph.w);
        ibase = address(ph);
        irg = 0;
        ikb = wave;
        igroup = ip;
        if constexpr (MOE) {
            const int4 gr = T.group[ip];
            const int flags = word(gr.w);
            ikb = begins(flags);
            iorder = flags & 0xFFFF;
            igroup = word(gr.z);
        }
    };
    auto settle = [&] {                                   // on to a linear of which this wave has a quad
        for (;;) {
            while (ikb >= inkb) { ikb -= inkb; irg++; }
            if (4 * irg < irows || it >= tokens) break;
            if (++ip == phases) { ip = 0; it++; }
            start();
        }
    };
    auto known = [&] {                                    // an expert's weights have no address before the choice
        if (it >= tokens) return false;
        if (!MOE || iorder == 0) return true;
        const bool yes = flag(L.chosen) >= it * routed + iorder;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");         // the addresses are read behind the flag
        return yes;
    };
    auto ask = [&] {
        if (MOE && iorder) ibase = address(T.phase[ip]);
        const unsigned stride = (unsigned)inkb * 1024u;
        const int left = irows - 1 - 4 * irg;             // a last group of fewer rows has the last one again
        unsigned voff[4];
#pragma unroll
        for (int r = 0; r < 4; r++) voff[r] = (unsigned)min(r, left) * stride + (unsigned)(lane ^ 2 * r) * 16u;
        block_to_lds(ibase + (size_t)(4 * irg) * stride + (size_t)ikb * 1024, voff, dst + islot * kQuad);
        islot = islot + 1 == slots ? 0 : islot + 1;
        ahead++;
        ikb += kStrWaves;
        settle();
    };
    start();
    settle();
    int slot = 0, n = 0;
    i32x4 x[4];                                           // the vector's operands of a block
    for (int ct = 0; ct < tokens; ct++)
        for (int cp = 0; cp < phases; cp++) {
            const int4 ph = T.phase[cp];
            int4 gr = make_int4(0, 0, cp, (int)(3u << 30));
            if constexpr (MOE) gr = T.group[cp];
            const int rows = word(ph.z), nkb = word(ph.w), flags = word(gr.w), cgroup = MOE ? word(gr.z) : cp;
            const bool first = !MOE || (flags >> 30 & 1), last = !MOE || flags < 0;
            const int total = (rows + 3) / 4 * nkb, from = MOE ? begins(flags) : wave;
            if (!first && !last && from >= total) continue;
            const char* x0 = reinterpret_cast<const char*>(MOE ? xs + word(gr.x) : xs);
            const char* x_get = x0 + part * nkb * 1024 + (piece ^ 2 * part) * 16;
            float* sums = red + (MOE ? word(gr.y) : cp == head ? head_off : 0);
            const bool held = nkb <= kStrWaves;           // one block of k per wave
            const int per = min(nkb, kStrWaves);          // sums of a row
            auto vector = [&](i32x4 (&v)[4], int kb) {
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const i32x4*>(x_get + kb * 1024 + i * 256);
            };
            auto read = [&](i32x4 (&u)[4]) {
#pragma unroll
                for (int i = 0; i < 4; i++) u[i] = *reinterpret_cast<const i32x4*>(get + slot * kQuad + i * 256);
                slot = slot + 1 == slots ? 0 : slot + 1;
                ahead--;
            };
            auto products = [&](const i32x4 (&u)[4], const i32x4 (&v)[4], f32x4& acc) {
#pragma unroll
                for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, u[i]), __builtin_bit_cast(bf16x8, v[i]), acc, 0, 0, 0);
            };
            // the sums of G groups of rows leave; group i is i * step behind rg
            bool bad = false;
            auto leave = [&](auto groups, float (&v)[4 * decltype(groups)::value], int rg, int step) {
                constexpr int G = decltype(groups)::value;
#pragma unroll
                for (int i = 0; i < 4 * G; i++) v[i] = meets ? v[i] : 0.0f;
                multi_sum_step<4 * G, 1>(v, lane);
                const int of = multi_row<4 * G>(lane & (4 * G - 1)), r = 4 * (rg + of / 4 * step) + (of & 3);
                bad = bad || isnan(v[0]);
                if (lane < 4 * G) sums[r * per + (from & (per - 1))] = v[0];
            };
            auto same = [&] { return igroup == cgroup && it == ct; };
            // When the ring is full, the linear's first quads move into registers.
            i32x4 u[4][4];
            int taken = 0;
            auto all_read = [&] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };      // the slots that have been read are free
            if (first) {
                n++;
                while (flag(L.ready) < (FREE ? kSvcWaves * n : n)) {
                    if (ahead < slots && known()) {
                        ask();
                        if constexpr (!FREE) wait_quads(0);
                    } else if (taken < (FREE && held ? 4 : 2) && ahead == slots && from + kStrWaves * taken < total) {
                        wait_quads(ahead - 1);
                        if (taken == 0) read(u[0]);
                        else if (taken == 1) read(u[1]);
                        else if (taken == 2) read(u[2]);
                        else read(u[3]);
                        all_read();
                        taken++;
                    } else {
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                if constexpr (FREE) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                else __syncthreads();                     // the vector is there
                while (ahead < slots && same()) ask();
            }
            auto fetch = [&](int count) {                 // the next quads, of which the first may be there already
                if (taken < 1) {
                    wait_quads(ahead - count);
                    read(u[0]);
                    if (count == 2) read(u[1]);
                } else if (taken < count) {
                    wait_quads(ahead - 1);
                    read(u[1]);
                }
            };
            auto used = [&] {                             // two of them: the others move up
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    u[0][i] = u[2][i];
                    u[1][i] = u[3][i];
                }
                taken = max(taken - 2, 0);
            };
            auto refill = [&] {
                all_read();
                while (ahead < slots && same()) ask();
            };
            int kb = from, rg = 0, q = from;
            while (kb >= nkb) { kb -= nkb; rg++; }
            if (held) {
                // experts' gate/up: all on the one vector, which is still there
                if (from < total && (first || word(gr.x) != 0 || from != wave)) vector(x, kb);
                const int step = kStrWaves / nkb;
                for (; q + kStrWaves < total; q += 2 * kStrWaves, rg += 2 * step) {       // two at a time, which hide each other's latencies
                    fetch(2);
                    f32x4 acc[2] = {};
                    products(u[0], x, acc[0]);
                    products(u[1], x, acc[1]);
                    refill();
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) v[i] = acc[i / 4][i % 4];
                    leave(std::integral_constant<int, 2>(), v, rg, step);
                    used();
                }
                if (q < total) {
                    fetch(1);
                    f32x4 acc = {};
                    products(u[0], x, acc);
                    refill();
                    float v[4] = {acc[0], acc[1], acc[2], acc[3]};
                    leave(std::integral_constant<int, 1>(), v, rg, 0);
                }
            } else {                                      // several blocks of each group of rows
                f32x4 acc = {};
                auto block = [&](const i32x4 (&u)[4], const i32x4 (&v)[4]) {
                    products(u, v, acc);
                    kb += kStrWaves;
                    if (kb < nkb) return;
                    float o[4] = {acc[0], acc[1], acc[2], acc[3]};
                    leave(std::integral_constant<int, 1>(), o, rg, 0);
                    acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    rg++;
                    kb -= nkb;
                };
                for (; q < total; q += 2 * kStrWaves) {
                    const int count = q + kStrWaves < total ? 2 : 1;
                    fetch(count);
                    taken = 0;
                    i32x4 x2[4];
                    vector(x, kb);
                    vector(x2, kb + kStrWaves < nkb ? kb + kStrWaves : kb + kStrWaves - nkb);
                    refill();
                    block(u[0], x);
                    if (count == 2) block(u[1], x2);
                }
            }
            // Not a number may be of the parts' own making, where an infinite weight meets parts of zero or of both signs or a value is infinite (what is left of it is
            // no number): the same sum with a float32 product per weight has the right of it.
            if (__builtin_amdgcn_ballot_w64(bad)) {
                all_read();
                for (int q = from; q < total; q += kStrWaves) {
                    const int r = q / nkb * 4, kb0 = q % nkb;
                    if (!held && kb0 >= kStrWaves) continue;
                    for (int i = 0; i < 4; i++) {
                        float& sum = sums[(r + i) * per + (from & (per - 1))];
                        if (!isnan(sum)) continue;
                        const char* w = address(T.phase[cp]) + (size_t)min(r + i, rows - 1) * nkb * 1024;
                        float s = 0.0f;
                        for (int kb = kb0; kb < nkb; kb += kStrWaves) {
                            float wv[8];
                            const i32x4 u = *global(reinterpret_cast<const i32x4*>(w + (size_t)kb * 1024 + lane * 16));
                            Chunk<bf16_t>::unpack(make_uint4(u[0], u[1], u[2], u[3]), wv);
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                auto at = [&](int p) { return __uint_as_float((unsigned)*reinterpret_cast<const unsigned short*>(x0 + (size_t)p * nkb * 1024 + ((kb * 64 + lane) ^ 2 * p) * 16 + 2 * e) << 16); };
                                const float h = at(0);
                                s = fma_f(wv[e], fabsf(h) < INFINITY ? (h + at(1)) + at(2) : h, s);
                            }
                        }
                        s = wave_sum(s);
                        if (lane == 0) sum = s;
                    }
                }
            }
            if (last) {
                if constexpr (FREE) add(L.done);
                else __syncthreads();                     // the sums are there
                while (flag(L.sent) < n) __builtin_amdgcn_s_sleep(1);      // they leave first: a store, too, stands in line
            }
        }
}

// ---- service waves ----------------------------------------------------------------------------------------------------
template <typename ET, int QW, int KIND, bool PARTS>
struct Service {
    static constexpr int CE = Chunk<ET>::N, PL = CE / 4, QE = kQuad / sizeof(ET);      // elements of a quad
    static constexpr bool FREE = kFree<KIND>;
    const WalkArgs& a;
    WalkLds& L;
    WalkTables T;
    MixerLds& M;
    float *xs, *red;
    Wait wait;
    const int t, lane, wave, wg;
    float *now, *other;                                   // the two sets
    f32x4 x[QW];                                          // residual: float4 t + 256 i
    int normed = 0;                                       // L.norm in turn
    int meetings = 0, ready = 0, sums = 0, sent = 0, chosen = 0;

    __device__ __forceinline__ Service(const WalkArgs& a_, WalkLds& L_, WalkTables T_, float* xs_, float* red_)
        : a(a_), L(L_), T(T_), M(*reinterpret_cast<MixerLds*>(xs_)), xs(xs_), red(red_), wait{a_, false}, t(threadIdx.x), lane(threadIdx.x & 63), wave(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))), wg(blockIdx.x) {}
    // The thread's number as the compiler does not know it: addresses made of it are not kept in registers from layer to layer.
    __device__ __forceinline__ int opaque() const {
        int v = threadIdx.x;
        asm volatile("" : "+v"(v));
        return v;
    }
    // Barrier of the service waves among themselves: the others may stand still for the sake of their requests.
    __device__ __forceinline__ void meet() {
        meetings += kSvcWaves;
        add(L.met);
        while (__hip_atomic_load(&L.met, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < meetings) {}
    }
    __device__ __forceinline__ void say(int& f, int n) {
        if (t == 0) __hip_atomic_store(&f, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    // to the stream waves: the vector is there
    __device__ __forceinline__ void vector_done() {
        if constexpr (FREE) {
            add(L.ready);
        } else {
            say(L.ready, ++ready);
            __syncthreads();
        }
    }
    // until the sums of all stream waves are there; then, behind put(): they have left
    __device__ __forceinline__ void sums_there() {
        if constexpr (FREE) {
            sums += kStrWaves;
            while (__hip_atomic_load(&L.done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < sums) __builtin_amdgcn_s_sleep(1);
        } else {
            __syncthreads();
        }
    }
    __device__ __forceinline__ void sums_done() { say(L.sent, ++sent); }
    __device__ __forceinline__ void put(unsigned at, float v) {
        store_past(now + at, unset(v) ? __int_as_float(0x7FC00000) : v);
        unput(at);
    }
    __device__ __forceinline__ void unput(unsigned at) { store_past(other + at, __int_as_float((int)kUnset)); }
    __device__ __forceinline__ void put_x(int k, int c, f32x4 v, int off = 0) {      // float4 c of the vector of k that starts at element off
        if constexpr (PARTS) {                            // part p's 16 bytes c at place c ^ 2p, see stream_parts
            char* x = reinterpret_cast<char*>(xs) + 6 * off + 8 * (c & 1);
#pragma unroll
            for (int p = 0; p < 3; p++) {
                uint2 o;
                o.x = __builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u);
                o.y = __builtin_amdgcn_perm(__float_as_uint(v[3]), __float_as_uint(v[2]), 0x07060302u);
                *reinterpret_cast<uint2*>(x + 2 * p * k + ((c >> 1) ^ 2 * p) * 16) = o;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] -= __uint_as_float(__float_as_uint(v[e]) & 0xFFFF0000u);
            }
        } else {
            const int at = PL == 1 ? c : (c & 1) * (k / CE) + (c >> 1);
            *reinterpret_cast<f32x4*>(xs + off + 4 * at) = v;
        }
    }
    // total of local row r of k
    __device__ __forceinline__ float total(int k, int r, int off = 0) const {
        const int n = walk_sums(PARTS, k, QE);
        const float* p = red + off + r * n;
        if constexpr (PARTS) {
            if (n == 2) return p[0] + p[1];
            f32x4 v = *reinterpret_cast<const f32x4*>(p);
            if (n == 8) v += *reinterpret_cast<const f32x4*>(p + 4);
            return (v[0] + v[1]) + (v[2] + v[3]);
        }
        float s = p[0];
        for (int i = 1; i < n; i++) s += p[i];
        return s;
    }
    // A vector of k words as it is
    __device__ __forceinline__ void take(unsigned at, int k) {
        const int t = opaque();
        const int n4 = k / 4;
        meet();                                           // the mixer's values lie where the vector will
        auto some = [&](auto n, int c0) {
            constexpr int N = decltype(n)::value;
            unsigned off[N];
            f32x4 v[N];
#pragma unroll
            for (int i = 0; i < N; i++) off[i] = 16u * (unsigned)min(c0 + t + kSvcT * i, n4 - 1);
            poll_words<N>(now + at, off, c0 + wave * 64 < n4, v, wait);
#pragma unroll
            for (int i = 0; i < N; i++)
                if (c0 + t + kSvcT * i < n4) put_x(k, c0 + t + kSvcT * i, v[i]);
        };
        int c0 = 0;
        while (n4 - c0 > 4 * kSvcT) { some(std::integral_constant<int, 8>(), c0); c0 += 8 * kSvcT; }
        if (n4 - c0 > 2 * kSvcT) some(std::integral_constant<int, 4>(), c0);
        else if (n4 - c0 > kSvcT) some(std::integral_constant<int, 2>(), c0);
        else if (n4 - c0 > 0) some(std::integral_constant<int, 1>(), c0);
        vector_done();
    }
    // x += y (normed and times gb where there is one) + the embedding of `again`; the vector becomes norm(x) * g.
    __device__ __forceinline__ void norm(bool have, unsigned at, const float* gb, const float* g, int again_token) {
        const int t = opaque();
        const int n4 = a.width / 4;
        f32x4 gv[QW], gbv[QW];
        unsigned off[QW];
#pragma unroll
        for (int i = 0; i < QW; i++) {
            const int c = min(t + kSvcT * i, n4 - 1);
            off[i] = 16u * (unsigned)c;
            gv[i] = *global(reinterpret_cast<const f32x4*>(g + 4 * c));
            if (have && gb) gbv[i] = *global(reinterpret_cast<const f32x4*>(gb + 4 * c));
        }
        if (have) {
            f32x4 y[QW];
            poll_words<QW>(now + at, off, wave * 64 < n4, y, wait);
            float rs = 0.0f;
            if (gb) {
                float ss = 0.0f;
#pragma unroll
                for (int i = 0; i < QW; i++)
                    if (t + kSvcT * i < n4)
#pragma unroll
                        for (int e = 0; e < 4; e++) ss = fma_f(y[i][e], y[i][e], ss);
                rs = root(ss, (float)a.width);
            }
#pragma unroll
            for (int i = 0; i < QW; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) x[i][e] = gb ? x[i][e] + y[i][e] * rs * gbv[i][e] : x[i][e] + y[i][e];
        }
        if (again_token >= 0)
#pragma unroll
            for (int i = 0; i < QW; i++) x[i] += embedding(again_token, min(t + kSvcT * i, n4 - 1));
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < QW; i++)
            if (t + kSvcT * i < n4)
#pragma unroll
                for (int e = 0; e < 4; e++) ss = fma_f(x[i][e], x[i][e], ss);
        const float rx = root(ss, (float)a.width);
#pragma unroll
        for (int i = 0; i < QW; i++) {
            f32x4 h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = x[i][e] * rx * gv[i][e];
            if (t + kSvcT * i < n4) put_x(a.width, t + kSvcT * i, h);
        }
        vector_done();
    }
    // 1 / rms of `count` values from the threads' sums of squares
    __device__ __forceinline__ float root(float ss, float count) {
        ss = wave_sum(ss);
        if (lane == 0) L.norm[normed][wave] = ss;
        meet();
        const float* n = L.norm[normed];
        normed ^= 1;
        return 1.0f / sqrtf(((n[0] + n[1]) + (n[2] + n[3])) / count + a.eps);
    }
    __device__ __forceinline__ f32x4 embedding(int token, int c) const {
        const bf16x4 b = *global(reinterpret_cast<const bf16x4*>(a.embed + (size_t)token * a.width + 4 * c));
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = (float)b[e] * a.embed_scale;
        return v;
    }
    __device__ __forceinline__ void embed(int token) {
        const int t = opaque();
#pragma unroll
        for (int i = 0; i < QW; i++) x[i] = embedding(token, min(t + kSvcT * i, a.width / 4 - 1));
    }

    // ---- attention over shared key/value rows (see shared_kv_attn.hip): a workgroup takes a split of the rows for one query head;
    // the heads that share rows are on one die.  (All four heads of a key/value head in one workgroup and four times the splits: 2.9 us
    // instead of 1.9 for 1531 rows, for the norms and sums of four heads.)  A split has a batch of rows for every group of lanes at
    // least: up to 128 rows of 64 (64 of 128, half as many in float32) need no join, which is 2.4 us.
    template <int D>
    __device__ __forceinline__ void shared_kv(RunPtr r, int pos) {
        const int t = opaque(), lane = t & 63;
        constexpr int LPK = D / CE, KS = kSvcT / LPK, U = 4, N = CE, PW = walk_part(D);
        const int G = r->kv_heads, rep = r->rep, S = r->splits, g = wg % G, idx = wg / G, split = idx / rep, head = g * rep + idx % rep;
        const int held = pos, per = max(((held + S - 1) / S + KS - 1) / KS * KS, U * KS), ns = max((held + per - 1) / per, 1);
        const int first = split * per, last = min(held, first + per);
        const int lc = lane % LPK, ks = wave * (64 / LPK) + lane / LPK, col = lc * CE;
        const unsigned part = r->x_part + (unsigned)((head * S + split) * PW);
        if (split < ns && pos < r->capacity) {            // others only take part in the join
            const bool own = split == 0;
            const auto* rows = global(static_cast<const ET*>(r->rows)) + (size_t)g * r->capacity * D;
            const auto* inv = global(r->inv_rms) + (size_t)g * r->capacity;
            i32x4 ua[U], ub[U];
            float ra[U], rb[U], wv[N];
            auto rows_at = [&](int b, int i) { return i == 0 || first + (b * U + i) * KS < last; };
            auto load = [&](int b, i32x4 (&u)[U], float (&ri)[U]) {
#pragma unroll
                for (int i = 0; i < U; i++) {
                    if (!rows_at(b, i)) break;
                    const int key = min(first + (b * U + i) * KS + ks, last - 1);
                    u[i] = *reinterpret_cast<const Global<i32x4>*>(rows + (size_t)key * D + col);
                    ri[i] = inv[key];
                }
            };
            const int nb = last > first ? (last - first + U * KS - 1) / (U * KS) : 0;
            if (nb > 0) load(0, ua, ra);
#pragma unroll
            for (int q = 0; q < N; q += 4) {
                const f32x4 v = *global(reinterpret_cast<const f32x4*>(r->kv_norm + col + q));
#pragma unroll
                for (int e = 0; e < 4; e++) wv[q + e] = v[e];
            }
            float f = r->scale * kWalkLog2e;
            if (r->temp_coef != 0.0f) f *= 1.0f + r->temp_coef * logf((float)((pos + 1) / r->temp_every) + 1.0f);
            if (wave == 0) {                              // the query, and the row of this step, into LDS
                unsigned off[1];
                f32x4 v[1];
                const bool isq = lane < D / 4, isk = own && lane >= D / 4 && lane < D / 2;
                off[0] = isq ? 4u * (unsigned)(head * D) + 16u * (unsigned)lane : 4u * (unsigned)(r->n_et + g * D) + 16u * (unsigned)(isk ? lane - D / 4 : 0);
                poll_words<1>(now + r->x_in, off, isq || isk, v, wait);
                if (isq) *reinterpret_cast<f32x4*>(M.q + 4 * lane) = v[0];
                if (isk) *reinterpret_cast<f32x4*>(M.kx + 4 * (lane - D / 4)) = v[0];
            }
            meet();
            float qv[N], acc[N], m = -1e30f, l = 0.0f;    // m finite, so that differences stay defined
            {
                float ss = 0.0f;
#pragma unroll
                for (int q = 0; q < N; q += 4) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(M.q + col + q);
#pragma unroll
                    for (int e = 0; e < 4; e++) { qv[q + e] = v[e]; ss = fma_f(v[e], v[e], ss); }
                }
                const float s = f / sqrtf(lanes_sum<LPK>(ss) / (float)D + a.eps);
#pragma unroll
                for (int e = 0; e < N; e++) { qv[e] *= s * wv[e]; acc[e] = 0.0f; }
            }
            auto score = [&](const float (&v)[N]) {
                float s = 0.0f;
#pragma unroll
                for (int e = 0; e < N; e++) s = fma_f(qv[e], v[e], s);
                return lanes_sum<LPK>(s);
            };
            auto take_rows = [&](int b, const i32x4 (&u)[U], const float (&ri)[U]) {
                float s[U], mx = m;
#pragma unroll
                for (int i = 0; i < U; i++) {
                    s[i] = -INFINITY;
                    if (!rows_at(b, i)) continue;
                    float v[N];
                    Chunk<ET>::unpack(make_uint4(u[i][0], u[i][1], u[i][2], u[i][3]), v);
                    const float z = score(v) * ri[i];
                    if (first + (b * U + i) * KS + ks < last) s[i] = z;
                    mx = fmaxf(mx, s[i]);
                }
                const float al = __builtin_amdgcn_exp2f(m - mx);
                m = mx;
                l *= al;
#pragma unroll
                for (int e = 0; e < N; e++) acc[e] *= al;
#pragma unroll
                for (int i = 0; i < U; i++) {
                    if (!rows_at(b, i)) break;
                    const float p = __builtin_amdgcn_exp2f(s[i] - mx);
                    l += p;
                    float v[N];
                    Chunk<ET>::unpack(make_uint4(u[i][0], u[i][1], u[i][2], u[i][3]), v);
#pragma unroll
                    for (int e = 0; e < N; e++) acc[e] = fma_f(p, v[e], acc[e]);
                }
            };
            for (int b = 0; b < nb; b += 2) {
                if (b + 1 < nb) load(b + 1, ub, rb);
                take_rows(b, ua, ra);
                if (b + 1 >= nb) break;
                if (b + 2 < nb) load(b + 2, ua, ra);
                take_rows(b + 1, ub, rb);
            }
            if (own && wave == 0) {                       // the row of this step: the first group of lanes takes it in, one head's workgroup stores it
                float v[N], ss = 0.0f;
#pragma unroll
                for (int e = 0; e < N; e++) {
                    v[e] = M.kx[col + e];
                    ss = fma_f(v[e], v[e], ss);
                    v[e] = (float)(ET)v[e];               // as a later step reads it
                }
                const float ri = 1.0f / sqrtf(lanes_sum<LPK>(ss) / (float)D + a.eps);
                if (ks == 0 && head == g * rep) {
                    const size_t row = (size_t)g * r->capacity + pos;
                    __attribute__((aligned(16))) ET o[N];
#pragma unroll
                    for (int e = 0; e < N; e++) o[e] = (ET)v[e];
                    float* dst = reinterpret_cast<float*>(static_cast<ET*>(r->rows) + row * D + col);
#pragma unroll
                    for (int i = 0; i < 4; i++) store_past(dst + i, reinterpret_cast<const float*>(o)[i]);
                    if (lc == 0) store_past(r->inv_rms + row, ri);
                }
                const float z = score(v) * ri, sc = ks == 0 ? z : -INFINITY;
                const float mx = fmaxf(m, sc), al = __builtin_amdgcn_exp2f(m - mx), p = __builtin_amdgcn_exp2f(sc - mx);
                m = mx;
                l = l * al + p;
#pragma unroll
                for (int e = 0; e < N; e++) acc[e] = fma_f(p, v[e], acc[e] * al);
            }
            // the groups of lanes of a wave meet
            const float mw = wave_max(m), w = __builtin_amdgcn_exp2f(m - mw), lw = wave_sum(lc == 0 ? l * w : 0.0f);
            if (lane == 0) { L.m[wave] = mw; L.l[wave] = lw; }
#pragma unroll
            for (int e = 0; e < N; e++) acc[e] *= w;
            constexpr int LEFT = N / (64 / LPK) > 0 ? N / (64 / LPK) : 1;
            multi_sum_step<N, LPK>(acc, lane);
            int r0 = 0;
#pragma unroll
            for (int mask = LPK, half = N / 2; mask < 64 && half > 0; mask *= 2, half /= 2)
                if (lane & mask) r0 += half;
#pragma unroll
            for (int i = 0; i < LEFT; i++) M.sums[wave][col + r0 + i] = acc[i];
            meet();
            // and the waves
            if (t < D) {
                const bool sink = ns == 1 && r->sink;
                float mt = fmaxf(fmaxf(L.m[0], L.m[1]), fmaxf(L.m[2], L.m[3])), v = 0.0f, lt = 0.0f;
                if (sink) mt = fmaxf(mt, 0.0f);
#pragma unroll
                for (int i = 0; i < kSvcWaves; i++) {
                    const float e = __builtin_amdgcn_exp2f(L.m[i] - mt);
                    v += e == 0.0f ? 0.0f : M.sums[i][t] * e;
                    lt = fma_f(L.l[i], e, lt);
                }
                if (sink) lt += __builtin_amdgcn_exp2f(-mt);
                if (ns == 1) {
                    put(r->x_att + (unsigned)(head * D + t), v / lt);
                    unput(part + t);
                    if (t < 2) unput(part + D + t);
                } else {
                    put(part + t, v);
                    if (t == 0) { put(part + D, mt); put(part + D + 1, lt); }
                }
            }
        } else if (split < S) {
            for (int i = t; i < D + 2; i += kSvcT) unput(part + i);
        }
        // the join: columns split * cw .. of the head belong to this workgroup; a lane per split and four columns
        if (ns > 1 && split < S && wave == 0) {
            const int cw = D / S, s = lane & (S - 1), c4 = lane / S, c = split * cw + 4 * c4;
            const bool cols = 4 * c4 < cw, mine = cols && s < ns;
            const unsigned at = 4u * (unsigned)((head * S + (mine ? s : 0)) * PW);
            unsigned off[2] = {at + 4u * (unsigned)(mine ? c : 0), at + 4u * (unsigned)D};
            f32x4 v[2];
            // the words behind the two of the second piece are never set
            poll_words<2, 2>(now + r->x_part, off, mine, v, wait);
            const float ms = mine ? v[1][0] : -INFINITY;
            float mt = ms;
            group(S, [&](auto k) { mt = fmaxf(mt, lane_xor_f<decltype(k)::value>(mt)); });
            if (r->sink) mt = fmaxf(mt, 0.0f);
            const float e = mine ? __builtin_amdgcn_exp2f(ms - mt) : 0.0f;
            float o[5];
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = e == 0.0f ? 0.0f : v[0][i] * e;
            o[4] = e == 0.0f ? 0.0f : v[1][1] * e;
            group(S, [&](auto k) {
#pragma unroll
                for (int i = 0; i < 5; i++) o[i] += lane_xor_f<decltype(k)::value>(o[i]);
            });
            const float lt = r->sink ? o[4] + __builtin_amdgcn_exp2f(-mt) : o[4];
            if (cols && s < 4) put(r->x_att + (unsigned)(head * D + c + s), (s == 0 ? o[0] : s == 1 ? o[1] : s == 2 ? o[2] : o[3]) / lt);
        }
    }

    // ---- gated linear attention: a workgroup has a slice of `cs` columns of a head's state.  The state does not hang on the step and is on
    // its way under the wait.  The head's norm needs all slices: the outputs leave times the norm's weight and the gate, with the slice's
    // sum of squares (in copies: a line that all workgroups ask for has them stand in line, 3 us), and who reads them divides (take_heads).  (A kernel with a workgroup per head: 8.2 us on 16 or 32 CUs.)
    __device__ __forceinline__ void gla(RunPtr r, int pos) {
        const int t = opaque(), lane = t & 63;
        constexpr int D = kWalkDim, NR = kWalkGlaRank;
        const int H = r->heads, NS = r->splits, cs = D / NS, h = wg % H, slice = wg / H, HD = H * D;
        if (slice >= NS) return;
        const int qd = cs / 4, c0 = slice * cs;           // float4 of a row of the slice
        float* S = r->state + (size_t)h * D * D + c0;
        const bool fresh = pos == 0;                      // a sequence starts from a zero state
        f32x4 st[2];
        int row[2];
        const int c4 = t % qd;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            row[i] = (t + kSvcT * i) / qd;
            if (row[i] < D && !fresh) st[i] = *global(reinterpret_cast<const f32x4*>(S + (size_t)row[i] * D + 4 * c4));
            else st[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        float w[NR], bias = 0.0f;
        if (t < D) {
            const ET* src = static_cast<const ET*>(r->a2) + (size_t)(h * D + t) * kKPad;       // rows are padded with zeros
#pragma unroll
            for (int i = 0; i < NR / CE; i++) {
                float v[CE];
                const i32x4 u = *global(reinterpret_cast<const i32x4*>(src + i * CE));
                Chunk<ET>::unpack(make_uint4(u[0], u[1], u[2], u[3]), v);
#pragma unroll
                for (int e = 0; e < CE; e++) w[i * CE + e] = v[e];
            }
            bias = *global(r->a2_bias + h * D + t);
        }
        const float nw = t < cs ? *global(r->head_norm + c0 + t) : 0.0f;
        float *sq = M.q, *sk = M.q + D, *sa = M.q + 2 * D, *sv = M.q + 3 * D, *sg = sv + 16, *s1 = sg + 16;
        if (wave == 0) {                                  // query and key
            unsigned off[1] = {4u * (unsigned)((lane < 32 ? 0 : HD) + h * D) + 16u * (unsigned)(lane & 31)};
            f32x4 v[1];
            poll_words<1>(now + r->x_in, off, true, v, wait);
            *reinterpret_cast<f32x4*>((lane < 32 ? sq : sk) + 4 * (lane & 31)) = v[0];
        } else if (wave == 1) {                           // the slice's values and gates, the decay's input
            const int n1 = (r->a_rank + 3) / 4, part = lane < 4 ? 0 : lane < 8 ? 1 : 2, i = part < 2 ? lane & 3 : lane - 8;
            const bool need = part < 2 ? i < qd : i < n1;
            const unsigned at = (unsigned)(part == 0 ? 2 * HD + h * D + c0 : part == 1 ? 3 * HD + h * D + c0 : 4 * HD);
            unsigned off[1] = {4u * at + 16u * (unsigned)(need ? i : 0)};
            f32x4 v[1];
            poll_words<1>(now + r->x_in, off, need, v, wait);
            if (part < 2) *reinterpret_cast<f32x4*>((part == 0 ? sv : sg) + 4 * i) = v[0];
            else if (i < NR / 4) *reinterpret_cast<f32x4*>(s1 + 4 * i) = v[0];         // zeros beyond the rank
        }
        meet();
        if (t < D) {
            float z = bias;
#pragma unroll
            for (int i = 0; i < NR; i++) z = i < r->a_rank ? fma_f(w[i], s1[i], z) : z;
            sa[t] = exp_f<false>(log_sigmoid_f(z) / r->tau);
            sq[t] *= 1.0f / sqrtf((float)D);
        }
        meet();
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        const f32x4 v = *reinterpret_cast<const f32x4*>(sv + 4 * c4);
#pragma unroll
        for (int i = 0; i < 2; i++)
            if (row[i] < D) {
                const float k = sk[row[i]], d = sa[row[i]], q = sq[row[i]];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    st[i][e] = fma_f(k, v[e], fresh ? 0.0f : st[i][e] * d);
                    acc[e] = fma_f(st[i][e], q, acc[e]);
                }
                *(Global<f32x4>*)(S + (size_t)row[i] * D + 4 * c4) = st[i];
            }
        // over the rows: lanes of the same four columns, then the waves
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (qd <= 2) acc[e] += lane_xor_f<2>(acc[e]);
            acc[e] += lane_xor_f<4>(acc[e]);
            acc[e] += lane_xor_f<8>(acc[e]);
            acc[e] += lane_xor_f<16>(acc[e]);
            acc[e] += lane_xor_f<32>(acc[e]);
        }
        if (lane < qd) *reinterpret_cast<f32x4*>(&M.sums[wave][4 * lane]) = acc;
        meet();
        if (wave == 0) {
            float x = 0.0f;
            if (t < cs) {
                x = (M.sums[0][t] + M.sums[1][t]) + (M.sums[2][t] + M.sums[3][t]);
                const float g = sg[t];
                put(r->x_att + (unsigned)(h * D + c0 + t), x * nw * (g * sigmoid_f(g)));
            }
            const float ss = wave_sum(x * x);
            if (t < kWalkCopies) put(r->x_part + (unsigned)(t * kWalkWG + h * NS + slice), ss);
        }
    }
    // The vector of gla(): every head over the root of its mean square.
    __device__ __forceinline__ void take_heads(RunPtr r) {
        const int t = opaque(), lane = t & 63;
        const int k = r->k_o, n4 = k / 4, NS = r->splits, H = r->heads;
        if (wave == 0) {
            const bool need = 4 * lane < H * NS;
            unsigned off[1] = {16u * (unsigned)(need ? lane : 0)};
            f32x4 v[1];
            poll_words<1>(now + r->x_part + wg % kWalkCopies * kWalkWG, off, need, v, wait);
            float ss = (v[0][0] + v[0][1]) + (v[0][2] + v[0][3]);
            ss += lane_xor_f<1>(ss);                      // two lanes per head, or four
            if (NS == 16) ss += lane_xor_f<2>(ss);
            if (need && lane % (NS / 4) == 0) L.of_head[lane / (NS / 4)] = 1.0f / sqrtf(ss / (float)kWalkDim + a.eps);
        }
        auto all = [&](auto n) {
            constexpr int N = decltype(n)::value;
            unsigned off[N];
            f32x4 v[N];
#pragma unroll
            for (int i = 0; i < N; i++) off[i] = 16u * (unsigned)min(t + kSvcT * i, n4 - 1);
            poll_words<N>(now + r->x_att, off, wave * 64 < n4, v, wait);
            meet();
#pragma unroll
            for (int i = 0; i < N; i++) {
                const int c = t + kSvcT * i;
                if (c < n4) put_x(k, c, v[i] * L.of_head[c / (kWalkDim / 4)]);
            }
        };
        if (n4 > 2 * kSvcT) all(std::integral_constant<int, 4>());
        else all(std::integral_constant<int, 2>());
        vector_done();
    }

    // ---- latent attention (see latent_attn.hip), a workgroup per head and slice throughout.  The query's slice of latent columns; a split of
    // the rows for the whole latent query; the context of all splits through the slice's rows of W_uv.  Weights and rows are on their way
    // under the waits.  (Three kernels: 19 us.)
    __device__ __forceinline__ void latent(RunPtr r, int pos) {
        const int t = opaque(), lane = t & 63;
        constexpr int D = kWalkDim, RK = kWalkRank, RW = kWalkRow2, PW = walk_part(RK), PCS = RK / CE / 64;      // pieces of a row per lane
        const int H = r->heads, NS = r->splits, h = wg % H, slice = wg / H;
        if (slice >= NS || pos >= r->capacity) return;
        {   // ---- W_uk's slice of columns against the head's query
            const int cols = RK / NS, pc = cols / CE, c0 = slice * cols, c = t % pc, g = t / pc, step = kSvcT / pc;       // 32 or 64 columns
            constexpr int NP = 8;                         // rows per thread at most: 128 / (256 / pc), pc at most 16
            i32x4 u[NP];
            const auto* w = global(static_cast<const ET*>(r->uk)) + (size_t)h * D * RK + c0 + c * CE;
#pragma unroll
            for (int i = 0; i < NP; i++)
                if (g + i * step < D) u[i] = *reinterpret_cast<const Global<i32x4>*>(w + (size_t)(g + i * step) * RK);
            if (wave == 0) {
                unsigned off[1] = {4u * (unsigned)(h * (D + kWalkRot)) + 16u * (unsigned)min(lane, 47)};
                f32x4 v[1];
                poll_words<1>(now + r->x_in, off, lane < 48, v, wait);
                if (lane < 48) *reinterpret_cast<f32x4*>(M.q + 4 * lane) = v[0];
            }
            meet();
            float acc[CE];
#pragma unroll
            for (int e = 0; e < CE; e++) acc[e] = 0.0f;
#pragma unroll
            for (int i = 0; i < NP; i++)
                if (g + i * step < D) {
                    float wv[CE];
                    Chunk<ET>::unpack(make_uint4(u[i][0], u[i][1], u[i][2], u[i][3]), wv);
                    const float q = M.q[g + i * step];
#pragma unroll
                    for (int e = 0; e < CE; e++) acc[e] = fma_f(wv[e], q, acc[e]);
                }
            // over the rows: lanes of the same piece (pc 4, 8 or 16), then the waves
#pragma unroll
            for (int e = 0; e < CE; e++) {
                if (pc <= 4) acc[e] += lane_xor_f<4>(acc[e]);
                if (pc <= 8) acc[e] += lane_xor_f<8>(acc[e]);
                acc[e] += lane_xor_f<16>(acc[e]);
                acc[e] += lane_xor_f<32>(acc[e]);
            }
            if (lane < pc)
#pragma unroll
                for (int e = 0; e < CE; e++) M.sums[wave][lane * CE + e] = acc[e];
            meet();
            if (t < cols) put(r->x_ql + (unsigned)(h * RW + c0 + t), (M.sums[0][t] + M.sums[1][t]) + (M.sums[2][t] + M.sums[3][t]));
            if (slice == 0 && wave == 3) {                // the rotated part
                const int j = lane >> 1, rh = kWalkRot / 2;
                const float x = M.q[D + 2 * j], y = M.q[D + 2 * j + 1], cs = *global(r->cos_t + (size_t)pos * rh + j), sn = *global(r->sin_t + (size_t)pos * rh + j);
                put(r->x_ql + (unsigned)(h * RW + RK + lane), lane & 1 ? y * cs + x * sn : x * cs - y * sn);
            }
        }
        // ---- a split of the rows: a wave takes U rows at a time, a lane 8 of their latent columns; their rotated parts, 64 columns each, lie side by
        // side over the lanes
        const int lo = r->window > 0 && pos - r->window + 1 > 0 ? pos - r->window + 1 : 0, end = r->own_rows ? pos : pos + 1;      // rows lo .. end-1 are in the cache
        constexpr int U = 4;
        const int n = end - lo, per = max(((n + NS - 1) / NS + 4 * U - 1) / (4 * U) * (4 * U), 64), ns = max((n + per - 1) / per, 1);
        const int first = lo + slice * per, last = min(end, first + per);
        const unsigned part = r->x_part + (unsigned)((h * NS + slice) * PW);
        if (slice < ns) {
            const bool own = r->own_rows && slice == ns - 1;
            const auto* rows = global(static_cast<const ET*>(r->rows));
            i32x4 u[U][PCS], v[U][PCS], ur, vr;
            auto load = [&](int k0, i32x4 (&x)[U][PCS], i32x4& xr) {
#pragma unroll
                for (int i = 0; i < U; i++)
#pragma unroll
                    for (int j = 0; j < PCS; j++) x[i][j] = *reinterpret_cast<const Global<i32x4>*>(rows + (size_t)min(k0 + i, last - 1) * RW + lane * 8 + j * CE);
                constexpr int LR = kWalkRot / CE;         // lanes per rotated part
                xr = *reinterpret_cast<const Global<i32x4>*>(rows + (size_t)min(k0 + lane / LR, last - 1) * RW + RK + lane % LR * CE);
            };
            const int k1 = first + wave * U;
            if (k1 < last) load(k1, u, ur);
            if (own) {                                    // the row of this step: normed and rotated by each head for itself, stored by the first
                f32x4 p[1];
                unsigned off[1] = {4u * (unsigned)r->n_et + 16u * (unsigned)min(t, RW / 4 - 1)};
                if (wave < 3) {
                    poll_words<1>(now + r->x_in, off, t < RW / 4, p, wait);
                    if (t < RW / 4) *reinterpret_cast<f32x4*>(M.kx + 4 * t) = p[0];
                }
                meet();
                const float x0 = M.kx[2 * t], x1 = M.kx[2 * t + 1];
                const float rs = root(fma_f(x0, x0, x1 * x1), (float)RK);
                float o0 = x0 * rs * *global(r->latent_norm + 2 * t), o1 = x1 * rs * *global(r->latent_norm + 2 * t + 1);
                float e0 = 0.0f, e1 = 0.0f;
                if (t < kWalkRot / 2) {
                    const float a0 = M.kx[RK + 2 * t], a1 = M.kx[RK + 2 * t + 1], cs = *global(r->cos_t + (size_t)pos * (kWalkRot / 2) + t), sn = *global(r->sin_t + (size_t)pos * (kWalkRot / 2) + t);
                    e0 = (float)(ET)(a0 * cs - a1 * sn);
                    e1 = (float)(ET)(a1 * cs + a0 * sn);
                    M.kx[RK + 2 * t] = e0;
                    M.kx[RK + 2 * t + 1] = e1;
                }
                o0 = (float)(ET)o0;
                o1 = (float)(ET)o1;
                M.kx[2 * t] = o0;
                M.kx[2 * t + 1] = o1;
                if (h == 0) {
                    ET* dst = static_cast<ET*>(r->rows) + (size_t)pos * RW;
                    auto pair = [&](ET* p, float a, float b) {
                        if constexpr (std::is_same<ET, float>::value) {
                            store_past(p, a);
                            store_past(p + 1, b);
                        } else {
                            __attribute__((aligned(4))) ET w[2] = {(ET)a, (ET)b};
                            store_past(reinterpret_cast<float*>(p), *reinterpret_cast<const float*>(w));
                        }
                    };
                    pair(dst + 2 * t, o0, o1);
                    if (t < kWalkRot / 2) pair(dst + RK + 2 * t, e0, e1);
                }
            }
            {
                unsigned off[1] = {4u * (unsigned)(h * RW) + 16u * (unsigned)min(t, RW / 4 - 1)};
                f32x4 p[1];
                if (wave < 3) {
                    poll_words<1>(now + r->x_ql, off, t < RW / 4, p, wait);
                    if (t < RW / 4) *reinterpret_cast<f32x4*>(M.ql + 4 * t) = p[0];
                }
                meet();
            }
            float ql[8], qr[CE], acc[8], m = -1e30f, l = 0.0f;
            const float f = r->scale * kWalkLog2e;
#pragma unroll
            for (int e = 0; e < 8; e++) { ql[e] = M.ql[lane * 8 + e] * f; acc[e] = 0.0f; }
            constexpr int LR = kWalkRot / CE;
#pragma unroll
            for (int e = 0; e < CE; e++) qr[e] = M.ql[RK + lane % LR * CE + e] * f;
            auto columns = [&](const i32x4 (&x)[PCS], float (&o)[8]) {
#pragma unroll
                for (int j = 0; j < PCS; j++) Chunk<ET>::unpack(make_uint4(x[j][0], x[j][1], x[j][2], x[j][3]), reinterpret_cast<float (&)[CE]>(o[j * CE]));
            };
            auto take_rows = [&](int k0, const i32x4 (&x)[U][PCS], const i32x4& xr) {
                float s[U], w[CE], rot = 0.0f;
                Chunk<ET>::unpack(make_uint4(xr[0], xr[1], xr[2], xr[3]), w);
#pragma unroll
                for (int e = 0; e < CE; e++) rot = fma_f(w[e], qr[e], rot);
                rot = lanes_sum<LR>(rot);                 // of row lane / LR
#pragma unroll
                for (int i = 0; i < U; i++) {
                    float o[8];
                    columns(x[i], o);
                    s[i] = 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) s[i] = fma_f(o[e], ql[e], s[i]);
                }
                multi_sum_step<U, 1>(s, lane);            // lane i has row multi_row(i)
                float z[U], mx = m;
#pragma unroll
                for (int i = 0; i < U; i++) {
                    int from = 0;                         // the lane with row i
#pragma unroll
                    for (int b = 1, half = U / 2; half >= 1; b *= 2, half /= 2)
                        if (i & half) from |= b;
                    const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[0]), from)) + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rot), i * LR));
                    z[i] = k0 + i < last ? v : -INFINITY;
                    mx = fmaxf(mx, z[i]);
                }
                const float al = __builtin_amdgcn_exp2f(m - mx);
                m = mx;
                l *= al;
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] *= al;
#pragma unroll
                for (int i = 0; i < U; i++) {
                    const float p = __builtin_amdgcn_exp2f(z[i] - mx);
                    l += p;
                    float o[8];
                    columns(x[i], o);
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[e] = k0 + i < last ? fma_f(p, o[e], acc[e]) : acc[e];
                }
            };
            for (int k0 = k1; k0 < last; k0 += 8 * U) {
                if (k0 + 4 * U < last) load(k0 + 4 * U, v, vr);
                take_rows(k0, u, ur);
                if (k0 + 4 * U >= last) break;
                if (k0 + 8 * U < last) load(k0 + 8 * U, u, ur);
                take_rows(k0 + 4 * U, v, vr);
            }
            if (own && wave == 3) {                       // the row of this step
                float o[8], s = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    o[e] = M.kx[lane * 8 + e];
                    s = fma_f(o[e], ql[e], s);
                }
                s = fma_f(M.kx[RK + lane], M.ql[RK + lane] * f, s);
                s = wave_sum(s);
                const float mx = fmaxf(m, s), al = __builtin_amdgcn_exp2f(m - mx), p = __builtin_amdgcn_exp2f(s - mx);
                m = mx;
                l = l * al + p;
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] = fma_f(p, o[e], acc[e] * al);
            }
            if (lane == 0) { L.m[wave] = m; L.l[wave] = l; }
#pragma unroll
            for (int e = 0; e < 8; e += 4) *reinterpret_cast<f32x4*>(&M.sums[wave][lane * 8 + e]) = f32x4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
            meet();
            const float mt = fmaxf(fmaxf(L.m[0], L.m[1]), fmaxf(L.m[2], L.m[3]));
            float lt = 0.0f, o[2] = {0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < kSvcWaves; w++) {
                const float e = __builtin_amdgcn_exp2f(L.m[w] - mt);
                lt = fma_f(L.l[w], e, lt);
#pragma unroll
                for (int i = 0; i < 2; i++) o[i] += e == 0.0f ? 0.0f : M.sums[w][t + kSvcT * i] * e;
            }
#pragma unroll
            for (int i = 0; i < 2; i++) put(part + t + kSvcT * i, o[i]);
            if (t == 0) { put(part + RK, mt); put(part + RK + 1, lt); }
        } else {
            for (int i = t; i < RK + 2; i += kSvcT) unput(part + i);
        }
        // ---- the context of all splits, and W_uv's rows of the slice: a wave takes every fourth one
        {
            const int nr = D / NS;                        // 8 or 16
            constexpr int NP = 4;
            i32x4 u[NP][PCS];
            const auto* w = global(static_cast<const ET*>(r->uv)) + (size_t)(h * D + slice * nr) * RK + lane * 8;
#pragma unroll
            for (int i = 0; i < NP; i++)
                if (wave + 4 * i < nr)
#pragma unroll
                    for (int j = 0; j < PCS; j++) u[i][j] = *reinterpret_cast<const Global<i32x4>*>(w + (size_t)(wave + 4 * i) * RK + j * CE);
            const unsigned base = 4u * (unsigned)(h * NS * PW);
            float ms, ls;
            {
                unsigned off[1] = {base + 4u * (unsigned)(min(lane, ns - 1) * PW + RK)};
                f32x4 v[1];
                poll_words<1, 2>(now + r->x_part, off, lane < ns, v, wait);
                ms = lane < ns ? v[0][0] : -INFINITY;
                ls = v[0][1];
            }
            const float mt = wave_max(ms), e = lane < ns ? __builtin_amdgcn_exp2f(ms - mt) : 0.0f, lt = wave_sum(e == 0.0f ? 0.0f : ls * e), share = e / lt;
            const int half = __builtin_amdgcn_readfirstlane(t >> 7), c4 = t & 127;        // two halves of the threads take splits in turn
            f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int s0 = 0; s0 < ns; s0 += 8) {
                unsigned off[4];
                f32x4 v[4];
#pragma unroll
                for (int i = 0; i < 4; i++) off[i] = base + 4u * (unsigned)(min(s0 + 2 * i + half, ns - 1) * PW + 4 * c4);
                poll_words<4>(now + r->x_part, off, true, v, wait);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int sp = s0 + 2 * i + half;
                    const float p = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(share), min(sp, 63)));
                    if (sp < ns && p != 0.0f) sum += v[i] * p;
                }
            }
            *reinterpret_cast<f32x4*>((half ? M.kx : M.q) + 4 * c4) = sum;      // nobody reads them any more, M.sums may still be read
            meet();
            float ctx[8];
#pragma unroll
            for (int i = 0; i < 8; i++) ctx[i] = M.q[lane * 8 + i] + M.kx[lane * 8 + i];
#pragma unroll
            for (int i = 0; i < NP; i++)
                if (wave + 4 * i < nr) {
                    float o = 0.0f;
#pragma unroll
                    for (int j = 0; j < PCS; j++) {
                        float wv[CE];
                        Chunk<ET>::unpack(make_uint4(u[i][j][0], u[i][j][1], u[i][j][2], u[i][j][3]), wv);
#pragma unroll
                        for (int q = 0; q < CE; q++) o = fma_f(wv[q], ctx[j * CE + q], o);
                    }
                    o = wave_sum(o);
                    if (lane == 0) put(r->x_att + (unsigned)(h * D + slice * nr + wave + 4 * i), o);
                }
        }
    }

    __device__ __forceinline__ int rows_of(int n, int& r0) const {
        r0 = walk_rows(n, wg);
        return walk_rows(n, wg + 1) - r0;
    }
    // ---- mixture of experts.  The choice is every workgroup's own, from the router's outputs; it gives the streams their addresses.
    __device__ __forceinline__ void mixture(RunPtr r) {
        const int t = opaque(), lane = t & 63;
        const int W = a.width, E = r->experts, top = r->top, ff = r->ff, sf = r->shared_ff, kr = (E + 4) / 4 * 4;
        int r0;
        int rows = rows_of(2 * sf + kr, r0);
        sums_there();                                    // the sums of [shared gate/up; router; shared gate] are there
        for (int j = t; j < rows; j += kSvcT) {
            const int row = r0 + j;
            if (row >= 2 * sf) {                          // in copies: all workgroups at one line stand in line
                const float z = total(W, j);
                for (int c = 0; c < kWalkCopies; c++) put(r->x_route + (unsigned)(c * kr + row - 2 * sf), z);
            } else if ((row & 1) == 0) {
                put(r->x_hid + (unsigned)(top * ff + row / 2), glu_f(r->glu, total(W, j), total(W, j + 1), r->shared_limit));
            }
        }
        sums_done();
        if (wave == 0) {
            unsigned off[1] = {16u * (unsigned)min(lane, kr / 4 - 1)};
            f32x4 v[1];
            poll_words<1>(now + r->x_route + wg % kWalkCopies * kr, off, 4 * lane < kr, v, wait);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (4 * lane + e <= E) L.z[4 * lane + e] = v[0][e];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            int pick;
            float weight;
            route_wave(L.z, E, top, pick, weight);
            if (lane < top) {
                L.choice_w[lane] = weight;
#pragma unroll
                for (int k = 0; k < 2; k++) {             // gate/up and down
                    const int p = r->phase + k * top + lane;
                    const WalkPhase ph = a.phases[p];
                    const uintptr_t w = reinterpret_cast<uintptr_t>(static_cast<const ET*>(ph.w) + (size_t)pick * ph.stride + (size_t)walk_rows(ph.n, wg) * ph.kpad);
                    T.phase[p].x = (int)(unsigned)w;
                    T.phase[p].y = (int)(unsigned)(w >> 32);
                }
            }
            if (lane == 0) L.choice_w[top] = sigmoid_f(L.z[E]);
            chosen++;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            say(L.chosen, chosen);
        }
        vector_done();                                    // the vector is still the same
        rows = rows_of(2 * ff, r0);
        sums_there();
        const int all = rows / 2 * top;
        for (int j = t; j < all; j += kSvcT) {
            const int s = j / (rows / 2), i = j - s * (rows / 2), o = s * walk_red(PARTS, 2 * ff, W, QE);
            put(r->x_hid + (unsigned)(s * ff + r0 / 2 + i), glu_f(r->glu, total(W, 2 * i, o), total(W, 2 * i + 1, o), r->limit));
        }
        sums_done();
        // the vectors of the chosen experts one after the other, then the shared one's
        const int n4 = (top * ff + sf) / 4;
        for (int c0 = 0; c0 < n4; c0 += 4 * kSvcT) {
            unsigned off[4];
            f32x4 v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) off[i] = 16u * (unsigned)min(c0 + t + kSvcT * i, n4 - 1);
            poll_words<4>(now + r->x_hid, off, c0 + wave * 64 < n4, v, wait);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int c = c0 + t + kSvcT * i, s = min(c / (ff / 4), top);
                if (c < n4) put_x(s < top ? ff : sf, c - s * (ff / 4), v[i], s * ff);
            }
        }
        vector_done();
        rows = rows_of(W, r0);
        sums_there();
        const int step = walk_red(PARTS, W, ff, QE);
        for (int j = t; j < rows; j += kSvcT) {
            float y = 0.0f;
            for (int s = 0; s < top; s++) y = fma_f(L.choice_w[s], total(ff, j, s * step), y);
            put(r->x_y2 + (unsigned)(r0 + j), fma_f(L.choice_w[top], total(sf, j, top * step), y));
        }
        sums_done();
    }

    // ---- one token: returns the next one
    // the sums of a linear of n rows of k leave as they are
    __device__ __forceinline__ void plain(int n, int k, unsigned at, const float* bias) {
        const int t = opaque();
        int r0;
        const int rows = rows_of(n, r0);
        const float b = bias && t < rows ? *global(bias + r0 + t) : 0.0f;      // under the products
        sums_there();                                    // the sums are there
        for (int j = t; j < rows; j += kSvcT) put(at + (unsigned)(r0 + j), total(k, j) + (j == t ? b : bias ? *global(bias + r0 + j) : 0.0f));
        sums_done();
    }
    __device__ __forceinline__ int step(int token, int pos, bool choose) {
        const int W = a.width;
        RunPtr runs = (RunPtr)(uintptr_t)a.runs;
        embed(token);
        bool have = false;
        unsigned y = 0;
        const float* gb = nullptr;
        for (int i = 0; i < a.n_runs; i++) {
            RunPtr r = runs + i;
            norm(have, y, gb, r->g1, r->again ? token : -1);
            plain(r->n_in, W, r->x_in, r->in_bias);
            if constexpr (KIND == kWalkSharedKv) {
                if (r->dim == 64) shared_kv<64>(r, pos);
                else shared_kv<128>(r, pos);
                take(r->x_att, r->k_o);
            } else if (r->mixer == kWalkGla) {
                gla(r, pos);
                take_heads(r);
            } else {
                latent(r, pos);
                take(r->x_att, r->k_o);
            }
            plain(W, r->k_o, r->x_y, nullptr);
            have = true; y = r->x_y; gb = r->g1b;
            if (r->ff == 0) continue;
            norm(true, y, gb, r->g2, -1);
            y = r->x_y2; gb = r->g2b;
            if constexpr (KIND == kWalkMixture)
                if (r->experts) {
                    mixture(r);
                    continue;
                }
            sums_there();
            int r0;
            const int t = opaque(), rows = rows_of(2 * r->ff, r0);
            for (int j = t; j < rows / 2; j += kSvcT)
                put(r->x_hid + (unsigned)(r0 / 2 + j), glu_f(r->glu, total(W, 2 * j), total(W, 2 * j + 1), r->limit));
            sums_done();
            take(r->x_hid, r->ff);
            plain(W, r->ff, r->x_y2, nullptr);
        }
        const int t = opaque();
        if (!choose && t < 2) unput(a.x_cand + (unsigned)(2 * wg + t));        // what is not handed out in this step is unset behind the last one all the same
        if (!a.head) return 0;
        norm(have, y, gb, a.g_final, -1);
        sums_there();
        int r0;
        const int rows = rows_of(a.vocab, r0);
        float best = -INFINITY;
        int bi = 0x7fffffff;
        for (int j = t; j < rows; j += kSvcT) {
            const float v = total(W, j, a.lds_head);
            if (a.logits) a.logits[r0 + j] = v;
            if (v > best) { best = v; bi = r0 + j; }
        }
        sums_done();
        if (!choose) return 0;
        auto better = [&](float ov, int oi) {
            if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
        };
        auto reduce = [&](int n) {
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) better(__shfl_xor(best, k), __shfl_xor(bi, k));
            if (lane == 0) { L.bestv[n][wave] = best; L.besti[n][wave] = bi; }
            meet();
            best = L.bestv[n][0]; bi = L.besti[n][0];
#pragma unroll
            for (int w = 1; w < kSvcWaves; w++) better(L.bestv[n][w], L.besti[n][w]);
        };
        __builtin_amdgcn_s_waitcnt(0x0F70);               // vmcnt(0): what this wave stored in this step has arrived
        reduce(0);
        if (t == 0) { put(a.x_cand + 2 * wg, best); put(a.x_cand + 2 * wg + 1, __int_as_float(bi)); }
        unsigned off[1] = {16u * (unsigned)min(t, kWalkWG / 2 - 1)};
        f32x4 v[1];
        poll_words<1>(now + a.x_cand, off, t < kWalkWG / 2, v, wait);
        best = -INFINITY;
        bi = 0x7fffffff;
        if (t < kWalkWG / 2) {
            better(v[0][0], __float_as_int(v[0][1]));
            better(v[0][2], __float_as_int(v[0][3]));
        }
        reduce(1);
        return (unsigned)bi < (unsigned)a.vocab ? bi : 0;
    }
};

// KIND: models of shared key/value rows, of latent rows and gated linear attention (kWalkLatent), or of those with mixtures of experts.  PARTS: the
// vectors lie as three bfloat16 parts.
template <typename ET, int QW, int KIND, bool PARTS>
__global__ __launch_bounds__(kWalkT) void walk_kernel(WalkArgs a, int slots, ResidentEnd end) {
    constexpr int QE = kQuad / sizeof(ET);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    WalkLds& L = *reinterpret_cast<WalkLds*>(lds);
    WalkTables T;
    T.phase = reinterpret_cast<int4*>(lds + sizeof(WalkLds));
    T.group = T.phase + a.n_phases + 1;
    float* xs = reinterpret_cast<float*>(T.group + (KIND == kWalkMixture ? a.n_phases + 1 : 0));
    float* red = xs + a.lds_xs;
    const int phases = a.n_phases + (a.head ? 1 : 0);
    for (int p = threadIdx.x; p < phases; p += kWalkT) {
        const WalkPhase ph = a.phases[p];
        const int r0 = walk_rows(ph.n, blockIdx.x), rows = walk_rows(ph.n, blockIdx.x + 1) - r0, rq = ph.kpad / QE;
        const uintptr_t w = reinterpret_cast<uintptr_t>(static_cast<const ET*>(ph.w) + (size_t)r0 * ph.kpad);
        T.phase[p] = make_int4((int)(unsigned)w, (int)(unsigned)(w >> 32), PARTS ? rows : rq ? rows * rq : rows / 2, PARTS ? ph.kpad / kBlockK : rq);
        // choices of few quads begin with another wave in turn
        if (KIND == kWalkMixture)
            T.group[p] = make_int4(PARTS ? ph.x_off / 2 * 3 : ph.x_off, p == a.n_phases ? a.lds_head : ph.red_off, ph.group, (int)((unsigned)ph.last << 31 | (unsigned)ph.first << 30 | (unsigned)(rq == 0 && ph.slot & 1 ? kStrWaves / 2 : 0) << 16 | (unsigned)ph.routed));
    }
    if (threadIdx.x == 0) L.met = L.ready = L.done = L.sent = L.chosen = 0;
    __syncthreads();
    if (threadIdx.x >= kSvcT) {
        const char* ring = reinterpret_cast<const char*>(red + a.lds_red);
        if constexpr (PARTS) stream_parts<KIND == kWalkMixture, kFree<KIND>>(L, T, xs, red, ring, slots, phases, a.steps, a.routed, a.n_phases, a.lds_head);
        else stream_waves<ET, KIND == kWalkMixture, kFree<KIND>>(L, T, xs, red, ring, slots, phases, a.steps, a.routed, a.n_phases, a.lds_head);
        return;
    }
    Service<ET, QW, KIND, PARTS> s(a, L, T, xs, red);
    const int pos0 = a.state[0], step0 = a.state[1];
    int token = a.token[0];
    if ((unsigned)token >= (unsigned)a.vocab) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.state[3] = 2;
        token = 0;
    }
    const auto first = [&] { return blockIdx.x == 0 && s.opaque() == 0; };
    for (int i = 0; i < a.steps; i++) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");             // rows that other workgroups stored a token ago
        const int set = (a.parity + i) & 1;
        s.now = a.words + set * a.set;
        s.other = a.words + (1 - set) * a.set;
        token = s.step(token, pos0 + i, a.tokens_out != nullptr);
        if (a.tokens_out && first()) a.tokens_out[step0 + i] = token;
    }
    if (a.tokens_out && first()) {
        a.token[0] = token;
        a.state[0] = pos0 + a.steps;
        a.state[1] = step0 + a.steps;
    }
    if (first()) resident_done(end);
}

// What the ring of the stream waves is given besides: as much as is left, in slots of a quad for each of them.
size_t walk_lds(const WalkArgs& a) { return sizeof(WalkLds) + (a.n_phases + 1) * sizeof(int4) * (a.routed ? 2 : 1) + sizeof(float) * ((size_t)a.lds_xs + a.lds_red); }
static_assert(kStrWaves * kQuad == kWalkSlotBytes && kQuad == kWalkRow && kStrWaves == kWalkStreams, "a quad per wave");
static_assert((kWalkLdsMax - sizeof(WalkLds) - kWalkMixerLds) / kWalkSlotBytes == kWalkMaxSlots, "wait_quads counts as many");

template <typename ET>
int walk_launch(const WalkArgs& a, hipStream_t st) {
    FX_REQUIRE(a.n_phases < kWalkMaxPhases && a.width % 512 == 0 && a.width <= kWalkMaxWidth && a.vocab >= kWalkWG && a.steps > 0, "walk: %d linears, width %d, vocabulary %d", a.n_phases, a.width, a.vocab);
    const size_t used = walk_lds(a);
    FX_REQUIRE(used + kWalkMinSlots * kWalkSlotBytes <= kWalkLdsMax, "walk: %zu bytes of LDS", used);
    const int slots = (int)((kWalkLdsMax - used) / kWalkSlotBytes);
    const size_t lds = used + slots * kWalkSlotBytes;
    auto go = [&](auto* k, std::atomic<bool>& opted_in) {
        if (!opted_in.load(std::memory_order_acquire)) {
            FX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWalkLdsMax));
            opted_in.store(true, std::memory_order_release);
        }
        return resident_launch(k, kWalkWG, kWalkT, lds, st, a, slots);
    };
    static std::atomic<bool> opted[2][6];
    auto kind = [&](auto parts) {
        constexpr bool P = decltype(parts)::value;
        if (a.kind == kWalkSharedKv) return a.width <= 2048 ? go(walk_kernel<ET, 2, kWalkSharedKv, P>, opted[P][0]) : go(walk_kernel<ET, 4, kWalkSharedKv, P>, opted[P][1]);
        if (a.routed) return a.width <= 2048 ? go(walk_kernel<ET, 2, kWalkMixture, P>, opted[P][4]) : go(walk_kernel<ET, 4, kWalkMixture, P>, opted[P][5]);
        return a.width <= 2048 ? go(walk_kernel<ET, 2, kWalkLatent, P>, opted[P][2]) : go(walk_kernel<ET, 4, kWalkLatent, P>, opted[P][3]);
    };
    if constexpr (std::is_same<ET, bf16_t>::value)
        if (a.parts) return kind(std::true_type());
    return kind(std::false_type());
}
template int walk_launch<bf16_t>(const WalkArgs&, hipStream_t);
template int walk_launch<float>(const WalkArgs&, hipStream_t);

}  // namespace fx
