// One kernel for whole decode steps of one token (csrc/decode_float.hip): what it is given, and when it can be used.
#pragma once
#include "float_ops.h"

namespace fx {

constexpr int kWalkWG = 256;               // workgroups, one per CU: all of them have to be resident at once
constexpr int kWalkCopies = 8;            // of few words that every workgroup reads
constexpr int kWalkMaxPhases = 256;
constexpr int kWalkPolls = 1 << 20;        // about a second
constexpr int kWalkMaxWidth = 4096;
constexpr size_t kWalkLdsMax = 160 * 1024;
constexpr size_t kWalkMixerLds = 16 * 1024;
constexpr int kWalkMinSlots = 2, kWalkMaxSlots = 4, kWalkSlotBytes = 32 * 1024;       // of the weights' ring
constexpr int kWalkRow = 4096;             // bytes that the rows of all linears are a multiple of

// A linear of the step: n rows of kpad elements, dealt to the workgroups in runs of neighbouring rows (walk_rows).  The experts' products are groups of
// such linears, one per choice, between whose products nobody waits.
struct WalkPhase {
    const void* w;                         // of choice `slot` of the experts: + stride elements times the expert
    int n, kpad;
    int group, first, last;                // number of its group; first and last of it
    int routed;                            // 0, or the number (from 1) of the mixture whose choice it waits for
    int slot;
    size_t stride;
    int x_off, red_off;                    // where the vector starts in LDS (element of those ahead of it), and where the sums do (in floats, the same in all workgroups)
};
enum WalkMixer { kWalkSharedKv = 0, kWalkLatent = 1, kWalkGla = 2, kWalkMixture = 3 };
struct WalkRun {
    const float *g1, *g1b, *g2, *g2b;      // norms ahead of and behind (null: none) the two sublayers
    const float *in_bias, *kv_norm;
    void* rows;
    float* inv_rms;
    int mixer, again, n_in, n_et, k_o, ff, glu;
    float limit;
    // shared key/value rows
    int heads, kv_heads, rep, splits, dim, sink, temp_every, capacity;     // splits: of the rows, or slices of a head's columns
    float scale, temp_coef;
    // latent rows
    const void *uk, *uv;
    const float *latent_norm, *cos_t, *sin_t;
    int own_rows, window;                  // 0: the rows of an earlier run
    // gated linear attention
    const void* a2;
    const float *a2_bias, *head_norm;
    float* state;
    int a_rank;
    float tau;
    // mixture of experts (experts 0: none)
    int experts, top, shared_ff;
    float shared_limit;
    int phase;                             // of the first choice's gate/up; the down projections follow, then the shared expert's
    // where the words that the workgroups hand to each other lie, in floats from the start of a set
    unsigned x_in, x_ql, x_part, x_att, x_y, x_hid, x_route, x_y2;
};
struct WalkArgs {
    const WalkRun* runs;
    const WalkPhase* phases;
    int routed;                            // mixtures of a token
    int n_runs, n_phases;                  // without the head's phase, which is entry n_phases
    int kind;                              // mixers: shared key/value rows (kWalkSharedKv), or the others (kWalkLatent)
    int width, vocab;
    float eps, embed_scale;
    const bf16_t* embed;
    const float* g_final;
    float* words;                          // two sets of `set` floats
    size_t set;
    unsigned x_cand;                       // candidates of the arg-max
    int parity;                            // set of the first token
    int* err;                              // raised when a wait has timed out, and
    int* told;                             // the same in host memory
    int polls;                             // of a word, behind which a wait times out
    int* state;                            // HybridSlot::pos
    int* token;                            // token fed in; after greedy steps the last one found
    int* tokens_out;                       // greedy steps: tokens_out[state[1] + step]; null: a single step
    float* logits;                         // null: not wanted
    int steps, head;
    int parts;                             // vectors lie in LDS as three bfloat16 parts, for the matrix cores
    int lds_xs, lds_red;                   // floats
    int lds_head;                          // where the head's sums lie from the other linears': beside its vector, where that of a feed-forward is longer
};
// Rows r0 .. r1-1 of n belong to workgroup w: pairs of rows stay together.
__host__ __device__ inline int walk_rows(int n, int w) {
    const int r = 2 * (int)(((long long)w * ((n + 1) / 2)) / kWalkWG);
    return r < n ? r : n;
}
// Rows that a workgroup has at most.
__host__ __device__ inline int red_rows(int n) { return 2 * (((n + 1) / 2 + kWalkWG - 1) / kWalkWG); }
// Sums that a row of k leaves in LDS: with parts one for each stream wave that has blocks of it, otherwise one for each quad (of qe elements).  And those of n rows.
constexpr int kBlockK = 512, kWalkStreams = 8;
__host__ __device__ inline int walk_sums(bool parts, int k, int qe) {
    const int n = parts ? k / kBlockK : k / qe;
    return parts && n > kWalkStreams ? kWalkStreams : n > 0 ? n : 1;
}
__host__ __device__ inline int walk_red(bool parts, int n, int k, int qe) { return (parts ? (red_rows(n) + 3) / 4 * 4 : red_rows(n)) * walk_sums(parts, k, qe); }
size_t walk_lds(const WalkArgs& a);        // bytes
constexpr int kWalkExperts = 255, kWalkTop = 16;        // most
template <typename ET> int walk_launch(const WalkArgs& a, hipStream_t st);
// Attention over shared key/value rows: splits of the rows per query head (one workgroup each, and at least four columns of the head for
// each in the join), and the words of a split: the sums, maximum and weight sum.
inline int walk_splits(int heads, int dim) {
    int s = 4;
    while (s < 16 && 2 * s * heads <= kWalkWG && 8 * s <= dim) s *= 2;
    return s;
}
__host__ __device__ constexpr int walk_part(int dim) { return dim + 4; }
// Rows up to which this is the faster way.  A split's workgroup reads its rows for one query head, 43 us per MB; the kernels of the chain
// (shared_kv_attn.hip) read a row once for up to four heads, in up to eight times as many splits, but have a few us of launches in every layer, more
// beside wider linears.  Two layers, 32 heads on 8 of 64, width 2048, bfloat16, us per token in one kernel and in the chain: 24000 rows 94 and 98,
// 32000 104 and 103, 48000 125 and 110; four layers with feed-forwards of 8192 at 32000 rows 235 and 250.  With two layers the two meet at 0.5 to 0.8 MB per split (widths
// of 2048, heads of 64 and 128, alone on their rows and up to eight, both types), 0.51 at 1024, 0.75 to 1.2 at 4096; more layers' linears move that on: the
// line is within 12 % of the better side.
inline int walk_shared_kv_rows(const SharedKvDims& d, int width, int es) {
    const long long per_split = (384 * 1024 + 160LL * width) / ((long long)d.dim * es);
    return (int)(per_split * walk_splits(d.heads, d.dim));
}
inline bool walk_shared_kv_ok(const SharedKvDims& d) { return (d.dim == 64 || d.dim == 128) && d.dimp == d.dim && 4 * d.heads <= kWalkWG; }
// The other two are made for one size of head: a slice of a head's columns per workgroup, 16 or 8 for each head, and which lane holds which
// columns of a row is fixed when they are compiled.  Other sizes keep the chain of kernels, which takes any.
constexpr int kWalkDim = 128, kWalkRot = 64, kWalkRank = 512, kWalkRow2 = kWalkRank + kWalkRot, kWalkGlaRank = 16;
inline int walk_slices(int heads) { return heads <= 16 ? 16 : 8; }
inline bool walk_latent_ok(const LatentDims& d) {
    return d.dim == kWalkDim && d.vdim == kWalkDim && d.rot_dim == kWalkRot && d.kv_rank == kWalkRank && d.kvp == kWalkRank && d.ldc == kWalkRow2 && d.heads <= 32;
}
inline bool walk_gla_ok(const GlaDims& d) { return d.dim == kWalkDim && d.vdim == kWalkDim && d.a_rank <= kWalkGlaRank && d.heads <= 32; }

}  // namespace fx
