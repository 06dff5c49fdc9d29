// The prefill's piece lists: what attn_prefill.hip's 64-rows-a-wave kernel and
// the merge of its partials (attn_decode.hip) share.
#pragma once

#include "fl_common.hpp"

namespace fl {

constexpr int PF_HD = 256;
constexpr int R64_BQ = 256;            // (token, q head) rows a row tile
constexpr int R64_PLAN_MAX = 1024;     // entries of a plan: 2 KiB of kernel arguments
struct R64Plan {
    uint16_t v[R64_PLAN_MAX];
};

// A call's work over one kv head as a list of pieces (STREAM): the row tiles'
// causal walks laid end to end and cut into `bins` runs of equal cost, one a
// workgroup, wherever the cuts fall. Bin b runs from tile start[b].tile, KV tile
// start[b].j, up to start[b + 1]. Every piece leaves a partial, a row tile's in
// slots slot0[tile] .. slot0[tile + 1] - 1 of its kv head in KV order (an uncut
// tile's in its one slot: a second epilogue for it costs more registers than
// the kernel has); `first[b]` is bin b's first piece's slot. v[]: start (2 (bins
// + 1)), first (bins), slot0 (row tiles + 1).
struct StreamAt {
    const uint16_t* v;
    int bins;
    __device__ __forceinline__ int at(int i) const {   // (uniform)
        return __builtin_amdgcn_readfirstlane((int)v[i]);
    }
    __device__ __forceinline__ int tile(int b) const { return at(2 * b); }
    __device__ __forceinline__ int j(int b) const { return at(2 * b + 1); }
    __device__ __forceinline__ int first(int b) const { return at(2 * (bins + 1) + b); }
    __device__ __forceinline__ int slot0(int t) const { return at(3 * bins + 2 + t); }
};

// The partials of all kv heads: O unnormalised [slot][256 rows][256], then the
// running max (natural-log units) and sum [slot][256 rows]; kv head h's slots
// start at h * n.
struct StreamOut {
    float* pacc;
    float* pm;
    float* pd;
    int n;   // slots a kv head (R64_PIECES), splits (R64_SPLIT)
};

// z (and the output gate, `gate` the call's q | gate rows or null) from a piece
// list's partials: T tokens of n_q_heads heads, G a kv head.
int launch_piece_merge(const StreamOut& so, const R64Plan& plan, int bins, void* z, int z_pitch,
                       const void* gate, int g_pitch, int T, int n_q_heads, int G,
                       hipStream_t stream);

}  // namespace fl
