// cx_shapes.h — which kernels a call takes and the scratch it needs, from its
// sizes alone.  Plain C++, so that the rules can be checked on the host over
// whole ranges of sizes.
//
// A context's scratch only grows, and growing frees the old buffer, which a
// captured graph may still use.  So what a call asks for covers every call of
// the same entry point and shape with fewer tokens, whatever kernels these take:
// a program that has run its largest call allocates no more, under capture too.
// Parts that belong together share one allocation: a context's first call pays
// for each.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace cx {

// Geometry of the fast grouped kernels.
constexpr int kKB = 128;        // k-block: one scale per 128 columns
constexpr int kTileRows = 16;   // MFMA 16x16x32: 16 weight rows per wave
constexpr int kTileTok = 16;    // 16 token (pair) columns per MFMA tile

constexpr int kDecSplitMaxTokens = 8;  // tokens whose shared gate/up runs as k-parts (8 selection waves)

// The ABI states no alignment of x, and a view's rows may start anywhere.  Direct
// global->LDS loads and bounded buffer loads, 16 bytes a lane, are only given rows
// (and weights) that start on 16 bytes; all others go through plain loads, which
// take any address.
inline bool dma_aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Activation rows of one work item that fit the LDS budget next to the
// reduction tile (<= 16 KB); 0 when staging is not worth it or not possible.
inline int lds_rows(int max_lds, int hidden, int max_pairs_per_item, bool x_dma) {
    if (!x_dma || hidden % 512 != 0) return 0;  // rows are copied in 1 KB wave chunks
    const int budget = std::min(max_lds, 65536) - 16384;
    const int rows = budget / (hidden * 2 + 16);
    return (max_pairs_per_item <= rows && max_pairs_per_item <= 4) ? max_pairs_per_item : 0;
}

// ---------------------------------------------------------------------------
// One expert over 1..4 tokens (split-K down launch).
constexpr int kDownKsRows = 4;    // tokens
constexpr int kDownKsGroups = 2;  // 16-row groups per workgroup

inline bool expert_small_shape(int hidden, int inter) {
    const int nkg = hidden / kKB, nkd = inter / kKB;
    return hidden % (kDownKsGroups * kTileRows) == 0 && (nkg == 56 || nkg == 8 || nkg == 4) && (nkd == 16 || nkd == 4);
}

// One expert over 5..64 tokens (single mode, cx_few.h): gate/up writes h in the
// order the down launch reads it, few_scratch_bytes of it.  The limits, one
// expert of 7168 x 2048, us a call: 1..4 tokens stay on the k-part launches,
// whose rows keep their bits whatever the batch (2 tokens 12.4 against 13.3, 4
// tokens 14.7 against 13.4); 5 tokens 23.7 / 13.5; 64 tokens 31.4 against 41.1
// with the ping-pong GEMM, 65 tokens 45.4 / 41.3.
constexpr int kFewMinTokens = 5, kFewMaxTokens = 64;
constexpr size_t kFewHBlk = 8192;  // h bytes of a 16-token tile and 128 columns: 2 planes x 4 steps x 1 KB
constexpr int kFewGuWaves = 8;     // waves of a gate/up workgroup

// LDS of a gate/up workgroup: a block of x, later a partial tile, per wave and tile.
constexpr int few_gu_lds(int tiles) { return kFewGuWaves * tiles * 4096; }

inline int few_tiles(int n_tokens) { return (n_tokens + kTileTok - 1) / kTileTok; }

// The most tokens whose LDS a workgroup of this device can have (32 with 64 KB).
inline int few_max_tokens(int max_lds) { return std::min(kFewMaxTokens, max_lds / few_gu_lds(1) * kTileTok); }

inline size_t few_scratch_bytes(int n_tokens, int inter) {
    return (size_t)few_tiles(n_tokens) * (inter / kKB) * kFewHBlk;
}

inline bool few_ok(int hidden, int inter, int n_tokens, int max_lds) {
    const int nkg = hidden / kKB, nkd = inter / kKB;
    return hidden % kKB == 0 && inter % kKB == 0 && (nkg == 56 || nkg == 8 || nkg == 4) && (nkd == 16 || nkd == 4) &&
           n_tokens >= kFewMinTokens && n_tokens <= few_max_tokens(max_lds);
}

// The ping-pong GEMM (cx_pp.h).
constexpr int kPpRowsGu = 128;  // inter rows (of gate and of up) per gate/up workgroup
constexpr int kPpRowsDn = 256;  // hidden rows per down workgroup
constexpr int kPpMinBlocks = 4;  // 128-column blocks of a row: the ring's last blocks are peeled off
constexpr int kPpLds = 160 * 1024;  // one workgroup per CU

inline bool pp_ok(int hidden, int inter, int max_lds) {
    return inter % kPpRowsGu == 0 && hidden % kPpRowsDn == 0 && hidden / kKB >= kPpMinBlocks &&
           inter / kKB >= kPpMinBlocks && max_lds >= kPpLds;
}

// Shapes with 64-pair grouped kernels of their own (cx_grouped.h).
inline bool grp_shape(int hidden, int inter) {
    const int nkg = hidden / kKB, nkd = inter / kKB;
    return hidden % kKB == 0 && inter % kKB == 0 && (nkg == 56 || nkg == 8 || nkg == 4) && (nkd == 16 || nkd == 4);
}

// A grouped call of at least this many pairs per resident expert, on average,
// takes 128-pair items through the ping-pong GEMM: there the matrix cores bound
// the work as much as HBM does, and 64-pair items stream an expert's weights once
// for each.  us a layer with 64 and with 128-pair items at 20 / 32 / 48 / 64 / 80 /
// 128 pairs per expert, 7168 x 2048 with the shared expert:
//   256 experts  2226 2524 3037 3917 4909 6704   2153 2354 2630 3154 3559 5357
//   64 experts   614 666 783 982 1243 1660       624 713 778 864 937 1406
//   64, none shared  535 598 708 904 1132 1514   523 569 622 741 816 1276
// The shared expert's items, all full, run last: where the others last for few
// rounds of the CUs, 128 pairs at the end cost more than fewer reads of the weights
// save, up to 63 pairs (8 experts, which fit one round, gain from 20: 121 / 105; 4
// gain up to 48, 121 / 117, and from 80, but lose between, 125 / 142 at 64).
// Rows of few blocks gain later, a ring's fill and drain being a larger part of an
// item, and the later the fewer the experts, as the halved count of items leaves CUs
// idle: 7168 x 512 (hidden x inter), 256 experts 683 765 908 1171 1488 2070 and 732
// 807 936 1048 1181 1728; 64 / 80 / 96 pairs of 1024 x 512, 64 experts 76 91 109 and
// 86 91 96, 16 experts 44 45 44 and 51 47 51.
constexpr int kBigPairs = 128;
inline int big_min_pairs(int hidden, int inter, int n_resident, bool shared, int n_cu) {
    if (!grp_shape(hidden, inter)) return 20;
    const int wgs = (n_resident + (shared ? 1 : 0)) * (inter / kPpRowsGu);  // gate/up, an item each
    if (hidden / kKB == 56 && inter / kKB == 16) return !shared || wgs <= n_cu || wgs >= 8 * n_cu ? 20 : 64;
    return n_resident >= 256 ? 64 : n_resident >= 32 ? 80 : kBigPairs;
}

// Kernels of one expert on the fast paths.  Above 16 tokens the 64-token items of
// the grouped kernels leave most CUs idle (16 gate/up workgroups at 17..64
// tokens): 66 / 108 us at 32 / 300 tokens against 42 / 59 with the ping-pong GEMM.
// x_dma, gu_dma, down_dma: x, the gate and up and the down weights are dma_aligned.
enum ExpertPath { kPathGeneric, kPathSmall, kPathTiles, kPathFew };

struct ExpertRoute {
    ExpertPath path;
    bool pp_gate_up, pp_down;  // kPathTiles: this launch by the ping-pong GEMM
    int np_lds;                // rows of x staged in LDS
};

inline ExpertRoute expert_route(int n_tokens, int hidden, int inter, int max_lds, bool x_dma, bool gu_dma, bool down_dma) {
    ExpertRoute r{kPathTiles, false, false, n_tokens <= kTileTok ? lds_rows(max_lds, hidden, n_tokens, x_dma) : 0};
    if (x_dma && few_ok(hidden, inter, n_tokens, max_lds)) {
        r.path = kPathFew;
    } else if (n_tokens <= kDownKsRows && expert_small_shape(hidden, inter)) {
        r.path = kPathSmall;
    } else if (n_tokens > kTileTok && pp_ok(hidden, inter, max_lds)) {
        r.pp_gate_up = x_dma && gu_dma;
        r.pp_down = down_dma;
    }
    return r;
}

// Scratch of a call on one expert: h in fp32 (generic kernels), in fragment order
// (few-token path), as fp32 k-part sums of gate and up (1..4 tokens), or as two
// bf16 planes, the lo plane at h_lo_offset.
constexpr size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
constexpr size_t gu_part_bytes(int n_tokens, int inter) { return sizeof(float) * 2 * 2 * (size_t)n_tokens * inter; }
constexpr size_t h_lo_offset(int n_tokens, int inter) { return align256((size_t)n_tokens * inter * 2); }

inline size_t expert_call_bytes(ExpertPath path, int n_tokens, int inter) {
    switch (path) {
        case kPathGeneric: return (size_t)n_tokens * inter * 4;
        case kPathSmall: return gu_part_bytes(n_tokens, inter);
        case kPathFew: return few_scratch_bytes(n_tokens, inter);
        default: return h_lo_offset(n_tokens, inter) + (size_t)n_tokens * inter * 2;
    }
}

// The same of a context, for the paths of all calls with up to n_tokens tokens.
// Above kFewMaxTokens tokens the lo plane has a buffer of its own (a first call of
// 300 tokens took 78 us with two allocations of 1.2 MB and 89 to 114 with one of 2.4).
struct ExpertScratch {
    size_t bytes, lo_bytes;
};

inline ExpertScratch expert_scratch(int n_tokens, int hidden, int inter, int max_lds) {
    const bool small = expert_small_shape(hidden, inter);
    const int few = std::min(n_tokens, few_max_tokens(max_lds)), both = std::min(n_tokens, kFewMaxTokens);
    const size_t plane = n_tokens > both ? (size_t)n_tokens * inter * 2 : 0;
    return {std::max({small ? expert_call_bytes(kPathSmall, std::min(n_tokens, kDownKsRows), inter) : 0,
                      few_ok(hidden, inter, few, max_lds) ? expert_call_bytes(kPathFew, few, inter) : 0,
                      small && n_tokens <= kDownKsRows ? 0 : expert_call_bytes(kPathTiles, both, inter), plane}),
            plane};
}

// ---------------------------------------------------------------------------
// Router logits of many tokens in 16 x 32 tiles (k_route_logits_mfma): widths.
constexpr int kLgWaves = 8;    // K split
constexpr int kLgRing = 4;     // chunks in flight per wave

inline bool route_mfma_ok(int hidden) { return hidden % (kLgWaves * 32 * kLgRing) == 0; }

// Router logits of 4 to 256 tokens (k_route_logits_split): K slices, 0: another
// kernel.  Its 16 x 16 tiles win while one round of 256 CUs holds them: us a call
// with them and with the 16 x 32 tiles, 256 experts 256 / 300 tokens 30.6 / 42.1 and
// 46.9 / 42.2; 384 experts 160 / 176 / 256 tokens 137 / 150, 155 / 150 and 153 / 147;
// 512 experts 128 / 129 / 256 tokens 34.0 / 43.8, 47.2 / 43.8 and 48.9 / 44.2.  The
// selection reads every slice of its experts, so that above 384 experts a workgroup
// per expert row is still the faster at 4 tokens (512 experts 18.6 against 20.8).
// (Widths that only they and the kernel of a workgroup per expert row take keep
// them up to 256 tokens.)
constexpr int kLsMinTokens = 4, kLsMaxTokens = 256;
constexpr int kLsMaxTiles = 256;
constexpr int kLsWaves = 4;
constexpr int kLsMaxSlices = 8;

inline int route_slices(int n_tokens, int hidden, int n_experts) {
    if (n_tokens < kLsMinTokens + (n_experts > 384) || n_tokens > kLsMaxTokens || hidden % (kLsWaves * 32) != 0) return 0;
    const int tiles = (n_experts + kTileRows - 1) / kTileRows * ((n_tokens + kTileTok - 1) / kTileTok);
    if (tiles > kLsMaxTiles && route_mfma_ok(hidden)) return 0;
    int s = n_tokens <= 32 ? 8 : n_tokens <= 64 ? 4 : n_tokens <= 128 ? 2 : 1;
    while (hidden % (kLsWaves * 32 * s) != 0) s /= 2;
    return s;
}

// Scratch of a router call, offsets in bytes: logits [T, E] in fp64; their slices
// (slices x tokens is at most 256: 8 x 32, 4 x 64, 2 x 128); and for a layer with a
// decode pipeline (`decode`) its one-token scores s, c [E] and, with a shared
// expert, the k-part gate/up sums of up to kDecSplitMaxTokens tokens (dec_inter: its
// inter, else 0).  Up to 16 tokens of such a layer need no slices.
constexpr int kLsPartTokens = 256;

struct RouteScratch {
    size_t part, scores, gu_part, bytes;
};

inline RouteScratch route_scratch(int n_tokens, int hidden, int n_experts, bool decode, int dec_inter) {
    const bool part = n_tokens >= kLsMinTokens && hidden % (kLsWaves * 32) == 0 && !(decode && n_tokens <= kTileTok);
    RouteScratch z;
    z.part = align256(sizeof(double) * (size_t)n_tokens * n_experts);
    z.scores = z.part + align256(part ? sizeof(double) * kLsPartTokens * (size_t)n_experts : 0);
    z.gu_part = z.scores + align256(decode ? sizeof(double) * 2 * (size_t)n_experts : 0);
    z.bytes = z.gu_part + (decode ? gu_part_bytes(std::min(n_tokens, kDecSplitMaxTokens), dec_inter) : 0);
    return z;
}

// ---------------------------------------------------------------------------
// The plan of a grouped call (PlanPtrs).
constexpr int kPlanHdrInts = 8;
constexpr size_t kItemRecBytes = 88, kSlotRecBytes = 24;

struct PlanSizes {
    int max_slots, max_pairs, max_items, item_cap, maxt;
};

inline PlanSizes plan_sizes(int n_tokens, int top_k, int n_experts, int has_shared) {
    PlanSizes z;
    z.maxt = n_tokens <= kTileTok ? 1 : 4;
    z.item_cap = kTileTok * z.maxt;
    z.max_slots = std::min(n_tokens * top_k, n_experts) + has_shared;
    z.max_pairs = n_tokens * top_k + n_tokens * has_shared;
    z.max_items = z.max_slots + (z.max_pairs + z.item_cap - 1) / z.item_cap;
    return z;
}

// dense: a decode plan, which also fills pair_row.
inline size_t plan_bytes(const PlanSizes& z, int n_tokens, int top_k, bool dense) {
    const size_t ints = kPlanHdrInts + 3 * (size_t)z.max_slots + 3 * (size_t)z.max_items +
                        2 * (size_t)z.max_pairs + (size_t)n_tokens * (top_k + 1) +
                        (dense ? (size_t)z.max_pairs : 0);
    return kItemRecBytes * (size_t)z.max_items + kSlotRecBytes * (size_t)z.max_slots + ints * 4;
}

// Bytes of the plan buffer: the plan with the smallest items (16 pairs) and
// pair_row, so that neither the item size nor the pipeline makes it shrink.
inline size_t plan_buffer_bytes(int n_tokens, int top_k, int n_experts, int has_shared) {
    PlanSizes z = plan_sizes(n_tokens, top_k, n_experts, has_shared);
    z.max_items = z.max_slots + (z.max_pairs + kTileTok - 1) / kTileTok;
    return plan_bytes(z, n_tokens, top_k, true);
}

}  // namespace cx
